"""qb_qubo_report.jobs counts the jobs run: replica blocks, or halves of them for an instance
that would outlast the others (replica block 4)."""
import pytest

import qublar_amd as qa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("replica_block", [4, 8])
def test_jobs_reported(replica_block):
    # one instance 60 times the others' size: its block of four takes longer than an even share
    # of the batch (on more than 4 CUs) and than half of itself; theirs do not
    inst = [qa.random_regular_qubo(12000, 8, 1, 11)] + [qa.random_regular_qubo(200, 4, 2 + k, 6) for k in range(5)]
    print(f"qubo jobs rb={replica_block}", flush=True)
    out = qa.QuboBatch(inst).anneal(qa.schedule(2.0, 0.1, 6, 0), replica_block=replica_block, block=256)
    long_job = 2 if replica_block == 4 else replica_block
    assert out["report"]["jobs"] == -(-11 // long_job) + 5 * -(-6 // replica_block)
    assert out["report"]["replica_block"] == replica_block
