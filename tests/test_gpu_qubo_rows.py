"""GPU parity of the batched QUBO engine where the row walk and the energies change shape:
rows of 0 to 40 entries mixed in one class (every remainder of the 16, 8, 4, 2 and 1 entry
steps, padding past the shorter rows), part-filled tiles, one to nine replicas, and an instance
past the 65,536 bits whose spins fit a workgroup's LDS. Spins bit-exact against the oracle,
energies within 1e-9 relative."""
import numpy as np
import pytest

import oracle as orc_mod
import qublar_amd as qa
from test_gpu_qubo import oracle_x, say

pytestmark = pytest.mark.gpu


def uneven(n, longest, seed, replicas):
    """n bits; bit i wants i % (longest + 1) partners drawn at random."""
    rng = np.random.default_rng(seed)
    pairs = set()
    for i in range(n):
        for j in rng.integers(0, n, (i % (longest + 1)) // 2):
            if i != j:
                pairs.add((min(i, int(j)), max(i, int(j))))
    ab = np.array(sorted(pairs), int).reshape(-1, 2)
    J = rng.normal(0, 1, len(ab)).astype(np.float32)
    u, v, w = np.r_[ab[:, 0], ab[:, 1]], np.r_[ab[:, 1], ab[:, 0]], np.r_[J, J]
    by = np.lexsort((v, u))
    row = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))])
    return qa.QuboInstance(row, v[by], w[by], rng.normal(0, 0.5, n), replicas, seed + 77)


@pytest.mark.parametrize("rb,block", [(4, 1024), (4, 256), (8, 1024), (16, 256), (32, 256)])
def test_rows_and_energies(rb, block):
    inst = [uneven(n, d, 10 * n + d, r) for n, d, r in ((1, 0, 1), (63, 0, 2), (64, 3, 3), (65, 8, 4), (700, 40, 9),
                                                        (1300, 17, 6))]
    if (rb, block) == (4, 1024):
        inst.append(uneven(65537, 4, 5, 3))
    B = qa.QuboBatch(inst)
    sched = qa.schedule(4.0, 0.1, 10, 2)
    say(f"replica block {rb} block {block}")
    out = B.anneal(sched, mode=0, replica_block=rb, block=block)
    for k, q in enumerate(inst):
        order, _ = B.colouring(k)
        ref = oracle_x(q, order, sched)
        assert np.array_equal(out["x"][k], ref), f"instance {k}: {(out['x'][k] != ref).sum()} spins differ"
        e_ref = np.array([orc_mod.qubo_energy(q.row_ptr, q.col, q.J, q.h, x) for x in ref])
        assert np.allclose(out["energy"][k], e_ref, rtol=1e-9, atol=1e-9)
