"""GPU parity of the dense engine's fields from scratch where the list of set bits changes
shape: fewer rows than one load of them, none at all (cold fields that flip nothing), a
recompute after every sweep, a part's last wave half empty, and more bits (8,257) than one
list holds; several workgroups per replica and one. Spins bit-exact against the oracle,
energies within 1e-9 relative."""
import numpy as np
import pytest

import oracle as orc_mod
import qublar_amd as qa
from test_gpu_dense import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,R,shift,sweeps", [
    (65, 2, 0.0, 6), (256, 65, 0.0, 4), (290, 2, 0.0, 6), (1100, 1, 0.0, 6),
    (300, 2, 9.0, 5), (130, 2, 9.0, 5),    # h far above zero: no bit is ever set, or a few
    (8257, 1, 0.0, 2),
])
def test_fields_from_scratch(n, R, shift, sweeps):
    Q, h = qa.dense_qubo(n, 11)
    h = (h + np.float32(shift * np.abs(Q).sum(axis=1).max() if shift else 0.0)).astype(np.float32)
    sched = qa.schedule(1.0, 0.05, sweeps, 0)
    say(f"dense n={n} R={R} shift={shift}")
    out = qa.DenseQubo(Q, h).anneal(sched, R, seed_offset=4, precision=qa.FP32, recompute_every=1)
    osched = orc_mod.schedule(1.0, 0.05, sweeps, 0)
    for b in range(R):
        ref = orc_mod.dense_anneal(Q, h, osched, b + 1 + 4, qa.FP32, 1)
        assert np.array_equal(out["x"][b], ref), f"replica {b}: {(out['x'][b] != ref).sum()} spins differ"
        e = orc_mod.dense_energy(Q, h, ref)
        assert abs(out["energy"][b] - e) <= 1e-9 * max(1.0, abs(e))
