"""The region posterior's marginals where they are small: group bits (the lowest five) with a
reach, beta times their fields and couplings, up to the 600 at which their weights stop being
made as products, and strongly biased bits outside the group. Every state of weight is a
double's ordinary value, so each marginal is held to its own size, against numpy's 2^n states.
An energy of either side has at most some 200 additions' rounding (200 * 2^-53 of its size), a
weight that times beta from both sides, and some 30 roundings of its own."""
import numpy as np
import pytest

import qublar_amd as qa
from test_gpu_roi_walk import states

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [13, 19, 24])   # thread bits alone, block bits, a walked bit
@pytest.mark.parametrize("signs", [(-1, -1, -1, -1, -1), (1, 1, 1, 1, 1), (-1, 1, -1, 1, -1)])
@pytest.mark.parametrize("reach,beta", [(100.0, 1.0), (300.0, 1.0), (500.0, 0.5), (590.0, 1.0)])
def test_small_marginals(n, signs, reach, beta):
    """Biased bits at a thread, a block and the last walked place where there is one: e^-60 to
    e^-260 each."""
    rng = np.random.default_rng([n, int(reach)])
    h, J = rng.normal(0, 2, n), np.triu(rng.normal(0, 1, (n, n)), 1)
    outside = {5: 230.0, 8: -260.0, n - 2: 250.0, n - 1: 60.0}
    for b, v in outside.items():
        h[b] = v / beta
    rest = np.abs(J[:5]).sum() + np.abs(J[:5, :5]).sum()   # a coupling inside the group counts for both its bits
    h[:5] = np.array(signs) * (reach / beta - rest) / 5.0
    print(f"roi marginals n={n} signs={signs} reach={reach}", flush=True)
    g = qa.roi_enumerate(h, J, beta)
    e = states(h, J)
    w = np.exp(-beta * (e - e.min()))
    z = w.sum()
    marginal = np.array([w.reshape(-1, 2, 1 << i)[:, 1].sum() for i in range(n)]) / z
    assert marginal.min() > 1e-300
    size = np.abs(h).sum() + np.abs(J).sum()
    rel = 2 * beta * 200 * 2.0 ** -53 * size + 30 * 2.0 ** -53
    assert np.all(np.abs(g["marginal"] - marginal) <= 2 * rel * marginal)
    assert abs(g["p_map"] * z - 1.0) <= 2 * rel
