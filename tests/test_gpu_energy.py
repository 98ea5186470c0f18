"""FP64 energies on the device against numpy at the sizes where the reduction changes
shape: one partial block, fewer blocks than threads, several rounds of the final sum; one
state, a full group of 16, and a group with one state. The sums differ from numpy's only
in order: 1e-12 of the terms' magnitude covers 1e5 additions of them."""
import numpy as np
import pytest

import qublar_amd as qa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_rays", [(1, 1), (16, 15), (17, 33), (5000, 4096), (45000, 70000)])
@pytest.mark.parametrize("states", [1, 16, 17])
def test_energy_sizes(n, n_rays, states):
    rng = np.random.default_rng(n + states)
    deg = rng.integers(0, min(n_rays, 6) + 1, n)
    row_ptr = np.concatenate([[0], np.cumsum(deg)])
    bit = np.repeat(np.arange(n), deg)
    # consecutive rays from a random start: distinct in a column
    ray = (np.repeat(rng.integers(0, n_rays, n), deg) + np.arange(len(bit)) - row_ptr[bit]) % n_rays
    a = rng.uniform(0.01, 0.5, len(ray)).astype(np.float32)
    d, w = rng.uniform(0, 1, n_rays), rng.uniform(1, 9, n_rays)
    nbr = np.array([j for i in range(n) for j in (i - 1, i + 1) if 0 <= j < n], np.int32)
    nbr_ptr = np.concatenate([[0], np.cumsum([(i > 0) + (i < n - 1) for i in range(n)])])
    field = rng.normal(0, 1, n)
    P = qa.ProblemArrays(row_ptr, ray, a, d, w, nbr_ptr, nbr, 0.7, 0.0, field, colour=None)
    X = (rng.random((states, n)) < 0.3).astype(np.uint8)
    print(f"energy n={n} rays={n_rays} states={states}", flush=True)
    tot, dat, pri = qa.Problem(P).energy(X)
    for k, x in enumerate(X):
        r = np.bincount(ray, weights=a.astype(np.float64) * x[bit], minlength=n_rays) - d
        ed = 0.5 * np.sum(w * r * r)
        ep = 0.7 * np.count_nonzero(x[:-1] != x[1:]) + np.sum(field * x)
        scale = ed + 0.7 * n + np.sum(np.abs(field))
        assert abs(dat[k] - ed) <= 1e-12 * scale and abs(pri[k] - ep) <= 1e-12 * scale
        assert abs(tot[k] - (ed + ep)) <= 1e-12 * scale
