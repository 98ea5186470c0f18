"""The region posterior at the sizes where its enumeration changes shape -- padded problems,
one thread block, no walked bits, each length of the walk -- and where its weights are made
one exponential each, against numpy's 2^n states. Energies of both differ by at most some
200 additions' rounding (1e-12 of their size), a weight by that times beta."""
import numpy as np
import pytest

import qublar_amd as qa

pytestmark = pytest.mark.gpu


def states(h, J):
    e = np.zeros(1)
    f = [np.full(1, v) for v in h]
    for i in range(len(h)):
        e = np.concatenate([e, e + f[i]])
        f = [np.concatenate([v, v + J[i, j]]) if j > i else v for j, v in enumerate(f)]
    return e


def check(h, J, beta):
    n = len(h)
    print(f"roi n={n} beta={beta}", flush=True)
    g = qa.roi_enumerate(h, J, beta)
    e = states(h, J)
    size = np.abs(h).sum() + np.abs(J).sum()
    tol = 1e-12 * size
    k = int(np.argmin(e))
    assert abs(g["e_min"] - e[k]) <= tol
    assert e[g["map_index"]] - e[k] <= tol
    w = np.exp(-beta * (e - e[k]))
    z = w.sum()
    rel = 1e-13 + 4 * beta * tol
    assert abs(g["log_z"] + beta * e[k] - np.log(z)) <= rel + 1e-13 * beta * abs(e[k])
    marginal = np.array([w.reshape(-1, 2, 1 << i)[:, 1].sum() for i in range(n)]) / z
    assert np.allclose(g["marginal"], marginal, rtol=2 * rel, atol=1e-300)
    assert abs(g["p_map"] * z - 1.0) <= rel
    return g, k


@pytest.mark.parametrize("n", [1, 4, 12, 13, 14, 21, 22, 23, 24, 25])
@pytest.mark.parametrize("beta", [1.0, 40.0])
def test_sizes(n, beta):
    """beta 40 puts the group bits' reach past 600: one exponential per state."""
    rng = np.random.default_rng(n)
    h, J = rng.normal(0, 2, n), np.triu(rng.normal(0, 1, (n, n)), 1)
    g, k = check(h, J, beta)
    assert g["map_index"] == k


@pytest.mark.parametrize("n", [3, 13, 19, 24])
def test_ties_take_the_smallest_state(n):
    """Whole couplings: every energy is exact, and many states share the minimum."""
    rng = np.random.default_rng(50 + n)
    h = rng.integers(-1, 2, n).astype(float)
    J = np.triu(rng.integers(-1, 2, (n, n)), 1).astype(float)
    g, k = check(h, J, 0.5)
    assert g["map_index"] == k and g["e_min"] == states(h, J)[k]


@pytest.mark.parametrize("n", [26, 27, 28, 29, 30, 31])
def test_walk_lengths(n):
    """Two coupled blocks and independent bits: log Z and marginals in closed form."""
    rng = np.random.default_rng(70 + n)
    h = rng.normal(0, 2, n)
    J = np.zeros((n, n))
    half = rng.permutation(n)[:14]
    for a in half:
        for b in half:
            if a < b:
                J[a, b] = rng.normal()
    print(f"roi n={n}", flush=True)
    g = qa.roi_enumerate(h, J, 1.0)
    half = np.sort(half)
    rest = np.setdiff1d(np.arange(n), half)
    e = states(h[half], J[np.ix_(half, half)])
    w = np.exp(-(e - e.min()))
    assert abs(g["log_z"] - (np.log(w.sum()) - e.min() + np.logaddexp(0.0, -h[rest]).sum())) <= 1e-11
    m = np.array([w.reshape(-1, 2, 1 << i)[:, 1].sum() for i in range(14)]) / w.sum()
    assert np.allclose(g["marginal"][half], m, rtol=1e-11)
    assert np.allclose(g["marginal"][rest], 1.0 / (1.0 + np.exp(h[rest])), rtol=1e-11)
    assert abs(g["e_min"] - (e.min() + np.minimum(h[rest], 0).sum())) <= 1e-11
