"""GPU parity of the one-workgroup-per-branch sweep (problems whose branch state fits one
CU's LDS) at the sizes where its tiles change shape, against the CPU oracle with the
engine's colouring and keys, and against the XCD-team sweep (an explicit workgroup count)
on the same problem: spins and p_void identical, energies within 1e-9 relative."""
import numpy as np
import pytest

import qublar_amd as qa
from test_gpu_parity import check_branches, gpu, say  # noqa: F401  (gpu is a fixture)

pytestmark = pytest.mark.gpu


def problem(columns, n_rays, lam, neighbours=4, dup=(), seed=0):
    """Bits with the given entry counts on random rays (a repeated ray in the columns of
    `dup`), each tied to the next `neighbours` / 2 bits on both sides."""
    rng = np.random.default_rng(seed)
    n = len(columns)
    rays, row_ptr = [], [0]
    for i, k in enumerate(columns):
        rs = rng.choice(n_rays, size=k, replace=False)
        if i in dup and k > 1:
            rs[-1] = rs[0]
        rays.append(rs)
        row_ptr.append(row_ptr[-1] + k)
    ray = np.concatenate(rays) if rays else np.zeros(0, np.int32)
    half = neighbours // 2
    nbr = [[j for j in range(i - half, i + half + 1) if 0 <= j < n and j != i] for i in range(n)]
    nbr_ptr = np.concatenate([[0], np.cumsum([len(v) for v in nbr])])
    return qa.ProblemArrays(row_ptr, ray, rng.uniform(0.002, 0.05, len(ray)), rng.uniform(0, 0.3, n_rays),
                            rng.uniform(2, 30, n_rays), nbr_ptr, np.concatenate(nbr) if nbr else [], lam, 0.9,
                            rng.normal(0.4, 0.7, n))


# one entry to a wide bit of several passes: 1, 16 and 17 chains around the tiles' lanes, 32
# and 33 around the wide bits', 128 and 129 around a pass of one
EDGES = [0, 1, 4, 5, 15, 16, 17, 32, 33, 128, 129, 255, 256, 257, 511, 512, 513, 600, 2047, 2048, 2049, 5000]


@pytest.mark.parametrize("precision,recompute", [(qa.FP64, 0), (qa.FP32, 3)])
@pytest.mark.parametrize("lam,neighbours", [(0.7, 4), (-0.4, 10)])
def test_column_lengths(gpu, precision, recompute, lam, neighbours):
    cols = EDGES + [int(v) for v in np.random.default_rng(1).integers(0, 40, 150)]
    P = problem(cols, 6000, lam, neighbours, dup=(4, 7, 13, 19, 30, 31))
    sched = qa.schedule(8.0, 0.3, 12, 3)
    _, a = check_branches(P, sched, 5, seed_offset=2, precision=precision, recompute_every=recompute,
                          sweeps_per_launch=4)
    _, b = check_branches(P, sched, 5, seed_offset=2, precision=precision, recompute_every=recompute, workgroups=256)
    assert np.array_equal(a["branches"], b["branches"])


def test_class_wider_than_the_draws_made_ahead(gpu):
    """700 bits of one class, each on a ray of its own."""
    P = problem([1] * 700, 1400, 0.0, neighbours=0)
    P.ray[:] = np.arange(700)
    check_branches(P, qa.schedule(4.0, 0.5, 15, 5), 9, precision=qa.FP32, recompute_every=4)


def test_more_branches_than_compute_units(gpu):
    P = qa.muon_scene(grid=20, sky_az=45, sky_th=12, log2_muons=22)
    prob = qa.Problem(P)
    sched = qa.schedule(20.0, 1.0, 6, 2)
    say("300 branches, one workgroup each, against the team sweep")
    a = prob.anneal_branches(sched, 300, 1, qa.FP32, 4)
    b = prob.anneal_branches(sched, 300, 1, qa.FP32, 4, workgroups=256)
    assert np.array_equal(a["branches"], b["branches"]) and np.array_equal(a["tri"], b["tri"])
    assert np.allclose(a["energy"], b["energy"], rtol=1e-9)


def test_spins_packed_in_bits(gpu):
    """130,000 spins that fit the LDS beside 8,000 residuals only as bits; one ray of 200
    bits makes 200 classes."""
    n = 130000
    cols = np.zeros(n, int)
    cols[:200] = 3
    P = problem(cols, 8000, 0.5, neighbours=2)
    P.ray[0:600:3] = 7999
    P.ray[1:600:3] = np.arange(200)
    P.ray[2:600:3] = np.arange(200, 400)
    check_branches(P, qa.schedule(4.0, 0.5, 3, 1), 3, precision=qa.FP32, recompute_every=2)
