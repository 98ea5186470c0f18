"""GPU parity of the reference's own float trajectory (anneal_branch) at the sizes where its
windows, batches and passes change shape, against the CPU oracle's reference mode: spins and
p_void identical, energies within 1e-9 relative."""
import numpy as np
import pytest

import qublar_amd as qa
from test_gpu_parity import check_branches_reference, gpu  # noqa: F401  (gpu is a fixture)
from test_gpu_solo import problem

pytestmark = pytest.mark.gpu


def columns(n, sizes):
    """n columns, every third one without rays, the rest taking the sizes in turn."""
    return [0 if i % 3 == 1 else sizes[i % len(sizes)] for i in range(n)]


@pytest.mark.parametrize("n,sizes,neighbours", [
    (1, [1], 0),                      # one lane, one entry
    (63, [3], 4), (64, [4], 6),       # a window's edges
    (65, [16, 17], 8), (129, [5], 12),  # register neighbours, and more than they hold
    (64, [0], 4), (200, [0], 10),     # no rays
    (64, [6], 4), (64, [18], 4),      # a block of 256 entries, a batch of 768, and one over
    (130, [60, 1, 255, 256, 257], 4), # several batches and passes
    (70, [3839, 3840, 3841, 767, 768, 769], 2),
])
def test_rayref_edges(gpu, n, sizes, neighbours):
    """Hot enough that bits with and without rays flip at the start, cold at the end."""
    P = problem(columns(n, sizes), 4000, 0.6, neighbours=neighbours, dup=(0, 12), seed=n)
    one = check_branches_reference(P, qa.schedule(20.0, 0.2, 12, 3), 6, seed_offset=3)
    two = check_branches_reference(P, qa.schedule(20.0, 0.2, 12, 3), 6, seed_offset=3, sweeps_per_launch=4)
    assert np.array_equal(one["branches"], two["branches"])


def test_rayref_spins_past_the_lds(gpu):
    """260,097 bits: the spins of a branch are bytes in global memory."""
    n = 260097
    cols = np.zeros(n, int)
    cols[[0, 63, 64, 5000, n - 1]] = 40
    check_branches_reference(problem(list(cols), 300, 0.6, seed=1), qa.schedule(4.0, 0.5, 3, 1), 2, sweeps_per_launch=2)


@pytest.mark.parametrize("t", [1e-310, 1e301])
def test_rayref_extreme_temperatures(gpu, t):
    """Temperatures whose reciprocal is no ordinary number: every exponential exact."""
    check_branches_reference(problem(columns(150, [9]), 200, 0.6, seed=2), qa.schedule(t, t, 3, 1), 4)
