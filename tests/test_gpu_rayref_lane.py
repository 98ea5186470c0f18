"""GPU parity of the reference's own float trajectory with a lane to a column (many branches of
short columns), against the CPU oracle's reference mode and against the few-branch kernel."""
import numpy as np
import pytest

import qublar_amd as qa
from test_gpu_parity import check_branches_reference, gpu  # noqa: F401  (gpu is a fixture)
from test_gpu_solo import problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,sizes,neighbours,R", [
    (1, [1], 0, 1501),                       # one lane, one entry; the last workgroup part filled
    (63, [3], 4, 2050), (64, [5], 0, 1900),  # a window's edges
    (65, [1, 2, 3], 8, 2400),                # neighbours in one round of eight
    (130, [2], 10, 2400),                    # and in two
    (130, [4, 0], 4, 4096),                  # half of the bits ray-free
    (100, [1] * 9 + [9], 2, 1800),           # a column of two rounds of entries
])
def test_many_branches_of_short_columns(gpu, n, sizes, neighbours, R):
    """Hot enough that bits with and without rays flip at the start, cold at the end; two columns
    repeat a ray."""
    P = problem([sizes[i % len(sizes)] for i in range(n)], 400, 0.6, neighbours=neighbours, dup=(2, 12), seed=n)
    prob = qa.Problem(P)
    assert prob.anneal_reference_kernel(R) == "ray_ref_lane"
    assert prob.anneal_reference_kernel(16) == "ray_ref"
    sched = qa.schedule(20.0, 0.2, 7, 2)
    one = check_branches_reference(P, sched, R, seed_offset=3)
    two = check_branches_reference(P, sched, R, seed_offset=3, sweeps_per_launch=4)
    assert np.array_equal(one["branches"], two["branches"])
    few = prob.anneal_branches_reference(sched, 16, 3)
    many = prob.anneal_branches_reference(sched, R, 3)
    assert np.array_equal(one["branches"][:16], few["branches"]) and np.array_equal(one["branches"], many["branches"])


@pytest.mark.parametrize("t", [1e-310, 1e301])
def test_extreme_temperatures(gpu, t):
    """Temperatures whose reciprocal is no ordinary number: every exponential exact."""
    check_branches_reference(problem([3] * 90, 200, 0.6, seed=2), qa.schedule(t, t, 3, 1), 2050)


def test_long_columns_and_ray_free_bits_stay(gpu):
    """Where the terms kernel is the shorter at any number of branches."""
    assert qa.Problem(problem([12] * 128, 400, 0.6)).anneal_reference_kernel(1 << 16) == "ray_ref"
    assert qa.Problem(problem([0] * 128, 400, 0.6)).anneal_reference_kernel(1 << 16) == "ray_ref"
    assert qa.Problem(problem([2] * 100 + [16], 400, 0.6)).anneal_reference_kernel(1 << 16) == "ray_ref"
