"""GPU parity of the integer kernels on 16-bit rows (graphs whose couplings share one
magnitude) at the sizes where their shape changes, replica by replica against the CPU
oracle: spins and tracked energies exact."""
import numpy as np
import pytest

import oracle as orc_mod
import qublar_amd as qa
from test_gpu_parity import check_int_batch, check_int_reference, gpu, say  # noqa: F401  (gpu is a fixture)

pytestmark = pytest.mark.gpu


def graph(n, degree, weight=1, signed=True, seed=0):
    g = qa.er_graph(n, min(1.0, degree / max(1, n - 1)), seed + 1)
    return qa.GraphArrays(g.n, g.eu, g.ev, weight * (g.ew if signed else np.abs(g.ew)))


# windows: shorter than a wave, exactly one, one and a bit; a complete graph (every lane a
# neighbour of every other); rows shorter and longer than a quarter wave, a wave, 64 entries;
# rows too long for the LDS; one replica and more than a workgroup's
GRAPHS = [(2, 1, 1), (63, 8, 3), (64, 63, 1), (65, 64, 2), (130, 129, 1), (200, 6, 5), (333, 30, 1), (400, 150, 1),
          (1500, 90, 7)]


@pytest.mark.parametrize("n,degree,weight", GRAPHS)
@pytest.mark.parametrize("R", [1, 9])
def test_reference_trajectory(gpu, n, degree, weight, R):
    g = graph(n, degree, weight, signed=n % 2 == 0)
    if g.m == 0:
        g = qa.GraphArrays(2, [0], [1], [weight])
    sched = qa.schedule(weight * max(1.0, degree) ** 0.5, 0.2 * weight, 25, 5)
    s, e, _ = check_int_reference(g, sched, R, 3)
    s2, e2, rep = check_int_reference(g, sched, R, 3, updates_per_launch=R * g.n * 7)
    assert rep["launches"] == 5 and np.array_equal(s, s2) and np.array_equal(e, e2)


def test_reference_trajectory_many_replicas(gpu):
    """More replicas than CUs: several per workgroup, the last workgroup part filled."""
    g = graph(100, 12)
    G = qa.Graph(g)
    sched = qa.schedule(3.0, 0.2, 12, 3)
    say("run_batch_reference R = 1037")
    s, e, _ = G.run_batch_reference(sched, 1, 1037)
    og = orc_mod.IntGraph(g.n, g.eu, g.ev, g.ew)
    for r in list(range(0, 1037, 61)) + [1034, 1035, 1036]:
        x, en = orc_mod.anneal_int(og, orc_mod.schedule(3.0, 0.2, 12, 3), 1 + r)
        assert np.array_equal((s[r, :g.n] > 0).astype(np.uint8), x) and e[r] == en


# the colour-class sweep: a workgroup per replica (classes of fewer bits than step waves, of
# more than a step holds, rows in L2), then several one-wave replicas per workgroup
@pytest.mark.parametrize("n,degree,weight", GRAPHS + [(2600, 3, 2)])
def test_colour_sweep_few_replicas(gpu, n, degree, weight):
    g = graph(n, degree, weight, signed=n % 2 == 0)
    if g.m == 0:
        g = qa.GraphArrays(2, [0], [1], [weight])
    sched = qa.schedule(weight * max(1.0, degree) ** 0.5, 0.2 * weight, 20, 4)
    check_int_batch(g, sched, 5, 3)
    check_int_batch(g, sched, 5, 3, updates_per_launch=5 * g.n * 7)


@pytest.mark.parametrize("n,degree,R", [(70, 69, 700), (150, 8, 1300), (600, 40, 1030), (900, 200, 520)])
def test_colour_sweep_many_replicas(gpu, n, degree, R):
    g = graph(n, degree, 3)
    check_int_batch(g, qa.schedule(3.0 * degree ** 0.5, 0.6, 6, 2), R, 11, updates_per_launch=R * n * 5)


def test_temperatures_outside_a_float(gpu):
    """Draws made ahead are bounded in float; temperatures past its range leave every uphill
    move to the FP64 exponential."""
    g = graph(90, 10)
    for t in (1e35, 1e-35):
        check_int_batch(g, qa.schedule(t, t, 6, 0), 3)
