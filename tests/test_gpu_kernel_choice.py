"""The parity tests of each kernel reach it: the problems and graphs of test_gpu_solo.py and
test_gpu_introws.py, by the kernel that their calls run. A rule that moves leaves one of these
failing, not a kernel untested."""
import numpy as np
import pytest

import qublar_amd as qa
from test_gpu_introws import GRAPHS, graph
from test_gpu_solo import EDGES, problem

pytestmark = pytest.mark.gpu


def test_one_workgroup_per_branch():
    cols = EDGES + [int(v) for v in np.random.default_rng(1).integers(0, 40, 150)]
    for lam, neighbours in ((0.7, 4), (-0.4, 10)):
        prob = qa.Problem(problem(cols, 6000, lam, neighbours, dup=(4, 7, 13, 19, 30, 31)))
        print("column lengths", flush=True)
        assert prob.anneal_kernel(5, qa.FP64) == prob.anneal_kernel(5, qa.FP32) == "ray_solo/bytes"
        assert prob.anneal_kernel(5, qa.FP64, workgroups=256) == "ray_team"
        assert prob.anneal_kernel(5, qa.FP64, group_width=2) == "ray_team"
    wide_class = problem([1] * 700, 1400, 0.0, neighbours=0)
    wide_class.ray[:] = np.arange(700)
    assert qa.Problem(wide_class).anneal_kernel(9, qa.FP32) == "ray_solo/bytes"
    many = qa.Problem(qa.muon_scene(grid=20, sky_az=45, sky_th=12, log2_muons=22))
    assert many.anneal_kernel(300, qa.FP32) == "ray_solo/bytes"


def test_one_workgroup_per_branch_spins_in_bits():
    cols = np.zeros(130000, int)
    cols[:200] = 3
    P = problem(cols, 8000, 0.5, neighbours=2)
    P.ray[0:600:3] = 7999
    P.ray[1:600:3] = np.arange(200)
    P.ray[2:600:3] = np.arange(200, 400)
    print("spins in bits", flush=True)
    assert qa.Problem(P).anneal_kernel(3, qa.FP32) == "ray_solo/bits"


def test_integer_kernels():
    def make(n, degree, weight, signed=True):
        g = graph(n, degree, weight, signed)
        return qa.Graph(g if g.m else qa.GraphArrays(2, [0], [1], [weight]))

    print("integer kernels", flush=True)
    few, ref = set(), set()
    for n, degree, weight in GRAPHS + [(2600, 3, 2)]:
        G = make(n, degree, weight, n % 2 == 0)
        few.add(G.run_batch_kernel(5))
        if (n, degree, weight) in GRAPHS:
            ref |= {G.run_batch_kernel(R, reference=True) for R in (1, 9)}
    many = {make(n, degree, 3).run_batch_kernel(R)
            for n, degree, R in [(70, 69, 700), (150, 8, 1300), (600, 40, 1030), (900, 200, 520)]}
    assert {"int_wide/lds", "int_wide/l2"} <= few
    assert {"int_rows/lds", "int_rows/l2"} <= many
    assert ref == {"int_ref_rows/lds", "int_ref_rows/l2"}
    assert make(100, 12, 1).run_batch_kernel(1037, reference=True) == "int_ref_rows/lds"
    g = graph(90, 10)
    assert qa.Graph(qa.GraphArrays(g.n, g.eu, g.ev, np.arange(1, g.m + 1))).run_batch_kernel(5) == "int_sweep"
    assert qa.Graph(g, force_global=True).run_batch_kernel(5) == "int_sweep"


@pytest.mark.parametrize("n,degree,R,kernel,reference", [
    (2000, 100, 3584, None, "int_ref"),          # rows of 100 entries: two rounds of 7 waves against one of 14
    (1500, 375, 4608, "int_sweep", "int_ref"),
    (2000, 48, 4096, "int_sweep", "int_ref_rows/l2"),   # of 48 the two rounds are the shorter
    (1000, 100, 4608, None, "int_ref_rows/l2"),  # two workgroups of nine side by side
])
def test_integer_rules_where_rounds_decide(n, degree, R, kernel, reference):
    """On 256 CUs; each line is the measured shorter of the two."""
    G = qa.Graph(qa.er_graph(n, degree / (n - 1), 5))
    print(n, degree, R, flush=True)
    assert G.run_batch_kernel(R, reference=True) == reference
    if kernel:
        assert G.run_batch_kernel(R) == kernel
