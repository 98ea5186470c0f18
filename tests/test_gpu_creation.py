"""What a handle holds on the device from its creation: its own structure, and nothing that only
one of its anneals reads (laid out by the first such call). Sizes at which the extra arrays
would exceed what the allocator's rounding can hide, 2 MiB a buffer."""
import gc

import numpy as np
import pytest
import torch

import qublar_amd as qa

pytestmark = pytest.mark.gpu
ROUND = 2 << 20


def held(make):
    """Device bytes that make() leaves allocated."""
    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.mem_get_info()
    before = torch.cuda.mem_get_info()[0]
    handle = make()
    after = torch.cuda.mem_get_info()[0]
    handle.close()
    return before - after


def test_problem_holds_no_reference_layout():
    """8 M bits without entries: the reference trajectory's column starts would be 64 MB."""
    n = 8_000_000
    zeros = np.zeros(n + 1, np.int32)
    P = qa.ProblemArrays(zeros, np.zeros(0, np.int32), np.zeros(0, np.float32), np.zeros(1), np.ones(1), zeros,
                         np.zeros(0, np.int32), 0.5, 0.9, np.zeros(n))
    qa.Problem(qa.ProblemArrays(zeros[:9], P.ray, P.a, P.d, P.w, zeros[:9], P.nbr, 0.5, 0.9, np.zeros(8))).close()
    print(f"problem of {n} bits", flush=True)
    # per bit: position and its inverse, column and neighbour starts, fields, the repeated-ray flag,
    # the draw's counter and key, eight light neighbours; 18 buffers
    per_bit = 4 + 4 + 4 + 4 + 8 + 1 + 4 + 8 + 32
    assert held(lambda: qa.Problem(P)) <= per_bit * n + 18 * ROUND


def test_graph_holds_no_rows_of_either_engine():
    """A one-magnitude graph of 6 M edges: the 16-bit rows of the two engines would be 48 MB."""
    n, per = 32768, 184
    rng = np.random.default_rng(3)
    eu = np.repeat(np.arange(n, dtype=np.int32), per)
    ev = ((eu + 1 + np.tile(np.arange(per, dtype=np.int32), n) * 7) % n).astype(np.int32)   # 1 + 7 k < n / 2: no repeats
    g = qa.GraphArrays(n, eu, ev, rng.choice([-3, 3], len(eu)).astype(np.int32))
    qa.Graph(qa.GraphArrays(4, eu[:1], ev[:1], g.ew[:1])).close()
    print(f"graph of {len(eu)} edges", flush=True)
    m = len(eu)
    # per edge: both directions' neighbours and weights, the edge list; per vertex: starts, fields,
    # position and its inverse, class starts; 10 buffers
    assert held(lambda: qa.Graph(g)) <= (2 * 8 + 12) * m + 5 * 4 * (n + 1) + 10 * ROUND


def test_rows_of_both_engines_on_one_handle():
    """Each engine's rows are laid out by its first call, in either order, whatever ran before."""
    g = qa.er_graph(333, 0.1, 8)
    sched = qa.schedule(4.0, 0.2, 20, 3)
    a, b = qa.Graph(g), qa.Graph(g)
    print("both engines", flush=True)
    first = [a.run_batch(sched, 1, 5), a.run_batch_reference(sched, 1, 5), a.run_batch(sched, 1, 5)]
    second = [b.run_batch_reference(sched, 1, 5), b.run_batch(sched, 1, 5), b.run_batch_reference(sched, 1, 5)]
    for x, y in ((0, 1), (1, 0), (2, 1), (1, 2)):
        assert np.array_equal(first[x][0], second[y][0]) and np.array_equal(first[x][1], second[y][1])
    assert set(np.abs(g.ew)) == {1}
