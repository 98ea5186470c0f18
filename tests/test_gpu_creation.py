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
