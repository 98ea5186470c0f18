"""Device memory of the one-workgroup-per-branch anneal with many branches: its spins take a bit
each, as the grouped layout's do, and once more as the masks of 16 branches that the read-out
and the energies share."""
import gc

import numpy as np
import pytest
import torch

import qublar_amd as qa
from test_gpu_solo import problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,kernel", [(100000, "ray_solo/bytes"), (130000, "ray_solo/bits")])
def test_many_branches_take_a_bit_a_spin(n, kernel):
    R, rays = 2000, 8000
    cols = np.zeros(n, int)
    cols[:200] = 3
    P = problem(cols, rays, 0.5, neighbours=2)
    P.ray[0:600:3] = rays - 1   # one ray of 200 bits: 200 classes
    P.ray[1:600:3] = np.arange(200)
    P.ray[2:600:3] = np.arange(200, 400)
    prob = qa.Problem(P)
    assert prob.anneal_kernel(R, qa.FP32) == kernel
    print(f"{R} branches of {n} bits, {kernel}", flush=True)
    sched = qa.schedule(4.0, 0.5, 2, 0)
    few = prob.anneal_branches(sched, 17, 0, qa.FP32, sweeps_per_launch=1)   # the plan, and what no branch adds to
    gc.collect()
    before = torch.cuda.mem_get_info()[0]
    many = prob.anneal_branches(sched, R, 0, qa.FP32, branches=False, sweeps_per_launch=1)
    held = before - torch.cuda.mem_get_info()[0]
    # a branch: its spins twice, its FP32 residuals, a double per 16 rays and bits (the energies'
    # partial sums), its energies; the buffers rounded to 2 MiB
    branch = 2 * n / 8 + 4 * (rays + 1) + 8 * ((rays + n) / 16 + 2) + 16
    assert held <= branch * (R + 16) + 8 * (2 << 20)
    assert np.array_equal(few["energy"], many["energy"][:17])
