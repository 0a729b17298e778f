"""The second population array of 2-D runs of several steps per launch is made
only from memory that is plentifully free: where it would take more than an
eighth of what the caller could still allocate, the run leaves that memory
alone and gives the same fields."""
import numpy as np
import pytest
import torch

import _pkg
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


def free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_second_array_leaves_the_callers_memory():
    L = _pkg.load()
    ni, nj = 3001, 2003
    state = (ni * nj + 2047) // 2048 * 2048 * 9 * 2 * 8
    kw = dict(dims=2, ni=ni, nj=nj, nsubs=2, tau=(0.8, 0.75), gaccel=(1e-5, 0, 0, 0, 0, 0))
    mask = np.zeros((nj, ni), np.uint8)
    c0 = np.random.default_rng(11).random(ni * nj)
    a = L.Lattice(mask=mask, **kw)
    a.init_rest(c0)
    torch.cuda.init()
    hog = torch.empty(free() - 6 * state, dtype=torch.uint8, device="cuda")
    a.run(1, write_last=False)  # the step kernels are loaded
    a.time = 0
    a.init_rest(c0)
    before = free()
    say(f"case scarce memory: state {state >> 20} MiB, free {before >> 20} MiB")
    a.run(9)
    taken = before - free()
    say(f"taken {taken >> 20} MiB")
    assert taken < state // 2
    scarce = a.mv(0), a.mv(1)
    del hog
    torch.cuda.empty_cache()
    # plenty is free: the array is made for the next geometry, with the same fields
    a.set_solids(mask)
    a.time = 0
    a.init_rest(c0)
    before = free()
    a.run(9)
    assert before - free() > state // 2
    for x, y in zip(scarce, (a.mv(0), a.mv(1))):
        assert all(np.array_equal(p, q) for p, q in zip(x, y))
    a.close()

def test_short_runs_take_no_memory():
    """two steps without row conditions are launched one by one: a program
    that runs no more at a time pays for no second array"""
    L = _pkg.load()
    ni, nj = 1201, 1103
    state = ni * nj * 9 * 2 * 8
    a = L.Lattice(mask=np.zeros((nj, ni), np.uint8), dims=2, ni=ni, nj=nj, nsubs=2, tau=(0.8, 0.75))
    a.init_rest()
    a.step()
    a.step()
    before = free()
    for _ in range(3):
        a.run(2)
    assert before - free() < state // 2
    a.run(4)
    assert before - free() > state // 2
    a.close()
