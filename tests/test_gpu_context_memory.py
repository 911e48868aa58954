"""Device memory that a context keeps from one Schwarz preconditioner to the
next: bounded, given back on request, when an allocation of the library finds
no room and when the context is closed, without touching what is in use."""
import ctypes

import numpy as np
import pytest
import torch

import aboria_amd as ab
from aboria_amd import _capi as C

pytestmark = pytest.mark.gpu

ABH_ERR_OUT_OF_MEMORY = 3
SLACK = 64 << 20  # small buffers and the allocator's granularity


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def setup(n, leaf):
    rng = np.random.default_rng(n)
    c = ab.Context(0)
    cl = ab.CellListOrdered(c, [0.0] * 2, [1.0] * 2, [False] * 2, leaf)
    cl.update_positions(torch.tensor(rng.random((n, 2)), device="cuda"))
    b = torch.tensor(rng.standard_normal(n), device="cuda")
    return c, cl, b


def make(c, cl):
    return ab.SchwartzPreconditioner(c, cl, ab.Kernel.gaussian(0.02), 0.1, 0.1)


def test_large_domain_leaves_no_work_memory():
    """One domain of 20,500 points: 3.4 GB of work memory, more than a context
    keeps; the preconditioner holds its inverse alone."""
    c, cl, _ = setup(20_500, 100_000.0)
    before = free_bytes()
    sw = make(c, cl)
    held = before - free_bytes()
    assert held <= sw.info["factor_bytes"] + SLACK
    del sw
    assert before - free_bytes() <= 4 * 2 ** 30 + SLACK  # its inverse may stay
    c.trim()
    assert before - free_bytes() <= SLACK
    c.close()


def test_kept_memory_is_given_back():
    c, cl, b = setup(40_000, 64.0)
    before = free_bytes()
    ref = make(c, cl).solve(b)
    assert 1 << 30 <= before - free_bytes() <= 7 * 2 ** 30 + SLACK
    c.trim()
    assert before - free_bytes() <= SLACK
    sw = make(c, cl)
    assert torch.equal(sw.solve(b), ref)
    # an allocation that cannot succeed gives back what is idle, not what is used
    p = ctypes.c_void_p()
    assert C.lib().abh_malloc(c.handle, ctypes.byref(p), 1 << 50) == ABH_ERR_OUT_OF_MEMORY
    assert before - free_bytes() <= sw.info["factor_bytes"] + SLACK
    assert torch.equal(sw.solve(b), ref)
    other = make(c, cl)  # work memory again, and a second inverse
    assert torch.equal(other.solve(b), ref)
    del other
    # closed, the context keeps nothing for preconditioners that cannot follow
    c.close()
    assert before - free_bytes() <= sw.info["factor_bytes"] + SLACK
    assert torch.equal(sw.solve(b), ref)
    del sw
