"""FMM plans where memory is short in all, not for single buffers: the near field's place
buffer takes what the plan's other buffers and its products' leave, and its passes get
smaller where that is not enough.

Tolerance: the same FP32 block sums are added in FP64 in another order, so results differ
by at most the final rounding.
"""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def host(t):
    return t.double().cpu().numpy().T


def products(pos, m, most):
    """Field and force on a fresh context that may allocate `most` bytes; the accepted sizes
    of the plan build, and the sizes asked for by the products."""
    import magforce
    taken, asked = [], []

    def hook(n):
        if sum(taken) + n > most:
            return True
        taken.append(n)
        return False

    c = magforce.Context(0)
    magforce.set_alloc_hook(hook)
    try:
        plan = magforce.Plan(c, pos, 2.0, mode=magforce.MODE_FMM)
        magforce.set_alloc_hook(lambda n: asked.append(n) and False)
        out = host(plan.field(m)), host(plan.force(m))
        plan.close()
    finally:
        magforce.set_alloc_hook(None)
    c.close()
    return out, taken, asked


def test_places_take_what_the_rest_leaves():
    """737,280 particles; the force's places are the largest buffer by far.  With 5/8 of it
    fewer bytes in all, everything else still has to be had."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(8)
    nx, ny, nz = 96, 96, 80
    k = torch.arange(nx * ny * nz, device="cuda")
    pos = torch.stack([k % nx, (k // nx) % ny, k // (nx * ny)]).float()
    pos += 0.2 * torch.rand(pos.shape, generator=g, device="cuda") - 0.1
    m = 0.5 * torch.randn(pos.shape, generator=g, device="cuda")
    want, taken, asked = products(pos, m, 1 << 62)
    assert not asked
    big = max(taken)
    assert big > 512 << 20  # halved at least twice before the smallest size is reached
    got, taken, asked = products(pos, m, sum(taken) - 5 * big // 8)
    print(f"largest {big}, then {max(taken)}")
    assert max(taken) < big and not asked
    for a, b in zip(got, want):
        assert rel_err(a, b) < 2.0 ** -23
