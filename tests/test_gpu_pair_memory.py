"""All-pairs products of a set on itself where the slots of all group distances cannot be had:
the walk takes more passes over fewer slots, and a size that was refused is not asked for
again by the next product.

Tolerance: as for the products in one or two passes (test_gpu_pair_once.py): 5e-6.
"""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 5e-6


def host(t):
    return t.double().cpu().numpy().T


@pytest.mark.parametrize("n,limit,passes", [
    (100_001, 300 << 20, True),  # 570 MB of slots, halved twice: several passes
    (4500, 5 << 20, False),      # 5.3 MB and too few for passes: the directed kernels' 3.2 MB
])
def test_slots_refused(n, limit, passes):
    import magforce
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    pos = 1.05 * n ** (1.0 / 3.0) * torch.rand((3, n), generator=g, device="cuda")
    m = 0.5 * torch.randn((3, n), generator=g, device="cuda")
    idx = torch.randperm(n, generator=g, device="cuda")[:500]
    idx[-1] = n - 1
    refused, taken = [], []

    def hook(size):
        (refused if size > limit else taken).append(size)
        return size > limit

    c = magforce.Context(0)
    plan = magforce.Plan(c, pos, 2.0)
    magforce.set_alloc_hook(hook)
    try:
        field, force = plan.field(m), plan.force(m)
        asked = len(refused) + len(taken)
        again = plan.field(m), plan.force(m)
    finally:
        magforce.set_alloc_hook(None)
    print(f"refused {refused}, taken {taken}")
    assert refused and len(refused) + len(taken) == asked
    assert (max(taken) > 100 << 20) == passes  # the directed kernels' chunks take 57 MB
    assert torch.equal(field, again[0]) and torch.equal(force, again[1])
    p64, m64 = pos.double(), m.double()
    want = magforce.field_allpairs_f64(c, p64[:, idx].contiguous(), p64, m64, 2.0)
    assert rel_err(host(field[:, idx]), host(want)) < TOL
    want = magforce.force_subset_f64(c, p64, m64, 2.0, idx)
    assert rel_err(host(force[:, idx]), host(want)) < TOL
    plan.close()
    c.close()
