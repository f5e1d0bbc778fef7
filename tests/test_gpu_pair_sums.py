"""The force of equal moments on a jittered lattice, whose terms nearly cancel, with every pair
evaluated once against the same with the directed kernels (taken where no slots can be had).

Tolerance: the directed kernels hold 64 terms in one FP32 chain, the pair-once kernels at
most 64 for either particle of a pair, with more partial sums: their errors against FP64,
over 6 sets, may differ by the scatter of a few percent: 5 %.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h", [2.0, 1.5])
def test_error_beside_directed(h):
    import magforce
    import torch
    n3 = (20, 20, 30)
    errors = []
    for refuse in (False, True):
        c = magforce.Context(0)
        e = []
        for seed in range(6):
            g = torch.Generator(device="cuda").manual_seed(seed)
            pos = torch.cartesian_prod(*[torch.arange(k, device="cuda") for k in n3]).t().float()
            pos = (pos + 0.2 * torch.rand(pos.shape, generator=g, device="cuda") - 0.1).contiguous()
            m = 0.03 * torch.randn(pos.shape, generator=g, device="cuda")
            m[2] += 0.35
            plan = magforce.Plan(c, pos, h)
            # the slots of 12,000 particles take 15 MB, the directed kernels' chunks 7
            magforce.set_alloc_hook((lambda size: size > 10 << 20) if refuse else None)
            try:
                got = plan.force(m).double()
            finally:
                magforce.set_alloc_hook(None)
            plan.close()
            want = magforce.force_allpairs_f64(c, pos.double(), m.double(), h)
            e.append(float((got - want).norm() / want.norm()))
        c.close()
        errors.append(np.exp(np.mean(np.log(e))))
    print(f"h = {h}: pairs once {errors[0]:.3e}, directed {errors[1]:.3e}")
    assert errors[0] < 1.05 * errors[1]
