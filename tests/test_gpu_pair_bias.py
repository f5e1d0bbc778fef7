"""The systematic error of the all-pairs field: equal moments on jittered lattices, the mean
over the particles of the error along the moments.  A coefficient that is rounded the same
way for all near pairs shows here long before it shows in a norm, and a solve's solution
and force inherit it.

Tolerance: v_rsq_f32 is low by 7.4e-9 in the mean, so the far pairs' r^-3 are low by 2.2e-8
of their part of the field; the near coefficients allow for it, and all other roundings
are as often up as down: 2.5e-8 of the field.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.tensor(np.ascontiguousarray(np.asarray(a).T), dtype=torch.float32,
                        device="cuda").contiguous()


@pytest.mark.parametrize("h", [2.0, 1.5, 1.0])
@pytest.mark.parametrize("shape", [(7, 8, 6), (12, 10, 9)])
def test_equal_moments(ctx, oracle, shape, h):
    import magforce
    bias = []
    for seed in range(8):
        rng = np.random.default_rng(seed)
        pos = np.stack(np.meshgrid(*[np.arange(k) for k in shape], indexing="ij"), -1).reshape(-1, 3)
        pos = (pos + rng.uniform(-0.1, 0.1, pos.shape)).astype(np.float32).astype(np.float64)
        m = np.tile(np.float32([0.0, 0.0, 0.35]).astype(np.float64), (len(pos), 1))
        plan = magforce.Plan(ctx, dev(pos), h)
        got = plan.field(dev(m)).double().cpu().numpy().T
        plan.close()
        want = oracle.field_allpairs(pos, pos, m, h)
        bias.append(np.mean((got - want)[:, 2]) / np.mean(np.linalg.norm(want, axis=1)))
    print(f"{len(pos)} particles, h = {h}: {np.mean(bias):+.1e}")
    assert abs(np.mean(bias)) < 2.5e-8
