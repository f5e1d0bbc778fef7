"""FMM plans of particle counts around a wave, a workgroup and the size up to which the plan
build's scans take one workgroup, each on a set whose leaves are nearly as many as its
particles (so the scans over leaves and blocks meet those sizes too).

Tolerance: p = 10 truncation with random moments stays below 5e-6 of the field; twice that.
"""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 8191, 8192, 8193, 16383, 16384, 16385])
def test_field_vs_fp64(ctx, n):
    import magforce
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    pos = 5.0 * max(1.0, n ** (1.0 / 3.0)) * torch.rand((3, n), generator=g, device="cuda")
    m = 0.5 * torch.randn((3, n), generator=g, device="cuda")
    plan = magforce.Plan(ctx, pos, 2.0, mode=magforce.MODE_FMM)
    got = plan.field(m).double().cpu().numpy()
    plan.update_positions(pos)
    assert np.array_equal(got, plan.field(m).double().cpu().numpy())
    want = magforce.field_allpairs_f64(ctx, pos.double(), pos.double(), m.double(), 2.0)
    assert rel_err(got.T, want.cpu().numpy().T) < 1e-5
    plan.close()
