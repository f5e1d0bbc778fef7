"""Products of one record set on itself at and above the size from which every
unordered pair is evaluated once: whole and partial tiles, groups and an empty
last group, coincident particles in different tiles, the conjugate-gradient
form, and a size whose walk takes two passes.

Tolerance: as for the directed all-pairs kernels (a pair's roundings and table
below 1.2e-6, sums over mixed signs may lose a factor of a few): 5e-6.
"""
import numpy as np
import pytest

from conftest import jittered_block, random_moments, rel_err

pytestmark = pytest.mark.gpu
TOL = 5e-6


def dev(a, dtype=None):
    import torch
    return torch.tensor(np.ascontiguousarray(np.asarray(a).T), dtype=dtype or torch.float32,
                        device="cuda").contiguous()


def host(t):
    return t.double().cpu().numpy().T


def f32(a):
    return np.asarray(a, dtype=np.float32).astype(np.float64)


def cloud(n, seed, shuffle):
    pos = jittered_block(18, 18, -(-n // 324), seed=seed)[:n]
    if shuffle:
        pos = pos[np.random.default_rng(seed).permutation(n)]
    return f32(pos)


@pytest.mark.parametrize("n,h,shuffle", [
    (4095, 2.0, False),  # directed
    (4096, 2.0, False),  # 16 groups and an empty one
    (4097, 0.7, False),  # 17 groups, the last one a single particle
    (4352, 2.0, True),   # 17 whole groups
    (4353, 2.0, False),  # 18 groups and an empty one
    (4929, 3.0, True),   # last tile of one particle, last group of two tiles
])
def test_products_vs_oracle(ctx, oracle, n, h, shuffle):
    import magforce
    pos = cloud(n, n, shuffle)
    pos[n - 2] = pos[3]  # coincident, in the first and the last tiles
    m = f32(random_moments(n, seed=n + 1))
    plan = magforce.Plan(ctx, dev(pos), h)
    got = host(plan.field(dev(m), hconst=[0.5, -1.0, 2.0]))
    assert rel_err(got, oracle.field_allpairs(pos, pos, m, h, hconst=[0.5, -1.0, 2.0])) < TOL
    F = host(plan.force(dev(m)))
    assert rel_err(F, oracle.force_allpairs(pos, m, h)) < TOL
    # the same sums on a second call
    assert np.array_equal(F, host(plan.force(dev(m))))


def test_solve_residual(ctx, oracle):
    import magforce
    n = 4300
    pos = cloud(n, 5, False)
    plan = magforce.Plan(ctx, dev(pos), 2.0)
    b = np.tile([0.0, 0.3, 1.0], (n, 1))
    res = plan.solve(0.5, dev(b), rtol=1e-6)
    x = host(res.x)
    r = b - (x - 0.5 * oracle.field_allpairs(pos, pos, x, 2.0))
    assert np.linalg.norm(r) < 5e-6 * np.linalg.norm(b)


def test_two_passes_vs_fp64(ctx):
    import magforce
    import torch
    n, k = 231_001, 1500
    rng = np.random.default_rng(9)
    pos = f32(rng.uniform(0.0, 90.0, size=(n, 3)))
    m = f32(random_moments(n, seed=10))
    idx = np.sort(rng.choice(n, size=k, replace=False))
    idx[-1] = n - 1
    plan = magforce.Plan(ctx, dev(pos), 2.0)
    p64, m64 = dev(pos, torch.float64), dev(m, torch.float64)
    want = host(magforce.field_allpairs_f64(ctx, dev(pos[idx], torch.float64), p64, m64, 2.0))
    assert rel_err(host(plan.field(dev(m)))[idx], want) < TOL
    F = host(plan.force(dev(m)))
    want = host(magforce.force_subset_f64(ctx, p64, m64, 2.0, torch.tensor(idx, device="cuda")))
    assert rel_err(F[idx], want) < TOL
