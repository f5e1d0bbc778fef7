"""FMM near field with every unordered pair of leaf blocks evaluated once: leaves
whose heads and tails have every width around the 16 lanes of a row, the 32 of a
tail and the 64 of a pass, next to each other and to empty ones, and a system
whose places are walked in two passes.

Tolerance: p = 10 truncation with random moments stays below 5e-6 of the field
on lattices and random layers; twice that is allowed.
"""
import numpy as np
import pytest

from conftest import random_moments, rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5


def dev(a, dtype=None):
    import torch
    return torch.tensor(np.ascontiguousarray(np.asarray(a).T), dtype=dtype or torch.float32,
                        device="cuda").contiguous()


def host(t):
    return t.double().cpu().numpy().T


WIDTHS = [1, 2, 15, 16, 17, 0, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80, 81, 95, 96, 97, 127, 128, 129,
          160, 161, 5, 0, 190]


@pytest.mark.parametrize("cells,seed", [(2, 0), (4, 1), (4, 2), (5, 3)])
def test_leaf_widths_vs_oracle(ctx, oracle, cells, seed):
    """cells^3 leaves of side 4 (h = 2) with particle counts drawn from WIDTHS; two corner
    particles pin the leaf grid.  Coincident particles in one leaf and across its blocks."""
    import magforce
    rng = np.random.default_rng(seed)
    grid = 1 << (cells - 1).bit_length()
    pos = [np.array([[0.05, 0.05, 0.05], [4.0 * grid - 0.05] * 3])]
    for k, ijk in enumerate(np.ndindex(cells, cells, cells)):
        w = WIDTHS[(k * 5 + seed) % len(WIDTHS)]
        pos.append(4.0 * np.array(ijk) + rng.uniform(0.1, 3.9, size=(w, 3)))
    pos = np.concatenate(pos)
    pos[-1] = pos[-3]
    pos = pos.astype(np.float32).astype(np.float64)
    m = random_moments(len(pos), seed=seed).astype(np.float32).astype(np.float64)
    plan = magforce.Plan(ctx, dev(pos), 2.0, mode=magforce.MODE_FMM)
    got = host(plan.field(dev(m), hconst=[0.5, -1.0, 2.0]))
    want = oracle.field_allpairs(pos, pos, m, 2.0, hconst=[0.5, -1.0, 2.0])
    F = host(plan.force(dev(m)))
    eg, ef = rel_err(got, want), rel_err(F, oracle.force_allpairs(pos, m, 2.0))
    print(f"{len(pos)} particles, {plan.info()['leaves']} leaves: field {eg:.2e} force {ef:.2e}")
    assert eg < TOL and ef < TOL
    assert np.array_equal(F, host(plan.force(dev(m))))  # the same sums again


def test_two_passes_vs_fp64(ctx):
    """15 million particles: the force's places exceed one pass's buffer."""
    import magforce
    import torch
    g = torch.Generator(device="cuda").manual_seed(4)
    nx, ny, nz = 256, 256, 230
    k = torch.arange(nx * ny * nz, device="cuda")
    pos = torch.stack([k % nx, (k // nx) % ny, k // (nx * ny)]).float()
    pos += 0.2 * torch.rand(pos.shape, generator=g, device="cuda") - 0.1
    m = 0.5 * torch.randn(pos.shape, generator=g, device="cuda")
    idx = torch.randint(0, pos.shape[1], (256,), generator=g, device="cuda")
    plan = magforce.Plan(ctx, pos, 2.0, mode=magforce.MODE_FMM)
    p64, m64 = pos.double(), m.double()
    want = magforce.field_allpairs_f64(ctx, p64[:, idx].contiguous(), p64, m64, 2.0)
    assert rel_err(host(plan.field(m)[:, idx]), host(want)) < TOL
    want = magforce.force_subset_f64(ctx, p64, m64, 2.0, idx)
    assert rel_err(host(plan.force(m)[:, idx]), host(want)) < TOL


def test_passes_where_memory_is_short():
    """737,280 particles where no allocation beyond 320 MiB succeeds: the force's places (about
    600 MiB) are walked in more passes.  The same FP32 block sums are added in FP64 in
    another order, so results differ by at most the final rounding."""
    import magforce
    import torch
    g = torch.Generator(device="cuda").manual_seed(8)
    nx, ny, nz = 96, 96, 80
    k = torch.arange(nx * ny * nz, device="cuda")
    pos = torch.stack([k % nx, (k // nx) % ny, k // (nx * ny)]).float()
    pos += 0.2 * torch.rand(pos.shape, generator=g, device="cuda") - 0.1
    m = 0.5 * torch.randn(pos.shape, generator=g, device="cuda")
    refused, out = [], []
    for limit in (1 << 62, 320 << 20):
        c = magforce.Context(0)
        magforce.set_alloc_hook(lambda n: n > limit and (refused.append(n) or True))
        try:
            plan = magforce.Plan(c, pos, 2.0, mode=magforce.MODE_FMM)
            out.append((host(plan.field(m)), host(plan.force(m))))
            plan.close()
        finally:
            magforce.set_alloc_hook(None)
        c.close()
    print(f"refused {refused}")
    assert refused
    for a, b in zip(*out):
        assert rel_err(b, a) < 2.0 ** -23
