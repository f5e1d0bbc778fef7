"""A batched solve whose near field takes several passes over its places (no allocation beyond
200 MiB succeeds), with systems that converge at different iterations, against the same
solve with one pass.

Tolerance: both solves stop at a relative residual of 1e-6, and the operator's condition is
below 4 at these kappas: 5e-6.
"""
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph_iters", [0, 2])
def test_solve_in_passes(graph_iters):
    import magforce
    import torch
    g = torch.Generator(device="cuda").manual_seed(2)
    blocks, off = [], [0]
    for nx, ny, nz in ((96, 96, 40), (64, 64, 8), (96, 90, 40)):
        k = torch.arange(nx * ny * nz, device="cuda")
        p = torch.stack([k % nx, (k // nx) % ny, k // (nx * ny)]).float()
        blocks.append(p + 0.2 * torch.rand(p.shape, generator=g, device="cuda") - 0.1)
        off.append(off[-1] + p.shape[1])
    pos = torch.cat(blocks, 1).contiguous()
    b = magforce.uniform_field(off[-1], [0.0, 0.3, 1.0])
    kappas, out, refused = [0.05, 0.3, 0.66], [], []
    for limit in (1 << 62, 200 << 20):
        c = magforce.Context(0)
        magforce.set_alloc_hook(lambda n: n > limit and (refused.append(n) or True))
        try:
            plan = magforce.BatchPlan(c, pos, off, 2.0)
            res = plan.solve(kappas, b, rtol=1e-6, graph_iters=graph_iters)
            F = plan.force(res.x)
            plan.close()
        finally:
            magforce.set_alloc_hook(None)
        assert res.stats["converged"] == 1
        out.append((res.x.cpu().numpy(), F.cpu().numpy()))
        c.close()
    assert refused
    for s in range(3):
        own = slice(off[s], off[s + 1])
        for a, w in zip(out[1], out[0]):
            assert rel_err(a[:, own], w[:, own]) < 5e-6, s
