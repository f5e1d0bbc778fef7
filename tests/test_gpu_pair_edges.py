"""All-pairs field, force tensor and force at the edges of their launch shape:
targets around one wave's 32, records around the 16 of a chunk group and the 64
of a tile, chunks that end inside a tile, targets far from, inside and on the
sources, and lengths far from 1.

Tolerance: a pair takes a reciprocal square root (1 ulp, to the fifth power), a
table of the smoothed coefficients (1.5e-7) and about ten roundings, together
below 1.2e-6 of the pair; sums over mixed signs may lose a factor of a few: 5e-6.
"""
import numpy as np
import pytest

from conftest import jittered_block, random_moments, rel_err

pytestmark = pytest.mark.gpu
TOL = 5e-6


def dev(a):
    import torch
    return torch.tensor(np.ascontiguousarray(np.asarray(a).T), dtype=torch.float32,
                        device="cuda").contiguous()


def host(t):
    return t.double().cpu().numpy().T


def f32(a):
    return np.asarray(a, dtype=np.float32).astype(np.float64)


@pytest.mark.parametrize("nt,ns", [(1, 1), (1, 2000), (15, 16), (31, 17), (32, 63), (33, 65),
                                   (64, 80), (65, 129), (97, 4081), (4097, 15), (700, 1041)])
def test_field_and_tensor_vs_oracle(ctx, oracle, nt, ns):
    import magforce
    pos = f32(jittered_block(17, 17, 17, seed=nt + ns))
    t, s, m = pos[:nt], pos[-ns:], f32(random_moments(ns, seed=ns))
    got = host(magforce.field_allpairs(ctx, dev(t), dev(s), dev(m), 2.0, hconst=[1, 2, 3]))
    assert rel_err(got, oracle.field_allpairs(t, s, m, 2.0, hconst=[1, 2, 3])) < TOL
    want = oracle.hessian_allpairs(t, s, m, 2.0)
    six = host(magforce.hessian_allpairs(ctx, dev(t), dev(s), dev(m), 2.0))
    sym = np.stack([want[:, 0, 0], want[:, 1, 1], want[:, 2, 2], want[:, 0, 1], want[:, 0, 2],
                    want[:, 1, 2]], 1)
    assert rel_err(six, sym) < TOL


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 64, 65, 257, 1025])
def test_plan_products_vs_oracle(ctx, oracle, n):
    """Field and force on one set; with n > 64 one particle appears twice."""
    import magforce
    pos = f32(jittered_block(11, 11, 11, seed=n))[:n]
    if n > 64:
        pos[7] = pos[40]
    m = f32(random_moments(n, seed=n + 1))
    plan = magforce.Plan(ctx, dev(pos), 2.0)
    assert rel_err(host(plan.field(dev(m))), oracle.field_allpairs(pos, pos, m, 2.0)) < TOL
    want = oracle.force_allpairs(pos, m, 2.0)
    got = host(plan.force(dev(m)))
    assert np.array_equal(got, want) if n == 1 else rel_err(got, want) < TOL


@pytest.mark.parametrize("scale", [1e-3, 50.0])
def test_other_lengths(ctx, oracle, scale):
    """The near tables hold h = 1 and are scaled by powers of h: micrometre
    droplets given in millimetres and the reverse."""
    import magforce
    pos, m = f32(scale * jittered_block(6, 7, 5, seed=4)), f32(random_moments(210, seed=5))
    plan = magforce.Plan(ctx, dev(pos), 2.0 * scale)
    h = float(np.float32(2.0 * scale))
    assert rel_err(host(plan.field(dev(m))), oracle.field_allpairs(pos, pos, m, h)) < TOL
    assert rel_err(host(plan.force(dev(m))), oracle.force_allpairs(pos, m, h)) < TOL


@pytest.mark.parametrize("n", [1, 63, 65, 300, 1025])
@pytest.mark.parametrize("method", ["cg", "gmres"])
@pytest.mark.parametrize("warm", [False, True])
def test_solve_edges_vs_oracle(ctx, oracle, n, method, warm):
    """The fused CG and the device-side Gram-Schmidt at small sizes, from zero
    and from a start; CG and GMRES stop at 1e-6, on a system whose condition
    number is at most 2."""
    import magforce
    pos = f32(jittered_block(11, 11, 11, seed=n))[:n]
    b = f32(random_moments(n, seed=n + 2))
    plan = magforce.Plan(ctx, dev(pos), 2.0)
    x0 = dev(f32(random_moments(n, seed=3))) if warm else None
    code = magforce.SOLVE_CG if method == "cg" else magforce.SOLVE_GMRES
    res = plan.solve(0.5, dev(b), x0=x0, method=code, rtol=1e-6)
    assert res.stats["converged"] == 1 and res.stats["rel_residual"] <= 1e-6
    want, _, _ = oracle.cg_solve(pos, 2.0, 0.5, b, rtol=1e-12)
    assert rel_err(host(res.x), want) < TOL


@pytest.mark.parametrize("ns", [1, 16, 17, 63, 64, 65, 127, 128, 129])
@pytest.mark.parametrize("nt", [1, 33, 1000])
def test_few_sources_vs_oracle(ctx, oracle, nt, ns):
    """Around the largest source count that one launch takes; targets on, near and far from the
    sources, and outputs that overwrite the targets and the sources, which get the same
    values as separate ones."""
    import ctypes
    import magforce
    import torch
    pos = f32(jittered_block(11, 11, 11, seed=nt + ns))
    t, s, m = pos[:nt], pos[max(nt - ns // 2, 0):][:ns], f32(random_moments(ns, seed=ns))
    dt, ds, dm = dev(t), dev(s), dev(m)
    got = magforce.field_allpairs(ctx, dt, ds, dm, 2.0, hconst=[1, 2, 3])
    assert rel_err(host(got), oracle.field_allpairs(t, s, m, 2.0, hconst=[1, 2, 3])) < TOL
    want = oracle.hessian_allpairs(t, s, m, 2.0).transpose(0, 2, 1).reshape(nt, 9)
    nine = host(magforce.hessian_allpairs9(ctx, dt, ds, dm, 2.0))
    assert rel_err(nine, want) < TOL
    # one buffer holds targets or sources first, and then the result
    for over in ("targets", "sources"):
        buf = torch.zeros((3, max(nt, ns)), device="cuda")
        first = dt if over == "targets" else ds
        buf[:, :first.shape[1]] = first
        row = [buf[k].data_ptr() for k in range(3)]
        tp = row if over == "targets" else [dt[k].data_ptr() for k in range(3)]
        sp = row if over == "sources" else [ds[k].data_ptr() for k in range(3)]
        p = [ctypes.c_void_p(v) for v in (*tp, *sp, *[dm[k].data_ptr() for k in range(3)], *row)]
        rc = magforce.lib().mf_field_allpairs(ctx.h, nt, *p[:3], ns, *p[3:9], 2.0,
                                              (ctypes.c_float * 3)(1, 2, 3), *p[9:])
        torch.cuda.synchronize()
        assert rc == magforce.MF_OK
        assert rel_err(host(buf[:, :nt]), host(got)) < 2 * TOL  # each within TOL of the oracle


@pytest.mark.parametrize("n", [1, 65, 700, 4096, 4999])
@pytest.mark.parametrize("maxit", [1, 3, 100])
def test_product_launched_ahead(oracle, n, maxit):
    """A CG solve launches the next product before it knows the residual, and with kernel
    timing on it waits first: the same solution, counts and residual bit for bit, from
    solves that converge and that maxit stops, one after the other on one context."""
    import magforce
    pos = f32(jittered_block(18, 18, 18, seed=n))[:n]
    b = f32(random_moments(n, seed=n + 5))
    out = []
    for timing in (False, True, False):
        c = magforce.Context(0)
        plan = magforce.Plan(c, dev(pos), 2.0)
        c.enable_timing(timing)
        res = [plan.solve(0.5, dev(b), rtol=rtol, maxit=maxit) for rtol in (1e-6, 1e-3)]
        out.append([(host(r.x), {k: r.stats[k] for k in ("matvecs", "iterations", "rel_residual",
                                                         "converged")}) for r in res])
        plan.close()
        c.close()
    for other in out[1:]:
        for (x, st), (y, su) in zip(out[0], other):
            assert np.array_equal(x, y) and st == su, (st, su)
    assert all(st["matvecs"] <= maxit for _, st in out[0])
    if maxit == 100:
        want, _, _ = oracle.cg_solve(pos, 2.0, 0.5, b, rtol=1e-12)
        assert rel_err(out[0][0][0], want) < TOL
