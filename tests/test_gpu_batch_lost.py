"""A batch in which one droplet holds a NaN (in its right-hand side, or in its start):
the batch is not reported as converged, and the other droplets are solved as ever, each
against the FP64 oracle's solution of that droplet alone.

Tolerance: the solve stops at a relative residual of 1e-6 and the operator's
condition is below 4 at chi <= 2; the FMM product adds 1e-6: 5e-6.
"""
import math

import numpy as np
import pytest

from conftest import jittered_block, rel_err

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.tensor(np.ascontiguousarray(np.asarray(a).T), dtype=torch.float32,
                        device="cuda").contiguous()


@pytest.mark.parametrize("graph_iters", [0, 2])
@pytest.mark.parametrize("where", ["b", "x0"])
def test_nan_in_one_system(ctx, oracle, where, graph_iters):
    import magforce
    sizes, bad = [900, 700, 1200], 1
    off = np.concatenate([[0], np.cumsum(sizes)]).tolist()
    systems = [jittered_block(11, 11, 10, seed=k)[:n].astype(np.float32).astype(np.float64)
               for k, n in enumerate(sizes)]
    b = np.tile([0.0, 0.3, 1.0], (off[-1], 1)).astype(np.float32).astype(np.float64)
    x0 = np.zeros_like(b)
    (b if where == "b" else x0)[off[bad] + 5, 2] = np.nan
    kappas = [0.3, 0.5, 0.6]
    plan = magforce.BatchPlan(ctx, dev(np.concatenate(systems)), off, 2.0)
    res = plan.solve(kappas, dev(b), x0=None if where == "b" else dev(x0), rtol=1e-6,
                     graph_iters=graph_iters)
    each = res.stats["sys_rel_residual"]
    assert res.stats["converged"] == 0 and math.isnan(res.stats["rel_residual"])
    assert math.isnan(each[bad])
    x = res.x.double().cpu().numpy().T
    for s in (0, 2):
        own = slice(off[s], off[s + 1])
        want, _, _ = oracle.cg_solve(systems[s], 2.0, kappas[s], b[own], rtol=1e-12)
        assert each[s] <= 1e-6 and rel_err(x[own], want) < 5e-6, s
