"""Batched CG on systems around the 2,048 particles of a reduction chunk, each
against the FP64 oracle's solution of that system alone.

Tolerance: the solve stops at a relative residual of 1e-6 and the operator's
condition is below 4 at chi <= 2; the FMM product adds 1e-6: 5e-6.
"""
import numpy as np
import pytest

from conftest import jittered_block, rel_err

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.tensor(np.ascontiguousarray(np.asarray(a).T), dtype=torch.float32,
                        device="cuda").contiguous()


@pytest.mark.parametrize("graph_iters", [0, 2])
def test_chunk_edges(ctx, oracle, graph_iters):
    import magforce
    sizes = [2047, 1, 2048, 0, 2049, 4097, 63]
    off = np.concatenate([[0], np.cumsum(sizes)]).tolist()
    systems = [jittered_block(17, 17, 15, seed=k)[:n].astype(np.float32).astype(np.float64)
               for k, n in enumerate(sizes)]
    pos = np.concatenate(systems)
    rng = np.random.default_rng(3)
    kappas = np.linspace(0.2, 0.66, len(sizes))
    b = np.concatenate([np.tile(rng.normal(size=3), (n, 1)) for n in sizes])
    b = b.astype(np.float32).astype(np.float64)
    plan = magforce.BatchPlan(ctx, dev(pos), off, 2.0)
    res = plan.solve(kappas, dev(b), rtol=1e-6, graph_iters=graph_iters)
    assert res.stats["converged"] == 1
    x = res.x.double().cpu().numpy().T
    for s, n in enumerate(sizes):
        if n:
            want, _, _ = oracle.cg_solve(systems[s], 2.0, kappas[s], b[off[s]:off[s + 1]],
                                         rtol=1e-12)
            assert rel_err(x[off[s]:off[s + 1]], want) < 5e-6, n
