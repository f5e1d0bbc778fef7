"""FMM products whose near field runs with one, two, four or eight waves per
leaf (by the number of leaves) and whose M2L runs with one or many parts per
tile, against the GPU FP64 all-pairs sums (themselves pinned to the oracle).

A uniform cloud of about three particles per leaf, and crowded leaves of 63 to
200 particles, so that full 64-target passes and remainders of every width
meet streams that do not divide by the wave count.

Tolerance: p = 10 truncation on a random layer of 12 particles per leaf is
2.1e-6 of the field.  Near pairs' share of the field falls with the density, so
the ratio grows as its inverse square root: 4.2e-6 at three per leaf, and twice
that is allowed.  p = 6 takes the truncation ratio of the two orders' own
bounds (5e-4 / 2e-6).
"""
import numpy as np
import pytest

from conftest import random_moments, rel_err

pytestmark = pytest.mark.gpu
TOL = {10: 1e-5, 6: 2.5e-3}


def dev(a, dtype=None):
    import torch
    return torch.tensor(np.ascontiguousarray(np.asarray(a).T), dtype=dtype or torch.float32,
                        device="cuda").contiguous()


def host(t):
    return t.double().cpu().numpy().T


def cloud(cells, seed):
    rng = np.random.default_rng(seed)
    side = 4.0 * np.asarray(cells, dtype=float)
    pos = [rng.uniform(0.0, 1.0, size=(3 * int(np.prod(cells)), 3)) * side]
    for k, n in enumerate((63, 64, 65, 127, 128, 129, 200)):
        corner = 4.0 * np.array([k % cells[0], (3 * k) % cells[1], k % cells[2]])
        pos.append(corner + rng.uniform(0.2, 3.8, size=(n, 3)))
    return np.concatenate(pos).astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("cells,leaves,order,prec", [
    ((3, 3, 3), (20, 64), 10, "bf16x3"),            # eight waves, shallow tree
    ((12, 12, 12), (1500, 3500), 10, "bf16x3"),     # eight waves, many parts
    ((12, 12, 12), (1500, 3500), 6, "fp32"),
    ((12, 12, 12), (1500, 3500), 10, "fp32"),
    ((22, 21, 19), (7300, 14000), 10, "bf16x3"),    # four waves, a few parts
    ((27, 26, 25), (14500, 28000), 6, "bf16x3"),    # two waves
    ((34, 32, 31), (29000, 60000), 10, "bf16x3"),   # one wave, one part
])
def test_products_vs_fp64(ctx, cells, leaves, order, prec):
    import magforce
    import torch
    pos = cloud(cells, seed=cells[0])
    n = pos.shape[0]
    m = random_moments(n, seed=n).astype(np.float32).astype(np.float64)
    code = {"fp32": magforce.M2L_FP32, "bf16x3": magforce.M2L_BF16X3}[prec]
    plan = magforce.Plan(ctx, dev(pos), 2.0, mode=magforce.MODE_FMM, order=order,
                         m2l_precision=code)
    assert leaves[0] <= plan.info()["leaves"] <= leaves[1], plan.info()
    p64, m64 = dev(pos, torch.float64), dev(m, torch.float64)
    eg = rel_err(host(plan.field(dev(m))),
                 host(magforce.field_allpairs_f64(ctx, p64, p64, m64, 2.0)))
    ef = rel_err(host(plan.force(dev(m))), host(magforce.force_allpairs_f64(ctx, p64, m64, 2.0)))
    print(f"{n} particles, {plan.info()['leaves']} leaves: field {eg:.2e} force {ef:.2e}")
    assert eg < TOL[order] and ef < TOL[order]
