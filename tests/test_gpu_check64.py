"""The FP64 check path against the CPU oracle where its source split and its
reciprocal square root can go wrong: one target, wave and block edges, fewer
targets than sources and the reverse, coincident particles, and distances at
whole multiples of h (a regular lattice), where the force curves change piece.

Tolerances: a sum of n terms in FP64 with a few roundings each is within about
1e-15 sqrt(n) of the oracle's, taken as 1e-13; the force keeps 1e-9 for the
oracle's rotation frame and its 1e-10 pole patch.
"""
import numpy as np
import pytest

from conftest import jittered_block, random_moments, rel_err

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.tensor(np.ascontiguousarray(np.asarray(a).T), dtype=torch.float64, device="cuda")


def host(t):
    return t.cpu().numpy().T


@pytest.mark.parametrize("nt,ns", [(1, 1), (1, 700), (63, 129), (64, 64), (65, 4097), (257, 256),
                                   (300, 1), (1000, 65)])
def test_field_split_vs_oracle(ctx, oracle, nt, ns):
    import magforce
    pos = jittered_block(17, 17, 17, seed=3)
    t, s, m = pos[:nt], pos[-ns:], random_moments(ns, seed=nt)
    got = host(magforce.field_allpairs_f64(ctx, dev(t), dev(s), dev(m), 2.0, hconst=[1, 2, 3]))
    assert rel_err(got, oracle.field_allpairs(t, s, m, 2.0, hconst=[1, 2, 3])) < 1e-13


def test_field_without_sources(ctx):
    import magforce
    t, none = jittered_block(3, 3, 3, seed=1), np.zeros((0, 3))
    got = host(magforce.field_allpairs_f64(ctx, dev(t), dev(none), dev(none), 2.0, hconst=[1, 2, 3]))
    assert np.array_equal(got, np.tile([1.0, 2.0, 3.0], (27, 1)))


@pytest.mark.parametrize("n,nt", [(1, 1), (65, 65), (1001, 1), (1001, 64), (1001, 300)])
def test_force_subset_vs_oracle(ctx, oracle, n, nt):
    import magforce
    import torch
    pos, m = jittered_block(11, 13, 7, seed=5)[:n], random_moments(n, seed=6)
    idx = np.sort(np.random.default_rng(n + nt).choice(n, size=nt, replace=False))
    got = host(magforce.force_subset_f64(ctx, dev(pos), dev(m), 2.0, torch.tensor(idx, device="cuda")))
    want = oracle.force_allpairs(pos, m, 2.0)
    if n == 1:  # no partner: no force
        assert np.array_equal(got, want)
    else:
        assert rel_err(got, want[idx]) < 1e-9


def test_whole_multiples_of_h_and_coincident(ctx, oracle):
    """Unjittered lattice of spacing h / 2 (pairs at q = 1, 2, 3 exactly) with
    one particle twice."""
    import magforce
    pos = np.stack(np.meshgrid(*[np.arange(7.0)] * 3, indexing="ij"), -1).reshape(-1, 3)
    pos = np.concatenate([pos, pos[100:101]])
    m = random_moments(pos.shape[0], seed=9)
    f = host(magforce.field_allpairs_f64(ctx, dev(pos), dev(pos), dev(m), 2.0))
    assert rel_err(f, oracle.field_allpairs(pos, pos, m, 2.0)) < 1e-13
    F = host(magforce.force_allpairs_f64(ctx, dev(pos), dev(m), 2.0))
    assert rel_err(F, oracle.force_allpairs(pos, m, 2.0)) < 1e-9


def test_refused_scratch_gives_the_same(ctx):
    """With every device allocation refused, a context without scratch still
    answers (one source chunk), within rounding of the split sum."""
    import magforce
    pos, m = jittered_block(10, 10, 10, seed=2), random_moments(1000, seed=3)
    args = (dev(pos), dev(pos), dev(m), 2.0)
    want = host(magforce.field_allpairs_f64(ctx, *args))
    c = magforce.Context(0)
    magforce.set_alloc_hook(lambda n: True)
    try:
        got = host(magforce.field_allpairs_f64(c, *args))
    finally:
        magforce.set_alloc_hook(None)
    c.close()
    assert rel_err(got, want) < 1e-13
