"""mf_field_allpairs_noalloc where the scratch array holds the chunk partials of the
allocating call only if nothing else takes room per target: both split the sources alike,
so their outputs agree bitwise."""
import pytest

pytestmark = pytest.mark.gpu


def test_partials_have_the_room(ctx):
    import magforce
    import torch
    g = torch.Generator(device="cuda").manual_seed(6)
    # five chunks of 6 MB of partials, beside which 8 MB of target records would not fit
    tpos = 80.0 * torch.rand((3, 250_000), generator=g, device="cuda")
    spos = 80.0 * torch.rand((3, 2560), generator=g, device="cuda")
    m = 0.5 * torch.randn((3, 2560), generator=g, device="cuda")
    got = magforce.field_allpairs_noalloc(ctx, tpos, spos, m, 2.0)
    want = magforce.field_allpairs(ctx, tpos, spos, m, 2.0)
    assert torch.equal(got, want)
