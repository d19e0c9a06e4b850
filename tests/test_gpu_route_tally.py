"""route_tally against the same sum in tensor operations (whole numbers: equal): no layer, one, lanes
of a wave not filled, more layers than lanes, and counts whose weighted sum passes 2^32."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,top", [(0, 9), (1, 9), (22, 4096), (64, 4096), (65, 2**31 - 1), (300, 2**31 - 1)])
def test_route_tally(L, top):
    import entropy_engine as ee
    g = torch.Generator(device="cuda").manual_seed(L)
    counts = torch.randint(0, top, (L, 3), device="cuda", generator=g, dtype=torch.int32)
    w = torch.randint(0, 8, (L, 1), device="cuda", generator=g, dtype=torch.int64)
    ref = (counts.to(torch.int64) * w).sum(0)
    ref[2] += 12345
    assert torch.equal(ee.route_tally(counts, w, 12345), ref)


def test_route_heads_writes_the_counts_it_is_given():
    import entropy_engine as ee
    h = torch.rand(2, 3, 50, device="cuda") * 8
    rows = torch.full((4, 3), -1, device="cuda", dtype=torch.int32)
    tier, idx, counts = ee.route_heads(h, 2.0, 5.0, counts=rows[1])
    ref = ee.route_heads(h, 2.0, 5.0)
    assert torch.equal(tier, ref[0]) and torch.equal(idx, ref[1]) and torch.equal(rows[1], ref[2])
    assert counts.data_ptr() == rows[1].data_ptr() and (rows[[0, 2, 3]] == -1).all()
    with pytest.raises(ValueError):
        ee.route_heads(h, 2.0, 5.0, counts=rows)
