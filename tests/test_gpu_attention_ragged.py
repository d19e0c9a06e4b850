"""attention_causal_any and qkv_rope(v_padded=True) at sequence lengths that are not
whole key blocks, against the unfused path (fp16 scores, softmax_entropy kernel, product with v), which
served them before, and an fp32 restatement.

Bars: out within 1e-2 of the largest reference value (its probabilities are rounded to fp16, 2^-11 each, at
another scale than the unfused ones), H within 1e-4 (both from the same fp16 scores in f32;
a score whose two summation orders round to neighbouring fp16 values moves it by less); padding exact.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ee():
    import entropy_engine
    return entropy_engine


def _inputs(ee, B, S, Hq, Hkv, qkv):
    d = 64
    cos = torch.ones(1, S, d, device="cuda", dtype=torch.float16)
    sin = torch.zeros(1, S, d, device="cuda", dtype=torch.float16)
    q, k, v = ee.qkv_rope(qkv, cos, sin, B, S, Hq, Hkv, d, d ** -0.5)
    q2, k2, vt = ee.qkv_rope(qkv, cos, sin, B, S, Hq, Hkv, d, d ** -0.5, v_padded=True)
    assert torch.equal(q, q2) and torch.equal(k, k2)
    return q, k, v, vt


# one row, around the 16-token groups, the 32-row halves and the 64-key blocks; both workgroup widths; batches
@pytest.mark.parametrize("S", [1, 15, 17, 33, 63, 64, 65, 127, 300, 511])
@pytest.mark.parametrize("B,Hq,Hkv", [(1, 32, 4), (3, 4, 2)])
def test_any_length_against_unfused(ee, B, S, Hq, Hkv):
    from entropy_engine.dispatch import _attention_entropy
    d = 64
    g = torch.Generator(device="cuda").manual_seed(B * S + Hq)
    qkv = (torch.randn(B * S, (Hq + 2 * Hkv) * d, device="cuda", generator=g) * 1.5).half()
    q, k, v, vt = _inputs(ee, B, S, Hq, Hkv, qkv)
    Sp = (S + 63) // 64 * 64
    vp = torch.zeros(B, Hkv, Sp, d, device="cuda", dtype=torch.float16)
    vp[:, :, :S] = v
    order = torch.tensor(ee.VT_ORDER, device="cuda")
    idx = (torch.arange(Sp // 16, device="cuda")[:, None] * 16 + order[None, :]).reshape(-1)
    assert torch.equal(vt, vp[:, :, idx, :].transpose(-1, -2))
    wide = torch.full((B * S + 1, Hq * d), 7.0, device="cuda", dtype=torch.float16)
    out, H = ee.attention_causal_any(q, k, vt, out=wide[:B * S])
    assert (wide[B * S:] == 7).all()                       # nothing stored past the last token
    o = out.view(B, S, Hq, d).transpose(1, 2).float()
    un_o, un_h = _attention_entropy(q, k, v, 1.0, causal=True)
    assert (o - un_o.float()).abs().max().item() <= 1e-2 * un_o.float().abs().max().item()
    assert torch.allclose(H, un_h, rtol=1e-4, atol=1e-4)
    G = Hq // Hkv
    kr, vr = k.repeat_interleave(G, dim=1).float(), v.repeat_interleave(G, dim=1).float()
    sc = (q.float() @ kr.transpose(-1, -2).contiguous()).half().float()
    sc = sc.masked_fill(~torch.ones(S, S, device="cuda", dtype=torch.bool).tril(), float("-inf"))
    ref = torch.softmax(sc, dim=-1) @ vr
    assert (o - ref).abs().max().item() <= 1e-2 * ref.abs().max().item()


def test_scores_at_minus_infinity(ee):
    """Scores that round to -inf do not count; a row with no other score is NaN in both paths."""
    from entropy_engine.dispatch import _attention_entropy
    B, S, Hq, Hkv, d = 1, 100, 4, 2, 64
    g = torch.Generator(device="cuda").manual_seed(5)
    qkv = torch.zeros(B * S, (Hq + 2 * Hkv) * d, device="cuda", dtype=torch.float16)
    qkv[:, :Hq * d] = 400.0
    qkv[::2, Hq * d:(Hq + Hkv) * d] = -400.0               # even keys: 64 * 50 * -400 -> -inf
    qkv[:, (Hq + Hkv) * d:] = torch.randn(S, Hkv * d, device="cuda", generator=g).half()
    q, k, v, vt = _inputs(ee, B, S, Hq, Hkv, qkv)
    out, H = ee.attention_causal_any(q, k, vt)
    un_o, un_h = _attention_entropy(q, k, v, 1.0, causal=True)
    o = out.view(B, S, Hq, d).transpose(1, 2).float()
    assert torch.isnan(o[:, :, 0]).all() and torch.isnan(H[:, :, 0]).all()
    assert torch.isnan(un_o[:, :, 0]).all() and torch.isnan(un_h[:, :, 0]).all()
    assert (o[:, :, 1:] - un_o[:, :, 1:].float()).abs().max().item() <= 1e-2 * v.abs().max().item()
    assert torch.allclose(H[:, :, 1:], un_h[:, :, 1:], rtol=1e-4, atol=1e-4)


def test_the_padded_layout_is_checked(ee):
    q = torch.zeros(1, 4, 96, 64, device="cuda", dtype=torch.float16)
    k = torch.zeros(1, 2, 96, 64, device="cuda", dtype=torch.float16)
    with pytest.raises(ValueError):
        ee.attention_causal_any(q, k, torch.zeros(1, 2, 64, 96, device="cuda", dtype=torch.float16))
