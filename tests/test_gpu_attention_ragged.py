"""attention_causal_any and qkv_rope(v_padded=True) at sequence lengths that are not
whole key blocks, against the unfused path (fp16 scores, softmax_entropy kernel, product with v), which
served them before, and restatements in 32 and 64 bits.

Bars with random inputs: out within 1e-2 of the largest reference value, H within 1e-4.  The probabilities
are those of the unfused path, but a score whose two summation orders round to neighbouring fp16 values (2^-11
of |x| <= ~8 apart) moves its probability by up to 2^-8.  With inputs whose scores are exact in any order
the roundings themselves are held to their bound (test_roundings_of_exact_scores); padding exact.
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


def test_what_is_refused_is_named(ee):
    from entropy_engine import _lib
    q = torch.zeros(1, 3, 64, 64, device="cuda", dtype=torch.float16)     # an odd number of query heads per kv head
    k, vt = (torch.zeros(1, 1, 64, 64, device="cuda", dtype=torch.float16) for _ in range(2))
    with pytest.raises(_lib.EngineError, match="even number") as any_s:
        ee.attention_causal_any(q, k, vt)
    with pytest.raises(_lib.EngineError, match="S % 64"):
        ee.attention_causal(q, k, vt)
    assert "S % 64" not in str(any_s.value)


# scores around 0 and around values where fp16 steps by 0.5, 8 and 32: e^(x - m) and its sum have to come from the
# difference itself
@pytest.mark.parametrize("offset,c", [(0, 1), (1000, 1), (10000, 8), (60000, 32)])
@pytest.mark.parametrize("S", [1, 37, 300, 1001, 2001])
def test_roundings_of_exact_scores(ee, S, offset, c):
    """q and k of few bits: every score is exact in f32 in any order, so only p = fp16(e / Z), the
    sums of out and its store round.  |out - 64 bits| <= 2^-11 (sum p |v| + |out|) + S 2^-25 max |v| (p
    below fp16's normal range) + f32's share; against the sum of the correctly rounded p, out differs in no more
    of its last bits than the unfused path's, whose roundings these are."""
    from entropy_engine.dispatch import _attention_entropy
    B, Hq, Hkv, d = 1, 4, 2, 64
    g = torch.Generator(device="cuda").manual_seed(S + offset)
    tri = lambda n: torch.randint(-1, 2, (S, n, d), device="cuda", generator=g).half()
    q, k = tri(Hq) * c, tri(Hkv)
    q[..., 0], k[..., 0] = 8.0, float(offset)              # (q carries a factor 1/8)
    v = torch.randn(S, Hkv, d, device="cuda", generator=g).half()
    qkv = torch.cat([q, k, v], dim=1).reshape(S, -1).contiguous()
    qh, kh, vh, vt = _inputs(ee, B, S, Hq, Hkv, qkv)
    out, H = ee.attention_causal_any(qh, kh, vt)
    un_o, un_h = _attention_entropy(qh, kh, vh, 1.0, causal=True)
    G = Hq // Hkv
    kr, vr = (t.repeat_interleave(G, dim=1).double() for t in (kh, vh))
    x = (qh.double() @ kr.transpose(-1, -2).contiguous()).half().double()
    x = x.masked_fill(~torch.ones(S, S, device="cuda", dtype=torch.bool).tril(), float("-inf"))
    p = torch.softmax(x, dim=-1)
    ref, best = p @ vr, (p.half().double() @ vr).half()
    bar = 2.0 ** -11 * (p @ vr.abs() + ref.abs()) + (S * 2.0 ** -25 + (S // 64 + 64) * 2.0 ** -23) * vr.abs().amax()
    o = out.view(B, S, Hq, d).transpose(1, 2)
    assert ((o.double() - ref).abs() <= bar).all()
    assert torch.equal(o[:, :, 0], vr[:, :, 0].half())                    # one key: p = 1
    off, off_un = ((t != best).double().mean().item() for t in (o, un_o))
    assert off <= 1.5 * off_un + 0.01, (off, off_un)
    s = x - x.amax(dim=-1, keepdim=True)
    h = torch.logsumexp(s, dim=-1) - (p * s.clamp(min=-1e4)).sum(-1)
    # f32 sums of a step's 32 terms and of the steps, e to 2^-23 and its argument to 2^-24 |s|
    tol = (S // 64 + 64) * 2.0 ** -23 * (1 + h)
    assert ((H.double() - h).abs() <= tol).all()
    assert ((un_h.double() - h).abs() <= tol).all()


def test_many_prompts_of_one_or_two_tokens_take_the_unfused_path(ee, monkeypatch):
    """Both sides of the line; the logits are the unfused path's there."""
    from entropy_engine import dispatch
    from test_gpu_parity import SMALL_LLAMA
    m = ee.EntropyGatedLlama.random_init(dict(SMALL_LLAMA, layers=1), seed=3)
    calls, fused = [], dispatch.K.attention_causal_any
    monkeypatch.setattr(dispatch.K, "attention_causal_any", lambda *a: calls.append(1) or fused(*a))
    Hq = SMALL_LLAMA["heads"]
    for S, line in ((1, 1024 // Hq), (2, 4096 // Hq)):
        for B in (line, line + 1):
            ids = torch.randint(0, SMALL_LLAMA["vocab"], (B, S), device="cuda")
            calls.clear()
            out = m.forward(ids)
            assert bool(calls) == (B == line)
            if B > line:
                m.fused_attention = False
                assert torch.equal(out, m.forward(ids))
                m.fused_attention = True
