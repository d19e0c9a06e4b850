"""Several rows per wave (eek_softmax_entropy_g*), rows at any 2-byte alignment in the vector
kernels, and the row mean, against the oracle."""
import numpy as np
import pytest
import torch

from test_gpu_parity import check_entropy, check_probs, cuda, host, logits_rows

pytestmark = pytest.mark.gpu


@pytest.fixture
def ee():
    import entropy_engine
    yield entropy_engine
    _opt(0)


def _opt(v):
    from entropy_engine import _lib
    _lib.check(_lib.lib().ee_engine_set_option(_lib.engine(), b"se_group", v))


def _last_kernel():
    from entropy_engine import _lib
    return _lib.lib().ee_last_kernel().decode()


def _strided(X, pad, lead):
    """X as a view of rows `pad` elements apart beyond their length, `lead` elements into the buffer."""
    R, S = X.shape
    buf = torch.full((lead + R * (S + pad),), float("nan"), dtype=torch.float16, device="cuda")
    v = buf[lead:lead + R * (S + pad)].view(R, S + pad)[:, :S]
    v.copy_(cuda(X))
    return buf, v


# S at the edges of the 128- and 256-column vectors and of the kernels; R with a ragged last wave
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("R,S", [(5, 16), (37, 17), (130, 127), (9, 128), (131, 129), (300, 255), (33, 300), (385, 384),
                                 (66, 385), (70, 511), (1031, 512), (41, 513), (1537, 768), (35, 769), (50, 1000),
                                 (2049, 1024)])
def test_softmax_group_rows(ee, orc, R, S, causal):
    rng = np.random.default_rng(R * 31 + S)
    X = logits_rows(rng, R, S)
    X[R // 2, : min(S, 9)] = X[R // 2].max()                 # several entries at the max
    if S > 4:
        X[R // 3, 3] = -np.inf
    H_ref, P_ref = orc.softmax_entropy(X, causal=causal)
    _opt(2)
    for pad, lead in ((0, 0), (1, 3)):
        _, x = _strided(X, pad, lead)
        out, p = _strided(np.zeros_like(X), pad, lead)
        _, h, tier = ee.softmax_entropy(x, causal=causal, thresholds=(0.41, 1.68), out_probs=p)
        assert "_g16_" in _last_kernel() or "_g32_" in _last_kernel()
        check_entropy(host(h), H_ref)
        check_probs(host(p), P_ref)
        assert np.array_equal(host(tier), orc.route(host(h), 0.41, 1.68)[0])
        if pad:                                               # nothing written between the rows
            gaps = out[lead:].view(R, S + pad)[:, S:]
            assert torch.isnan(gaps).all() and torch.isnan(out[:lead]).all()
        _, h2, _ = ee.softmax_entropy(x, causal=causal, probs=False)
        assert np.array_equal(host(h2), host(h))


@pytest.mark.parametrize("S", [64, 500, 1000])
def test_softmax_group_rows_without_a_finite_max(ee, orc, S):
    rng = np.random.default_rng(S)
    X = rng.standard_normal((11, S)).astype(np.float16)
    X[1] = -np.inf
    X[3, S // 3] = np.nan
    X[10, S - 1] = np.nan
    X[5, 7] = np.inf
    X[6] = np.float16(-65504)
    H_ref, P_ref = orc.softmax_entropy(X)
    _opt(2)
    p, h, _ = ee.softmax_entropy(cuda(X))
    h, p = host(h), host(p)
    assert np.array_equal(np.isnan(h), np.isnan(H_ref))
    ok = ~np.isnan(H_ref)
    check_entropy(h[ok], H_ref[ok])
    check_probs(p[ok], P_ref[ok])
    assert np.array_equal(np.isnan(p), np.isnan(P_ref.astype(np.float16)))


@pytest.mark.parametrize("wpr", [0, 1, 2, 4, 8])
@pytest.mark.parametrize("S", [100, 512, 1777, 4096])
def test_softmax_rows_at_the_lowest_fp16(ee, orc, S, wpr):
    """Rows whose entries are all at or next to -65504 (a mask of the type's lowest value), alone or beside
    -inf ones, and the padding past S: none of the -inf counts as an entry."""
    from entropy_engine import _lib
    X = np.full((6, S), -65504, np.float16)
    X[1, ::2] = -np.inf
    X[2, 3:] = -np.inf
    X[3, 5] = np.float16(-65472)
    X[3, S // 2:] = -np.inf
    X[4, 1:] = -np.inf
    X[5] = np.linspace(-3, 3, S).astype(np.float16)
    H_ref, P_ref = orc.softmax_entropy(X)
    _lib.check(_lib.lib().ee_engine_set_option(_lib.engine(), b"se_wpr", wpr if S <= 512 * wpr * 4 else 0))
    try:
        _, x = _strided(X, 1, 1)
        p, h, _ = ee.softmax_entropy(x)
        check_entropy(host(h), H_ref)
        check_probs(host(p), P_ref)
    finally:
        _lib.check(_lib.lib().ee_engine_set_option(_lib.engine(), b"se_wpr", 0))


# one row per several waves, rows that are not 16-byte aligned: the generic kernel's shapes before
@pytest.mark.parametrize("R,S,causal", [(40, 1777, False), (33, 4095, True), (9, 16383, False), (5, 20001, True)])
def test_softmax_unaligned_long_rows(ee, orc, R, S, causal):
    rng = np.random.default_rng(S)
    X = logits_rows(rng, R, S)
    H_ref, P_ref = orc.softmax_entropy(X, causal=causal)
    _, x = _strided(X, 1, 1)
    out, p = _strided(np.zeros_like(X), 2, 5)
    _, h, _ = ee.softmax_entropy(x, causal=causal, out_probs=p)
    assert "generic" not in _last_kernel()
    check_entropy(host(h), H_ref)
    check_probs(host(p), P_ref)
    assert torch.isnan(out[5:].view(R, S + 2)[:, S:]).all()


# the non-temporal loads of the 2-, 4- and 8-wave rows, from rows at any alignment
@pytest.mark.parametrize("wpr,S", [(2, 4095), (4, 8191), (8, 16383), (8, 20001)])
@pytest.mark.parametrize("causal", [False, True])
def test_softmax_unaligned_rows_non_temporal(ee, orc, wpr, S, causal):
    from entropy_engine import _lib
    rng = np.random.default_rng(S)
    X = logits_rows(rng, 9, S)
    H_ref, P_ref = orc.softmax_entropy(X, causal=causal)
    _, x = _strided(X, 1, 3)
    out, p = _strided(np.zeros_like(X), 2, 5)
    for key, v in ((b"se_wpr", wpr), (b"se_nt", 2)):
        _lib.check(_lib.lib().ee_engine_set_option(_lib.engine(), key, v))
    try:
        _, h, _ = ee.softmax_entropy(x, causal=causal, out_probs=p)
        assert _last_kernel().endswith("_nt")
    finally:
        for key in (b"se_wpr", b"se_nt"):
            _lib.check(_lib.lib().ee_engine_set_option(_lib.engine(), key, 0))
    check_entropy(host(h), H_ref)
    check_probs(host(p), P_ref)
    assert torch.isnan(out[5:].view(9, S + 2)[:, S:]).all() and torch.isnan(out[:5]).all()


@pytest.mark.parametrize("B,H,S", [(1, 1, 1), (3, 5, 33), (2, 7, 64), (8, 32, 512), (2, 3, 171)])
def test_row_mean(ee, B, H, S):
    g = torch.Generator(device="cuda")
    g.manual_seed(S)
    x = torch.randn(B, H, S, S, generator=g, device="cuda").half()
    _, ent = ee.fused_softmax_entropy(x, causal=True)
    _, h, _ = ee.softmax_entropy(x.view(B * H * S, S), causal=True)
    ref = h.double().view(B, -1).mean(dim=1)
    # f32 sums of n non-negative values, at most 64 of them in a row
    assert ((ent.double() - ref).abs() <= 64 * 2.0 ** -23 * ref + 1e-30).all()


@pytest.mark.parametrize("R,S,causal,group", [(1, 256, False, True), (2559, 257, True, False), (2560, 384, False, True),
                                              (4095, 385, False, False), (4096, 512, True, True), (2047, 513, False, False),
                                              (2048, 768, False, True), (2048, 1024, True, True),
                                              (2048, 1024, False, False), (16384, 1024, False, True),
                                              (16384, 1025, False, False)])
def test_softmax_group_choice(ee, R, S, causal, group):
    """Both sides of each line between one row per wave and several."""
    x = torch.randn(R, S, device="cuda").half()
    ee.softmax_entropy(x, causal=causal)
    assert ("_g16_" in _last_kernel() or "_g32_" in _last_kernel()) == group


@pytest.mark.parametrize("B,H,S,own", [(512, 2, 8, True), (513, 2, 8, False), (513, 64, 64, True), (1030, 1, 1, False)])
def test_row_mean_of_many_elements(ee, B, H, S, own):
    """One workgroup per element only where those fill the card no worse than a reduction over rows."""
    g = torch.Generator(device="cuda").manual_seed(B)
    x = torch.randn(B, H, S, S, generator=g, device="cuda").half()
    _, ent = ee.fused_softmax_entropy(x, causal=True)
    assert ("mean" in _last_kernel()) == own
    _, h, _ = ee.softmax_entropy(x.view(B * H * S, S), causal=True)
    ref = h.double().view(B, -1).mean(dim=1)
    assert ((ent.double() - ref).abs() <= 64 * 2.0 ** -23 * ref + 1e-30).all()
