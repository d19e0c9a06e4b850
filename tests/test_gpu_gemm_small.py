"""The few-rows GEMM kernels (eek_gemm_m64w*, engine option gemm_small) against the
larger tiles' bits: every tier sums K in the same order, so plain, SwiGLU, W8A16-from-codes
and routed outputs are bit-identical, and INT8 also equals the oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def ee():
    import entropy_engine
    yield entropy_engine
    _opt(0)


def _opt(v):
    from entropy_engine import _lib
    _lib.check(_lib.lib().ee_engine_set_option(_lib.engine(), b"gemm_small", v))


def _last_kernel():
    from entropy_engine import _lib
    return _lib.lib().ee_last_kernel().decode()


def _bits(t):
    torch.cuda.synchronize()
    return t.view(torch.int16)


def _weight(ee, N, K, seed=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).half()
    codes, scale = ee.quantize_weight_codes(w)
    return ee.PackedWeight(codes, scale).materialize(), g


# K: one stage up to several passes over the register ring, with partial chunks and passes
SHAPES = [(1, 128, 4), (8, 256, 64), (9, 1152, 36), (16, 2176, 520), (17, 1024, 132), (32, 4096, 96), (33, 1920, 260),
          (64, 640, 128), (65, 2048, 68), (130, 1408, 192), (300, 384, 64)]


@pytest.mark.parametrize("cols", [16, 32, 64])
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_small_gemm_bits(ee, M, K, N, cols):
    pw, g = _weight(ee, N, K, seed=M + N)
    x = torch.randn(M, K + 16, generator=g, device="cuda").half()[:, :K]     # a row stride of its own
    x[0] *= 30.0
    i8, f8 = ee.quantize_activations(x, "dispatcher"), ee.quantize_activations(x, "fp8")
    calls = [("int8", i8[0], pw.i8, i8[1], pw.scale), ("fp8", f8[0], pw.f8, f8[1], pw.scale),
             ("fp16", x, pw.f16, None, None)]
    for kind, a, b, sa, sb in calls:
        _opt(1)
        ref = ee.gemm(kind, a, b, sa, sb)
        assert "m64" not in _last_kernel()
        _opt(cols)
        assert torch.equal(_bits(ee.gemm(kind, a, b, sa, sb)), _bits(ref)), kind
        assert "m64w" in _last_kernel()
        if kind == "fp16":
            assert torch.equal(_bits(ee.gemm("w8a16", x, pw.i8, None, pw.scale)), _bits(ref)), "w8a16"
            assert "m64w" in _last_kernel()


@pytest.mark.parametrize("cols", [16, 32])
@pytest.mark.parametrize("M,K,F", [(1, 128, 32), (8, 2048, 352), (20, 640, 96), (40, 1152, 64), (70, 512, 160)])
def test_small_gemm_swiglu_bits(ee, M, K, F, cols):
    pw, g = _weight(ee, 2 * F, K, seed=M)
    x = torch.randn(M, K, generator=g, device="cuda").half()
    i8, f8 = ee.quantize_activations(x, "dispatcher"), ee.quantize_activations(x, "fp8")
    for kind, a, b, sa, sb in [("int8", i8[0], pw.i8, i8[1], pw.scale), ("fp8", f8[0], pw.f8, f8[1], pw.scale),
                               ("fp16", x, pw.f16, None, None)]:
        _opt(1)
        ref = ee.gemm(kind, a, b, sa, sb, swiglu=True)
        _opt(cols)
        assert torch.equal(_bits(ee.gemm(kind, a, b, sa, sb, swiglu=True)), _bits(ref)), kind
        if kind == "fp16":
            assert torch.equal(_bits(ee.gemm("w8a16", x, pw.i8, None, pw.scale, swiglu=True)), _bits(ref)), "w8a16"


# the FP8 SwiGLU form of 33 to 64 rows: one buffer of A, K from one stage to several passes over four, with remainders
@pytest.mark.parametrize("M", [33, 64, 100])
@pytest.mark.parametrize("K", [128, 256, 512, 640, 2048, 2176])
def test_fp8_swiglu_of_64_rows(ee, M, K):
    pw, g = _weight(ee, 192, K, seed=K)
    x = torch.randn(M, K, generator=g, device="cuda").half()
    a, s = ee.quantize_activations(x, "fp8")
    _, idx, cnt = ee.route(torch.full((M,), 2.0, device="cuda"), 1.5, 2.5)
    _opt(1)
    ref = ee.gemm("fp8", a, pw.f8, s, pw.scale, swiglu=True)
    for cols in (16, 32):
        _opt(cols)
        assert torch.equal(_bits(ee.gemm("fp8", a, pw.f8, s, pw.scale, swiglu=True)), _bits(ref))
        out = torch.full_like(ref, float("nan"))
        assert torch.equal(_bits(ee.routed_linear(x, pw, idx, cnt, out=out, swiglu=True)), _bits(ref))
        assert _last_kernel() == "eek_gemm_routed_m64w1_swiglu"


def test_small_gemm_int8_accumulators_and_oracle(ee, orc):
    rng = np.random.default_rng(3)
    M, K, N = 21, 1280, 100
    a = rng.integers(-127, 128, (M, K), dtype=np.int8)
    b = rng.integers(-127, 128, (N, K), dtype=np.int8)
    sa, sb = rng.random(M, dtype=np.float32) + 0.1, rng.random(N, dtype=np.float32) * 1e-3
    acc = torch.zeros((M, N), dtype=torch.int32, device="cuda")
    _opt(16)
    c = ee.gemm("int8", *(torch.from_numpy(t).cuda() for t in (a, b, sa, sb)), acc_out=acc)
    ref = a.astype(np.int64) @ b.astype(np.int64).T
    assert np.array_equal(acc.cpu().numpy(), ref)
    out = ((ref.astype(np.float32) * sa[:, None]) * sb[None, :]).astype(np.float16)
    assert np.array_equal(c.cpu().numpy().view(np.uint16), out.view(np.uint16))


# rows of the three tiers: empty tiers, edges of the 16- and 64-row groups, several M-tiles
@pytest.mark.parametrize("counts", [(1, 0, 0), (0, 1, 0), (0, 0, 1), (3, 4, 1), (16, 17, 33), (64, 0, 65), (5, 130, 20)])
@pytest.mark.parametrize("K,N,sw", [(1024, 512, False), (2048, 260, False), (512, 192, True)])
def test_small_routed_bits(ee, counts, K, N, sw):
    M = sum(counts)
    pw, g = _weight(ee, N, K, seed=M)
    x = torch.randn(M, K, generator=g, device="cuda").half()
    h = torch.cat([torch.full((c,), t + 1.0) for t, c in enumerate(counts)])[torch.randperm(M)].cuda()
    _, idx, cnt = ee.route(h, 1.5, 2.5)
    _opt(1)
    ref = ee.routed_linear(x, pw, idx, cnt, swiglu=sw)
    assert "m64" not in _last_kernel()
    for cols in (16, 32):
        _opt(cols)
        out = torch.full_like(ref, float("nan"))
        ee.routed_linear(x, pw, idx, cnt, out=out, swiglu=sw)
        assert "m64w" in _last_kernel()
        assert torch.equal(_bits(out), _bits(ref))


def test_small_gemm_choice(ee):
    """Decode shapes take the small tiles, the headline shape does not; W8A16 from the codes
    gives the FP16 tier's bits through the public call."""
    from entropy_engine import _lib
    L, e = _lib.lib(), _lib.engine()
    for kind in range(4):
        assert L.ee_gemm_small_waves(e, kind, 4, 4096, 4096, 0) > 0
        assert L.ee_gemm_small_waves(e, kind, 1024, 4096, 4096, 0) == 0
        assert L.ee_gemm_small_waves(e, kind, 4, 4096, 4104, 0) == 0        # K of whole 128-byte stages only
    pw, g = _weight(ee, 1000, 1024)
    x = torch.randn(5, 1024, generator=g, device="cuda").half()
    lin = torch.nn.Linear(1024, 1000, bias=False, device="cuda", dtype=torch.float16)
    layer = ee.EntropyDispatchedLinear.from_linear(lin)
    y = layer(x)
    assert "w8a16" in _last_kernel()
    _opt(1)
    assert torch.equal(_bits(y), _bits(layer(x)))


def test_few_rows_pack_the_weight_that_a_captured_call_reads(ee):
    """A warm-up on decode rows, then a longer call under capture: an eager call before the
    graph's first replay finds the fp16 weights filled."""
    from entropy_engine.kernels import gemm_fp16_tier
    g = torch.Generator(device="cuda").manual_seed(11)
    codes, scale = ee.quantize_weight_codes((torch.randn(4096, 1024, generator=g, device="cuda") / 32).half())
    x = torch.randn(1024, 1024, generator=g, device="cuda").half()
    ref = ee.gemm("fp16", x, ee.PackedWeight(codes, scale).f16)
    pw = ee.PackedWeight(codes, scale)
    gemm_fp16_tier(x[:4], pw)
    assert "w8a16" in _last_kernel()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = gemm_fp16_tier(x, pw)
    assert "w8a16" not in _last_kernel()
    assert torch.equal(_bits(gemm_fp16_tier(x, pw)), _bits(ref))
    for _ in range(3):
        y.zero_()
        graph.replay()
        assert torch.equal(_bits(y), _bits(ref))


@pytest.mark.parametrize("entry", ["linear", "linear_swiglu", "linear_noalloc", "gemm", "gemm_swiglu"])
@pytest.mark.parametrize("M", [3, 40])
def test_routed_c_calls_take_b_f16_as_it_is(ee, entry, M):
    """The C calls do not ask that b_f16 was packed from b_i8 and b_scale: the FP16 rows are b_f16's, with few
    rows too.  ee_routed_linear_packed does ask it, and refuses flags that it does not know."""
    from entropy_engine import _lib
    L, e = _lib.lib(), _lib.engine()
    K, N, sw = 512, 320, entry.endswith("swiglu")
    pw, g = _weight(ee, N, K, seed=M)
    other = torch.randn(N, K, generator=g, device="cuda").half()          # not the codes' values
    x = torch.randn(M, K, generator=g, device="cuda").half()
    h = torch.where(torch.arange(M, device="cuda") % 3 == 0, 1.0, 3.0)    # INT8 and FP16 rows
    tier, idx, cnt = ee.route(h, 1.5, 2.5)
    out = torch.empty(M, N // 2 if sw else N, device="cuda", dtype=torch.float16)
    codes = torch.zeros(M, K, device="cuda", dtype=torch.uint8)
    scale = torch.ones(M, device="cuda")
    head = [e, x.data_ptr(), K, M, K, N, idx.data_ptr(), cnt.data_ptr(), pw.i8.data_ptr(), pw.f8.data_ptr(),
            other.data_ptr(), pw.scale.data_ptr(), out.data_ptr(), out.shape[1]]
    ws = [] if entry == "linear_noalloc" else [codes.data_ptr(), scale.data_ptr()]
    _lib.check(getattr(L, "ee_routed_" + entry)(*head, *ws, _lib.stream_handle()))
    ref = ee.gemm("fp16", x, other, swiglu=sw)
    rows = (tier == 2).nonzero().squeeze(1)
    assert rows.numel() and torch.equal(_bits(out[rows]), _bits(ref[rows]))
    with pytest.raises(_lib.EngineError, match="flags"):
        _lib.check(L.ee_routed_linear_packed(*head, codes.data_ptr(), scale.data_ptr(), 4, _lib.stream_handle()))


def test_few_rows_choice_of_the_codes_for_wide_weights(ee):
    """From 32 Mi weights on the codes pay up to 128 rows, and up to 256 without SwiGLU where the small tiles pull
    at most 3/4 of the large tile's bytes; 300 rows of 14336 columns and 700 of 11264 keep the 256-row tiles."""
    from entropy_engine import _lib
    L, e, W8 = _lib.lib(), _lib.engine(), _lib.EE_GEMM_W8A16
    assert L.ee_gemm_small_waves(e, W8, 100, 14336, 4096, 0) > 0
    assert L.ee_gemm_small_waves(e, W8, 129, 5632, 8192, 0) > 0
    for M, N, K, sw in [(300, 14336, 4096, 0), (700, 11264, 4096, 0), (384, 11264, 8192, 1), (129, 8192, 4096, 1)]:
        assert L.ee_gemm_small_waves(e, W8, M, N, K, sw) == 0


# both sides of each line of the routed choice, on the 256 CUs of an MI355X
@pytest.mark.parametrize("M,K,N,sw,kernel", [
    (64, 128, 11008, False, "m64w2_dense"), (65, 128, 11008, False, "eek_gemm_routed"), (65, 128, 2560, False, "m64w1"),
    (32, 128, 8448, False, "m64w2"), (33, 128, 8448, False, "eek_gemm_routed"), (33, 2048, 8448, False, "m64w2"),
    (64, 128, 8448, True, "m64w1_swiglu"), (65, 128, 8448, True, "eek_gemm_routed_swiglu"),
    (128, 128, 8192, True, "m64w1_swiglu"), (129, 128, 8192, True, "eek_gemm_routed_swiglu")])
def test_routed_choice(ee, M, K, N, sw, kernel):
    pw, g = _weight(ee, N, K, seed=M)
    x = torch.randn(M, K, generator=g, device="cuda").half()
    _, idx, cnt = ee.route(torch.randint(1, 4, (M,), generator=g, device="cuda").float(), 1.5, 2.5)
    out = ee.routed_linear(x, pw, idx, cnt, swiglu=sw)
    assert _last_kernel() == (kernel if kernel.startswith("eek") else "eek_gemm_routed_" + kernel)
    _opt(1)
    assert torch.equal(_bits(ee.routed_linear(x, pw, idx, cnt, swiglu=sw)), _bits(out))


# the form with half the LDS (8 KB chunks: one stage of 33 to 64 rows, one of FP8's 64), which LM heads and wide projections
# of up to 64 rows take; N with a remainder, K of one stage, five and nine
@pytest.mark.parametrize("counts", [(1, 0, 0), (3, 4, 1), (16, 17, 31), (0, 0, 64), (0, 64, 0), (64, 0, 0), (5, 40, 19)])
@pytest.mark.parametrize("K,N", [(128, 32004), (640, 11008), (1152, 11012)])
def test_dense_routed_bits(ee, counts, K, N):
    M = sum(counts)
    pw, g = _weight(ee, N, K, seed=M)
    x = torch.randn(M, K, generator=g, device="cuda").half()
    h = torch.cat([torch.full((c,), t + 1.0) for t, c in enumerate(counts)])[torch.randperm(M)].cuda()
    _, idx, cnt = ee.route(h, 1.5, 2.5)
    _opt(1)
    ref = ee.routed_linear(x, pw, idx, cnt)
    assert "m64" not in _last_kernel()
    _opt(0)
    out = torch.full_like(ref, float("nan"))
    ee.routed_linear(x, pw, idx, cnt, out=out)
    assert _last_kernel() == "eek_gemm_routed_m64w2_dense"
    assert torch.equal(_bits(out), _bits(ref))
