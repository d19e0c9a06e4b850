"""The 128-tile routed grid (eek_gemm_routed): every XCD takes an eighth of each tier's tiles,
counted on the device."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def ee():
    import entropy_engine
    from entropy_engine import _lib
    opt = lambda v: _lib.check(_lib.lib().ee_engine_set_option(_lib.engine(), b"gemm_tile", v))
    opt(128)
    yield entropy_engine
    opt(0)


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


@pytest.mark.parametrize("M", [1, 130, 385])
def test_routed_128_tiles_share_of_each_xcd(ee, M):
    """The 128-tile routed grid's tile lists (an eighth of each tier's tiles per XCD), N-tile counts
    that are no multiple of 8, every tier empty in turn: rows equal the per-tier GEMMs'."""
    K, N = 256, 128 * 11 + 4
    pw, g = _weight(ee, N, K, seed=M)
    x = torch.randn(M, K, generator=g, device="cuda").half()
    i8, f8 = ee.quantize_activations(x, "dispatcher"), ee.quantize_activations(x, "fp8")
    refs = [ee.gemm("int8", i8[0], pw.i8, i8[1], pw.scale), ee.gemm("fp8", f8[0], pw.f8, f8[1], pw.scale),
            ee.gemm("fp16", x, pw.f16)]
    for only in (None, 0, 1, 2):
        h = torch.randint(0, 3, (M,), generator=g, device="cuda") + 1.0 if only is None else torch.full((M,), only + 1.0, device="cuda")
        tier, idx, cnt = ee.route(h, 1.5, 2.5)
        out = ee.routed_linear(x, pw, idx, cnt)
        assert _last_kernel() == "eek_gemm_routed"
        ref = torch.stack(refs)[tier.long(), torch.arange(M, device="cuda")]
        assert torch.equal(_bits(out), _bits(ref))
