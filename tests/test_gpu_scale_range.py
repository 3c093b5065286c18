"""Scales over the whole range of fp16 in every GEMM kernel: subnormal ones (a quantiser gives them for rows whose largest value is
below 4e-4), zero, the smallest normal ones and the largest.  The kernels take their products from mixed-precision multiply-adds
and from matrix instructions with fp16 inputs; an instruction that flushed subnormal inputs would zero whole rows or channels
here.  Against the oracle, to the last bit of fp16 (the group fold's rounding to float32 is emulated there in float64)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# 2^-24, 1e-6, 5e-5 and 2^-14 - 2^-24 are subnormal or next to it
SMALL = np.array([2.0 ** -24, 1e-6, 5e-5, 2.0 ** -14 - 2.0 ** -24, 2.0 ** -14, 0.0, 0.01, 300.0], np.float16)
LARGE = np.array([65504.0, 2048.0, 100.0, 1.0, 0.02, 2.0 ** -24, 3e-5, 0.5], np.float16)


@pytest.fixture(scope="module")
def ops():
    from flh_amd import _ops
    return _ops


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# kernel: tokens, channels, K, (tile, K split) to force, 6-bit operands
KERNELS = {"decode": (5, 40, 1280, (0, 0), False), "stream_16": (16, 11016, 512, (0, 0), False), "stream": (40, 100, 1280, (0, 0), False),
           "stream_64": (64, 14336, 512, (0, 0), False), "tile_64": (100, 72, 1280, (64, 0), False), "tile_128": (130, 136, 1280, (128, 0), False),
           "tile_256": (260, 136, 1280, (256, 0), False), "f6_64": (70, 72, 1280, (64, 0), True), "f6_128": (130, 136, 1280, (128, 0), True),
           "square": (130, 136, 1792, (128, 2), False), "f6_square": (130, 136, 1792, (128, 2), True),
           "f6_narrow": (260, 136, 1792, (256, 2), True), "f6_wide": (260, 264, 1792, (256, 1), True)}


@pytest.mark.parametrize("kind", ["row", "token", "group"])
@pytest.mark.parametrize("kernel", KERNELS)
def test_against_the_oracle(ops, gemm_tuning, kernel, kind):
    from oracle import gemm as G
    m, n, k, tuning, f6 = KERNELS[kernel]
    a_cols, b_cols = {"row": (1, 1), "token": (1, k // 128), "group": (k // 128, k // 128)}[kind]
    rng = np.random.default_rng(m + n)
    a, w = (rng.integers(0, 256, size=(r, k // 2), dtype=np.uint8) for r in (m, n))
    sa, sw = rng.choice(SMALL, size=(m, a_cols)), rng.choice(LARGE, size=(n, b_cols))
    with np.errstate(over="ignore"):
        want, _ = G.gemm_i4_dequant(a, w, sa, sw)
    ad, wd, sad, swd = dev(a), dev(w), dev(sa), dev(sw)
    gemm_tuning(*tuning)
    if not f6:
        got = ops.gemm_i4_dequant(ad, wd, sad, swd, 128)
    elif kind == "row":
        got = ops.gemm_f6_dequant_o16(ops.encode_f6(ad), ops.encode_f6(wd), sad, swd)
    else:
        got = ops.gemm_f6_dequant_o16_gs(ops.encode_f6(ad), ops.encode_f6(wd), sad, swd)
    got = got.cpu().numpy()
    subnormal = (sa[:, 0] > 0) & (sa[:, 0] < 2.0 ** -14)
    assert subnormal.any() and (np.abs(want[subnormal].astype(np.float32)) > 1e-3).any()      # a flush would show
    if kind == "row":
        assert np.array_equal(got.view(np.uint16), want.view(np.uint16))
        return
    g, v = got.astype(np.float64), want.astype(np.float64)
    assert np.array_equal(np.isinf(g), np.isinf(v)) and not np.isnan(g).any()
    ok = np.isfinite(v)
    # one unit in the last place: where the emulated float32 rounding of a fold differs
    assert (np.abs(g[ok] - v[ok]) <= np.maximum(np.abs(v[ok]) * 2.0 ** -10, 2.0 ** -24)).all()
    assert np.mean(got.view(np.uint16) != want.view(np.uint16)) < 1e-3


@pytest.mark.parametrize("cols", [1, 32])
def test_decode_gemm_with_its_own_quantiser(ops, cols):
    """Tokens whose scales are subnormal or zero, weights over the whole range: the bits of the two launches."""
    from flh_amd import synthetic as syn
    rng = np.random.default_rng(cols)
    x = (syn.activations(3, 4096, seed=1).astype(np.float32) * np.array([[1e-5], [0.0], [1.0]])).astype(np.float16)
    w, s = dev(rng.integers(0, 256, size=(200, 2048), dtype=np.uint8)), dev(rng.choice(LARGE, size=(200, cols)))
    q, a = ops.rotate_and_quantize_i4(dev(x), hadamard="exact")
    assert 0 < float(a[0, 0]) < 2.0 ** -14
    assert torch.equal(ops.rotate_quantize_gemm_i4(dev(x), w, s), ops.gemm_i4_dequant_o16(q, w, a, s))
