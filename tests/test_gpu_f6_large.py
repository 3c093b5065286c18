"""The large-tile kernels of the 6-bit matrix instruction (persistent workgroups, 256 x 256 and 256 x 128 tiles), forced where
they can go wrong: rows and channels that end inside a tile, the shortest K they take, K whose last block of eight scale
groups is short, several tiles per workgroup, several weight matrices, every epilogue.  The sums are exact integers and the
epilogues' roundings are specified, so the bar is equality with the library's int8 kernels, which the parity tests pin to
the oracle."""
import numpy as np
import pytest

from flh_amd import synthetic as syn

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from flh_amd import _ops
    return _ops


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def operands(m, ns, k, a_cols, b_cols, seed):
    rng = np.random.default_rng(seed)
    a = dev(rng.integers(0, 256, size=(m, k // 2), dtype=np.uint8))
    ws = [dev(rng.integers(0, 256, size=(n, k // 2), dtype=np.uint8)) for n in ns]
    sa = dev(syn.weight_scales(m, a_cols, seed + 1))
    sw = [dev(syn.weight_scales(n, b_cols, seed + 2 + i)) for i, n in enumerate(ns)]
    return a, ws, sa, sw


# (tile, K split) of the tuning hook: the 256 x 256 tile, the 256 x 128 tile
TILES = [(256, 1), (256, 2)]
SHAPES = [(1, 8, 1024), (31, 136, 1024), (255, 128, 1792), (257, 264, 1024), (300, 256, 4096), (513, 392, 2048), (1000, 1032, 1792)]


def scale_columns(kind, k):
    return {"row": (1, 1), "token": (1, k // 128), "group": (k // 128, k // 128)}[kind]


@pytest.mark.parametrize("kind,tile", [("row", TILES[0]), ("row", TILES[1]), ("token", TILES[1]), ("group", TILES[1])])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_plain_and_residual(ops, gemm_tuning, m, n, k, kind, tile):
    a_cols, b_cols = scale_columns(kind, k)
    a, (w,), sa, (sw,) = operands(m, [n], k, a_cols, b_cols, m + n)
    res = dev(np.random.default_rng(7).standard_normal((m, n)).astype(np.float16))
    want, want_add = ops.gemm_i4_dequant(a, w, sa, sw, 128), ops.gemm_i4_dequant_add(a, w, sa, sw, res, 128)
    a6, w6 = ops.encode_f6(a), ops.encode_f6(w)
    gemm_tuning(*tile)
    got = ops.gemm_f6_dequant_o16(a6, w6, sa, sw) if kind == "row" else ops.gemm_f6_dequant_o16_gs(a6, w6, sa, sw)
    assert torch.equal(got, want)
    assert torch.equal(ops.gemm_f6_dequant_add(a6, w6, sa, sw, res), want_add)


@pytest.mark.parametrize("kind,tile", [("row", TILES[0]), ("row", TILES[1]), ("token", TILES[1]), ("group", TILES[1])])
@pytest.mark.parametrize("m,n", [(40, 72), (600, 200), (2100, 1096)])
def test_swiglu(ops, gemm_tuning, m, n, kind, tile):
    k = 1024
    a_cols, b_cols = scale_columns(kind, k)
    a, (g, u), sa, (sg, su) = operands(m, [n, n], k, a_cols, b_cols, m)
    want = ops.gemm_i4_swiglu(a, g, u, sa, sg, su, 128)
    gemm_tuning(*tile)
    assert torch.equal(ops.gemm_f6_swiglu(ops.encode_f6(a), ops.encode_f6(g), ops.encode_f6(u), sa, sg, su), want)


@pytest.mark.parametrize("kind,tile", [("row", TILES[0]), ("row", TILES[1]), ("token", TILES[1]), ("group", TILES[1])])
def test_several_matrices_and_tiles_per_workgroup(ops, gemm_tuning, kind, tile):
    """More tiles than workgroups, three matrices that end inside a tile; two calls, the second on other data."""
    m, ns, k = 2200, [5000, 1032, 3336], 1024
    a_cols, b_cols = scale_columns(kind, k)
    for seed in (1, 2):
        a, ws, sa, sw = operands(m, ns, k, a_cols, b_cols, seed)
        want = ops.gemm_i4_dequant_multi(a, ws, sa, sw, 128)
        a6, w6 = ops.encode_f6(a), [ops.encode_f6(w) for w in ws]
        gemm_tuning(*tile)
        for x, y in zip(ops.gemm_f6_dequant_multi(a6, w6, sa, sw), want):
            assert torch.equal(x, y)
        gemm_tuning(0)


@pytest.mark.parametrize("kind,tile", [("row", TILES[0]), ("row", TILES[1]), ("token", TILES[1]), ("group", TILES[1])])
@pytest.mark.parametrize("batch,t,hq,hkv", [(1, 70, 4, 1), (3, 101, 5, 3), (2, 700, 8, 2)])
def test_qkv_rope(ops, gemm_tuning, batch, t, hq, hkv, kind, tile):
    k, max_len = 1024, t + 9
    a_cols, b_cols = scale_columns(kind, k)
    a, ws, sa, sw = operands(batch * t, [hq * 128, hkv * 128, hkv * 128], k, a_cols, b_cols, t)
    rng = np.random.default_rng(t)
    cos, sin = dev(rng.uniform(-1, 1, (t, 128)).astype(np.float16)), dev(rng.uniform(-1, 1, (t, 128)).astype(np.float16))
    pos = torch.arange(5, 5 + t, device="cuda")
    caches = [torch.zeros(batch, hkv, max_len, 128, dtype=torch.float16, device="cuda") for _ in range(4)]
    want = ops.gemm_i4_qkv_rope(a, sa, ws, sw, cos, sin, pos, caches[0], caches[1], batch, 128)
    gemm_tuning(*tile)
    got = ops.gemm_f6_qkv_rope(ops.encode_f6(a), sa, [ops.encode_f6(w) for w in ws], sw, cos, sin, pos, caches[2], caches[3], batch)
    assert torch.equal(got, want) and torch.equal(caches[2], caches[0]) and torch.equal(caches[3], caches[1])


@pytest.mark.parametrize("kind", ["token", "group"])
@pytest.mark.parametrize("k", [1792, 2048, 2816])
def test_blocks_of_scales_across_tiles(ops, gemm_tuning, kind, k):
    """Several tiles per workgroup with two full blocks of eight scale groups, and with two and three the last of which is short:
    the double buffer's turn carries over into the next tile.  Every form of launch, more than 256 tiles of 256 x 128 each."""
    m, ns, n, hq, hkv = 2200, [5000, 1032, 3336], 2208, 20, 6
    a_cols, b_cols = scale_columns(kind, k)
    a, ws, sa, sw = operands(m, ns, k, a_cols, b_cols, k)
    _, (g, u), _, (sg, su) = operands(m, [n, n], k, a_cols, b_cols, k + 1)
    _, wr, _, sr = operands(m, [hq * 128, hkv * 128, hkv * 128], k, a_cols, b_cols, k + 2)
    rng = np.random.default_rng(k)
    res = dev(rng.standard_normal((m, ns[0])).astype(np.float16))
    cos, sin = (dev(rng.uniform(-1, 1, (m, 128)).astype(np.float16)) for _ in range(2))
    pos = torch.arange(3, 3 + m, device="cuda")
    caches = [torch.zeros(1, hkv, m + 3, 128, dtype=torch.float16, device="cuda") for _ in range(4)]
    want = [*ops.gemm_i4_dequant_multi(a, ws, sa, sw, 128), ops.gemm_i4_dequant_add(a, ws[0], sa, sw[0], res, 128),
            ops.gemm_i4_swiglu(a, g, u, sa, sg, su, 128),
            ops.gemm_i4_qkv_rope(a, sa, wr, sr, cos, sin, pos, caches[0], caches[1], 1, 128), caches[0], caches[1]]
    a6, w6, r6 = ops.encode_f6(a), [ops.encode_f6(w) for w in ws], [ops.encode_f6(w) for w in wr]
    gemm_tuning(256, 2)
    got = [*ops.gemm_f6_dequant_multi(a6, w6, sa, sw), ops.gemm_f6_dequant_add(a6, w6[0], sa, sw[0], res),
           ops.gemm_f6_swiglu(a6, ops.encode_f6(g), ops.encode_f6(u), sa, sg, su),
           ops.gemm_f6_qkv_rope(a6, sa, r6, sr, cos, sin, pos, caches[2], caches[3], 1), caches[2], caches[3]]
    assert all(torch.equal(x, y) for x, y in zip(got, want))
