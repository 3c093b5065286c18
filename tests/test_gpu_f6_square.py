"""The eight-wave 128 x 128 tile of the 6-bit group-scale kernels (and the 256 x 128 one beside it) where it can go wrong: rows and
channels that end inside a tile, the shortest K, a last block of scale groups that is short (the ring of six stages is read
two blocks ahead), several tiles per workgroup, several weight matrices, every epilogue.  Exact sums and specified roundings:
the bar is equality with the int8 kernels."""
import numpy as np
import pytest

from flh_amd import synthetic as syn

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def weights(ns, k, rng):
    return ([dev(rng.integers(0, 256, size=(n, k // 2), dtype=np.uint8)) for n in ns],
            [dev(syn.weight_scales(n, k // 128, int(rng.integers(1 << 30)))) for n in ns])


@pytest.mark.parametrize("tile", [(128, 2), (256, 2)])
@pytest.mark.parametrize("kind", ["token", "group"])
@pytest.mark.parametrize("m,n,k", [(1, 8, 1024), (33, 136, 1792), (127, 120, 1024), (129, 264, 2816), (300, 256, 2048), (1000, 1032, 1792),
                                   (1500, 3464, 1024)])
def test_every_launch_form(gemm_tuning, m, n, k, kind, tile):
    from flh_amd import _ops as ops
    rng = np.random.default_rng(m + n + k)
    a = dev(rng.integers(0, 256, size=(m, k // 2), dtype=np.uint8))
    sa = dev(syn.weight_scales(m, 1 if kind == "token" else k // 128, m))
    ws, sw = weights([n, n, 8 * (n // 24 + 1)], k, rng)
    heads, kv_heads = n // 128 + 1, n // 256 + 1
    wr, sr = weights([heads * 128, kv_heads * 128, kv_heads * 128], k, rng)
    res = dev(rng.standard_normal((m, n)).astype(np.float16))
    cos, sin = (dev(rng.uniform(-1, 1, (m, 128)).astype(np.float16)) for _ in range(2))
    pos = torch.arange(3, 3 + m, device="cuda")
    caches = [torch.zeros(1, kv_heads, m + 3, 128, dtype=torch.float16, device="cuda") for _ in range(4)]
    want = [*ops.gemm_i4_dequant_multi(a, ws, sa, sw, 128), ops.gemm_i4_dequant_add(a, ws[0], sa, sw[0], res, 128),
            ops.gemm_i4_swiglu(a, ws[0], ws[1], sa, sw[0], sw[1], 128),
            ops.gemm_i4_qkv_rope(a, sa, wr, sr, cos, sin, pos, caches[0], caches[1], 1, 128), caches[0], caches[1]]
    a6, w6, r6 = ops.encode_f6(a), [ops.encode_f6(w) for w in ws], [ops.encode_f6(w) for w in wr]
    gemm_tuning(*tile)
    got = [*ops.gemm_f6_dequant_multi(a6, w6, sa, sw), ops.gemm_f6_dequant_add(a6, w6[0], sa, sw[0], res),
           ops.gemm_f6_swiglu(a6, w6[0], w6[1], sa, sw[0], sw[1]),
           ops.gemm_f6_qkv_rope(a6, sa, r6, sr, cos, sin, pos, caches[2], caches[3], 1), caches[2], caches[3]]
    for i, (x, y) in enumerate(zip(got, want)):
        assert torch.equal(x, y), i
