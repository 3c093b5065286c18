"""The eight-wave 128 x 128 tiles of the int8 kernels for group-scaled weights, forced where they can go wrong: rows and channels
that end inside a tile, the shortest K, a last block of scale groups that is short, several tiles per workgroup, several
weight matrices, every epilogue -- against the 128 x 128 tiles of four waves, which the parity tests pin to the oracle -- and the
largest codes, whose sums use every bit, against the integer sums."""
import numpy as np
import pytest

from flh_amd import synthetic as syn

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("kind", ["token", "group"])
@pytest.mark.parametrize("m,n,k", [(1, 8, 1024), (33, 136, 1792), (127, 120, 1024), (129, 264, 2816), (300, 256, 2048), (1000, 1032, 1792),
                                   (1500, 3464, 1024)])
def test_every_launch_form(gemm_tuning, m, n, k, kind):
    from flh_amd import _ops as ops
    rng = np.random.default_rng(m + n + k)
    a = dev(rng.integers(0, 256, size=(m, k // 2), dtype=np.uint8))
    sa = dev(syn.weight_scales(m, 1 if kind == "token" else k // 128, m))

    def weights(ns):
        return ([dev(rng.integers(0, 256, size=(w, k // 2), dtype=np.uint8)) for w in ns],
                [dev(syn.weight_scales(w, k // 128, int(rng.integers(1 << 30)))) for w in ns])
    ws, sw = weights([n, n, 8 * (n // 24 + 1)])
    heads, kv_heads = n // 128 + 1, n // 256 + 1
    wr, sr = weights([heads * 128, kv_heads * 128, kv_heads * 128])
    res = dev(rng.standard_normal((m, n)).astype(np.float16))
    cos, sin = (dev(rng.uniform(-1, 1, (m, 128)).astype(np.float16)) for _ in range(2))
    pos = torch.arange(3, 3 + m, device="cuda")

    def run():
        caches = [torch.zeros(1, kv_heads, m + 3, 128, dtype=torch.float16, device="cuda") for _ in range(2)]
        return [*ops.gemm_i4_dequant_multi(a, ws, sa, sw, 128), ops.gemm_i4_dequant(a, ws[0], sa, sw[0], 128),
                ops.gemm_i4_dequant_add(a, ws[0], sa, sw[0], res, 128), ops.gemm_i4_swiglu(a, ws[0], ws[1], sa, sw[0], sw[1], 128),
                ops.gemm_i4_qkv_rope(a, sa, wr, sr, cos, sin, pos, *caches, 1, 128), *caches]
    gemm_tuning(128, 1)
    want = run()
    gemm_tuning(128, 2)
    for i, (x, y) in enumerate(zip(run(), want)):
        assert torch.equal(x, y), i


@pytest.mark.parametrize("token", [True, False])
def test_largest_sums(gemm_tuning, token):
    """All codes -8: every group's sum is 8192; scales are powers of two, so the result is exact."""
    from flh_amd import _ops as ops
    m, n, k = 130, 136, 2048
    a, w = torch.full((m, k // 2), 0x88, dtype=torch.uint8, device="cuda"), torch.full((n, k // 2), 0x88, dtype=torch.uint8, device="cuda")
    sa = torch.full((m, 1 if token else k // 128), 2.0 ** -4, device="cuda").half()
    sw = torch.full((n, k // 128), 2.0 ** -5, device="cuda").half()
    gemm_tuning(128, 2)
    assert torch.equal(ops.gemm_i4_dequant(a, w, sa, sw, 128), torch.full((m, n), 64.0 * k / 512, device="cuda").half())


@pytest.mark.parametrize("kind", ["token", "group"])
@pytest.mark.parametrize("m,columns,tiles", [(640, 3584, 140), (1152, 2048, 144), (256, 16384, 256), (256, 16512, 258), (64, 18432, 144),
                                             (65, 18432, 144)])
def test_around_the_lines(m, columns, tiles, kind):
    """The automatic choice on either side of every line: from 144 tiles of 128 x 128 on, with token scales up to 256, plain
    launches from 65 rows on -- the product of gate and up, and q / k / v, whatever the rows."""
    from flh_amd import _ops as ops
    k = 1024
    assert -(-m // 128) * -(-columns // 128) == tiles
    rng = np.random.default_rng(m + columns)

    def weights(n):
        return dev(rng.integers(0, 256, size=(n, k // 2), dtype=np.uint8)), dev(syn.weight_scales(n, 8, n))
    a, sa = dev(rng.integers(0, 256, size=(m, k // 2), dtype=np.uint8)), dev(syn.weight_scales(m, 1 if kind == "token" else 8, m))
    w, sw = weights(columns)
    (gate, sg), (up, su) = weights(columns // 2), weights(columns // 2)
    kv = columns // 128 // 4
    wr, sr = zip(*[weights(n * 128) for n in (columns // 128 - 2 * kv, kv, kv)])
    cos, sin = (dev(rng.uniform(-1, 1, (m, 128)).astype(np.float16)) for _ in range(2))
    pos = torch.arange(m, device="cuda")

    def run():
        caches = [torch.zeros(1, kv, m, 128, dtype=torch.float16, device="cuda") for _ in range(2)]
        return [ops.gemm_i4_dequant(a, w, sa, sw, 128), ops.gemm_i4_swiglu(a, gate, up, sa, sg, su, 128),
                ops.gemm_i4_qkv_rope(a, sa, list(wr), list(sr), cos, sin, pos, *caches, 1, 128), *caches]
    got = run()
    ops.gemm_set_tuning(128, 1)
    try:
        want = run()
    finally:
        ops.gemm_set_tuning(0, 0)
    for i, (x, y) in enumerate(zip(got, want)):
        assert torch.equal(x, y), i
