"""The small-tile kernel between decoding and prefill (gemm_i4_stream.hip) where it can go wrong: rows and channels that end
inside a tile, the shortest K it takes, K whose last stage of four groups is short, more scale pairs than one load
instruction holds, several weight matrices, residual and rotary epilogues, both sides of its dispatch rule.  The sums are
exact integers and the epilogues' roundings are specified, so the bar is equality with the tile and decode kernels (reached
by forcing a tile), which the parity tests pin to the oracle."""
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


def operands(m, ns, k, kind, seed):
    a_cols, b_cols = {"row": (1, 1), "token": (1, k // 128), "group": (k // 128, k // 128)}[kind]
    rng = np.random.default_rng(seed)
    a = dev(rng.integers(0, 256, size=(m, k // 2), dtype=np.uint8))
    ws = [dev(rng.integers(0, 256, size=(n, k // 2), dtype=np.uint8)) for n in ns]
    return a, ws, dev(syn.weight_scales(m, a_cols, seed + 1)), [dev(syn.weight_scales(n, b_cols, seed + 2 + i)) for i, n in enumerate(ns)]


KINDS = ["row", "token", "group"]
# 16 x 64, 32 x 32 and 64 x 32 tiles; K of one stage, of stages the last of which is short, and the longest with a table
SHAPES = [(5, 11010, 512), (4, 12304, 512), (2, 17408, 512), (7, 22016, 512), (16, 11013, 768), (1, 14336, 2816), (17, 36, 512), (33, 250, 768), (45, 1023, 11008), (64, 64, 16384),
          (65, 100, 1280), (100, 1030, 1024), (127, 8200, 512), (250, 2090, 2816), (64, 20000, 768)]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_plain_and_residual(ops, gemm_tuning, m, n, k, kind):
    print(f"case stream {m}x{n}x{k} {kind}", flush=True)
    a, (w,), sa, (sw,) = operands(m, [n], k, kind, m + n)
    res = dev(np.random.default_rng(7).standard_normal((m, n)).astype(np.float16))
    got, got_add = ops.gemm_i4_dequant(a, w, sa, sw, 128), ops.gemm_i4_dequant_add(a, w, sa, sw, res, 128)
    gemm_tuning(64)
    assert torch.equal(got, ops.gemm_i4_dequant(a, w, sa, sw, 128))
    assert torch.equal(got_add, ops.gemm_i4_dequant_add(a, w, sa, sw, res, 128))


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("m", [16, 40, 130])
def test_several_weight_matrices(ops, gemm_tuning, m, kind):
    ns, k = [8200, 2056, 1100], 768
    a, ws, sa, sw = operands(m, ns, k, kind, m)
    got = ops.gemm_i4_dequant_multi(a, ws, sa, sw, 128)
    gemm_tuning(64)
    assert all(torch.equal(g, w) for g, w in zip(got, ops.gemm_i4_dequant_multi(a, ws, sa, sw, 128)))


@pytest.mark.parametrize("kind", ["token", "group"])
@pytest.mark.parametrize("batch,t", [(1, 65), (3, 40), (2, 129)])
def test_rotary_and_cache(ops, gemm_tuning, batch, t, kind):
    hq, hkv, k, length = 4, 2, 768, t + 9
    a, ws, sa, sw = operands(batch * t, [hq * 128, hkv * 128, hkv * 128], k, kind, t)
    rng = np.random.default_rng(t)
    cos, sin = (dev(rng.standard_normal((t, 128)).astype(np.float16)) for _ in range(2))
    pos = torch.arange(5, 5 + t, device="cuda")
    outs = []
    for tile in (0, 128):
        gemm_tuning(tile)
        caches = [torch.zeros(batch, hkv, length, 128, dtype=torch.float16, device="cuda") for _ in range(2)]
        outs.append([ops.gemm_i4_qkv_rope(a, sa, ws, sw, cos, sin, pos, *caches, batch), *caches])
    assert all(torch.equal(x, y) for x, y in zip(*outs))


def test_scales_that_dword_loads_cannot_fetch(ops, gemm_tuning):
    """An odd number of groups, and scales at an odd element offset: the other kernels serve them."""
    for k, offset in ((1152, 0), (1024, 1)):
        a, (w,), sa, (sw,) = operands(40, [96], k, "group", k)
        sw = torch.cat([sw.flatten()[:1]] * offset + [sw.flatten()])[offset:].view(sw.shape)
        got = ops.gemm_i4_dequant(a, w, sa, sw, 128)
        gemm_tuning(64)
        assert torch.equal(got, ops.gemm_i4_dequant(a, w, sa, sw, 128))
        gemm_tuning(0)
