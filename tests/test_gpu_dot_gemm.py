"""One to four tokens on packed codes: the dot-product kernel against the oracle's contraction, its edges (ragged channels, odd and
short K, scales off the alignment, residual, several matrices) against the int32 accumulators and scales."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    assert torch.cuda.is_available(), "these tests need the GPU"
    from flh_amd import _ops
    return _ops


def codes(rows, k, gen):
    return torch.randint(0, 256, (rows, k // 2), dtype=torch.uint8, device="cuda", generator=gen)


def scales(rows, cols, gen, offset=0):
    flat = torch.empty(rows * cols + offset, dtype=torch.float16, device="cuda").uniform_(0.005, 0.02, generator=gen)
    return flat[offset:].view(rows, cols)


def expected(q, w, a, s, k):
    """The epilogue by its definition, from the oracle's unpacked codes: ascending groups, one float32 fused multiply-add each."""
    from oracle.pack import unpack_i4
    x = unpack_i4(q.cpu().numpy()).astype(np.int64)
    y = unpack_i4(w.cpu().numpy()).astype(np.int64)
    a, s = a.cpu().numpy(), s.cpu().numpy()
    if s.shape[1] == 1 and a.shape[1] == 1:
        return np.float16(np.float32(x @ y.T) * (a.astype(np.float32) * s.astype(np.float32).T))
    out = np.zeros((x.shape[0], y.shape[0]), np.float64)
    for g in range(k // 128):
        part = x[:, g * 128:g * 128 + 128] @ y[:, g * 128:g * 128 + 128].T
        scale = s[:, min(g, s.shape[1] - 1)].astype(np.float64)[None]
        if a.shape[1] > 1:
            scale = np.float64(np.float32(a[:, g].astype(np.float32)[:, None] * np.float32(scale)))
        out = np.float64(np.float32(out + part * scale))   # (float64 holds the product exactly: one rounding to float32)
    if a.shape[1] == 1:
        out = np.float64(np.float32(np.float32(out) * a.astype(np.float32)))
    return np.float16(np.float32(out))


# K: one group, an odd number of groups, a wave's two, four, six and eight double steps, and their edges
@pytest.mark.parametrize("k", [128, 384, 2176, 4096, 4224, 8192, 8320, 11008, 12416, 16384])
@pytest.mark.parametrize("n", [16, 50])
def test_against_the_definition(ops, k, n):
    gen = torch.Generator(device="cuda").manual_seed(k + n)
    kt = k // 128
    for m in (1, 2, 3, 4):
        q, w = codes(m, k, gen), codes(n, k, gen)
        for a_cols, b_cols, offset in {(1, 1, 0), (1, kt, 0), (kt, kt, 0), (kt, kt, 1)}:
            a, s = scales(m, a_cols, gen), scales(n, b_cols, gen, offset)
            got = ops.gemm_i4_dequant(q, w, a, s, 128).cpu().numpy()
            assert np.array_equal(got.view(np.uint16), expected(q, w, a, s, k).view(np.uint16)), (m, a_cols, b_cols, offset)


def test_residual_and_several_matrices(ops):
    gen = torch.Generator(device="cuda").manual_seed(1)
    k, m = 4096, 3
    q, a = codes(m, k, gen), scales(m, 32, gen)
    ws, ss = [codes(n, k, gen) for n in (40, 16, 100)], [scales(n, 32, gen) for n in (40, 16, 100)]
    outs = ops.gemm_i4_dequant_multi(q, ws, a, ss, 128)
    for w, s, got in zip(ws, ss, outs):
        want = ops.gemm_i4_dequant(q, w, a, s, 128)
        assert torch.equal(got, want)
        r = torch.randn(m, w.size(0), device="cuda", generator=gen).half()
        assert torch.equal(ops.gemm_i4_dequant_add(q, w, a, s, r, 128), r + want)
