"""Up to sixteen tokens on packed codes: which kernel takes a launch by the share of K that its waves fill, the channels and the tokens,
and the outputs on both sides of every line against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    assert torch.cuda.is_available(), "these tests need the GPU"
    from flh_amd import _ops
    return _ops


def operands(m, n, k, scales, seed, offset=0):
    """Codes and scales; offset: halves by which the scales miss the alignment of dword loads."""
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def scale(rows, cols):
        flat = torch.empty(rows * cols + offset, dtype=torch.float16, device="cuda").uniform_(0.005, 0.02, generator=gen)
        return flat[offset:].view(rows, cols)
    q = torch.randint(0, 256, (m, k // 2), dtype=torch.uint8, device="cuda", generator=gen)
    w = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device="cuda", generator=gen)
    return q, w, scale(m, k // 128 if scales == "group" else 1), scale(n, 1 if scales == "row" else k // 128)


def same_as_oracle(got, q, w, a, s):
    """All tokens of the first, some middle and the last (ragged) channels."""
    from oracle.gemm import gemm_i4_dequant
    n = w.size(0)
    for lo, hi in {(0, min(n, 32)), (n // 2, min(n, n // 2 + 17)), (max(0, n - 40), n)}:
        want, _ = gemm_i4_dequant(q.cpu().numpy(), w[lo:hi].cpu().numpy(), a.cpu().numpy(), s[lo:hi].cpu().numpy())
        assert np.array_equal(got[:, lo:hi].cpu().numpy().view(np.uint16), want.view(np.uint16)), (lo, hi)


def kernel_of(call):
    """Name of the one kernel that `call` launches."""
    call()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    names = [e.name for e in prof.events() if "gemm_i4" in e.name]
    assert len(names) == 1, names
    return names[0]


KERNELS = {"dot": "gemm_i4_dot_kernel", "lines": "gemm_i4_lines_kernel", "half": "gemm_i4_decode_kernel", "stream": "gemm_i4_stream_kernel",
           "dealt": "gemm_i4_dealt_kernel"}

# tokens, channels, K, scales, kernel.  A wave has room for 2, 4, 6 or 8 steps of 2048 codes: rows that fill less than that and few tokens
# on wide launches are where the kernels change places.
ROUTES = [
    # full shares
    (1, 4096, 4096, "row", "dot"), (4, 4096, 4096, "token", "dot"), (8, 4096, 4096, "group", "lines"), (16, 4096, 4096, "row", "lines"),
    (5, 13824, 4096, "group", "lines"), (9, 13824, 4096, "group", "stream"), (5, 13824, 8192, "row", "lines"), (4, 16384, 8192, "group", "dot"),
    # a share of two steps half full and less
    (1, 1000, 512, "row", "half"), (16, 1000, 512, "token", "half"), (2, 2048, 1024, "group", "half"), (8, 16384, 1024, "row", "dealt"),
    (3, 16384, 1024, "group", "stream"), (2, 2048, 1792, "row", "dot"), (3, 8192, 2048, "token", "half"), (16, 8192, 2048, "group", "half"),
    (8, 8192, 2048, "row", "lines"),
    # of four, five eighths full
    (3, 5120, 5120, "row", "half"), (16, 5120, 5120, "group", "half"), (8, 13824, 5120, "token", "stream"), (4, 13824, 5120, "group", "stream"),
    (8, 13824, 5120, "row", "dealt"), (2, 13824, 5120, "row", "dealt"), (2, 18432, 5120, "row", "dot"), (1, 13824, 5120, "group", "dot"),
    # of four, nearly full
    (4, 5120, 6656, "group", "dot"), (8, 5120, 6656, "group", "lines"), (8, 3072, 6400, "group", "half"), (5, 18432, 7936, "row", "lines"),
    (5, 13824, 7168, "row", "dealt"), (8, 2048, 8192, "group", "half"),
    # of six and eight
    (5, 3072, 9728, "row", "lines"), (5, 10240, 9728, "row", "half"), (5, 8192, 12800, "row", "half"), (2, 13824, 15360, "row", "dealt"),
    (2, 16384, 12416, "group", "dot"),
    # an odd number of groups
    (16, 3072, 3456, "group", "half"), (16, 4096, 3200, "row", "half"), (5, 11008, 3200, "row", "lines"),
]


@pytest.mark.parametrize("m,n,k,scales,kernel", ROUTES)
def test_routes(ops, m, n, k, scales, kernel):
    q, w, a, s = operands(m, n, k, scales, m + n + k)
    name = kernel_of(lambda: ops.gemm_i4_dequant(q, w, a, s, 128))
    assert KERNELS[kernel] in name, name
    same_as_oracle(ops.gemm_i4_dequant(q, w, a, s, 128), q, w, a, s)


# whole lines through LDS: every share, full and not, a row that ends in half a line (K = 128 * odd), a ragged last tile
@pytest.mark.parametrize("n,k", [(40, 2048), (8200, 2176), (8200, 3456), (50, 3840), (50, 4096), (50, 5376), (50, 8192), (50, 9728), (50, 12288),
                                 (50, 12800), (50, 16384)])
def test_lines_one_scale_per_row(ops, n, k):
    for m in (5, 16):
        for offset in (0, 1):
            q, w, a, s = operands(m, n, k, "row", n + k + m, offset)
            same_as_oracle(ops.gemm_i4_dequant(q, w, a, s, 128), q, w, a, s)
        r = torch.randn(m, n, device="cuda").half()
        assert torch.equal(ops.gemm_i4_dequant_add(q, w, a, s, r, 128), r + ops.gemm_i4_dequant(q, w, a, s, 128))
    assert KERNELS["lines"] in kernel_of(lambda: ops.gemm_i4_dequant(q, w, a, s, 128))


@pytest.mark.parametrize("n,k", [(50, 3328), (50, 3584), (50, 4096), (5130, 6400), (5130, 7168), (3080, 7936), (3080, 8192)])
@pytest.mark.parametrize("scales", ["token", "group"])
def test_lines_group_scales(ops, n, k, scales):
    for m in (5, 11, 16):
        for offset in (0, 1, 2):
            q, w, a, s = operands(m, n, k, scales, n + k + m, offset)
            same_as_oracle(ops.gemm_i4_dequant(q, w, a, s, 128), q, w, a, s)
        r = torch.randn(m, n, device="cuda").half()
        assert torch.equal(ops.gemm_i4_dequant_add(q, w, a, s, r, 128), r + ops.gemm_i4_dequant(q, w, a, s, 128))
    assert KERNELS["lines"] in kernel_of(lambda: ops.gemm_i4_dequant(q, w, a, s, 128))


def test_lines_of_several_matrices(ops):
    """q / k / v and gate / up in one launch: the channels of all of them count."""
    ns, k = (4096, 1024, 1030), 6400
    q, _, a, _ = operands(8, 16, k, "group", 1)
    ws, ss = zip(*(operands(8, n, k, "group", n)[1::2] for n in ns))
    call = lambda: ops.gemm_i4_dequant_multi(q, list(ws), a, list(ss), 128)
    assert KERNELS["lines"] in kernel_of(call)
    for got, w, s in zip(call(), ws, ss):
        same_as_oracle(got, q, w, a, s)
