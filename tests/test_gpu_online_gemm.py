"""The GEMM that quantises its own activations: every prologue, tile count and token count against the quantiser's and the
GEMM's own launches, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu

K = 4096


@pytest.fixture(scope="module")
def ops():
    assert torch.cuda.is_available(), "these tests need the GPU"
    from flh_amd import _ops
    return _ops


def make(ns, cols, seed, offset=0):
    """Weights and scales of `ns` channels; offset: halves by which the scales miss the 16-byte alignment."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    Bs = [torch.randint(0, 256, (n, K // 2), dtype=torch.uint8, device="cuda", generator=gen) for n in ns]
    Ss = []
    for n in ns:
        flat = torch.empty(n * cols + offset, dtype=torch.float16, device="cuda").uniform_(0.005, 0.02, generator=gen)
        Ss.append(flat[offset:].view(n, cols))
    x = torch.randn(8, K, device="cuda", generator=gen).half()
    x[:, ::100] *= 20
    add = torch.randn(8, K, device="cuda", generator=gen).half()
    w = (torch.rand(K, device="cuda", generator=gen) + 0.5).half()
    return x, add, w, Bs, Ss


# one tile per workgroup, a ragged last tile, every tile count, more tiles than one round of workgroups (two of five and of six), several
# matrices
CHANNELS = [(16,), (40, 8), (4096, 24, 1000), (8200,), (12300,), (16000, 40), (24000,), (28672,), (33000,), (44000, 1100)]


@pytest.mark.parametrize("ns", CHANNELS)
@pytest.mark.parametrize("cols", [1, 32])
def test_whole_rows(ops, ns, cols):
    x, add, w, Bs, Ss = make(ns, cols, sum(ns) + cols)
    for m in (1, 2, 3, 4):
        q, a = ops.rotate_and_quantize_i4(x[:m], hadamard="exact")
        for B, S, got in zip(Bs, Ss, ops.rotate_quantize_gemm_i4_multi(x[:m], Bs, Ss)):
            assert torch.equal(got, ops.gemm_i4_dequant(q, B, a, S, 128)), ("rotation", m, B.size(0))
        for addend in (None, add[:m].contiguous()):
            for weight in (w, None):
                total, outs = ops.rmsnorm_rotate_quantize_gemm_i4_multi(x[:m], addend, weight, 1e-5, Bs, Ss)
                stream = x[:m] if addend is None else x[:m] + addend
                assert addend is None or torch.equal(total, stream)
                q, a = ops.rmsnorm_rotate_and_quantize_i4(stream, weight, 1e-5)
                for B, S, got in zip(Bs, Ss, outs):
                    assert torch.equal(got, ops.gemm_i4_dequant(q, B, a, S, 128)), (m, addend is None, weight is None, B.size(0))


@pytest.mark.parametrize("ns", CHANNELS)
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("through", ["ctypes", "extension"])
def test_groups(ops, ns, offset, through):
    """The one launch (ctypes) and what the decoder layer calls: one launch or two, by tokens and channels (extension)."""
    import flh_amd._ext_ops as extension
    op = (ops if through == "ctypes" else extension).rmsnorm_group_quantize_gemm_i4_multi
    x, _, w, Bs, Ss = make(ns, 32, sum(ns) + 7, offset)
    for m in (1, 2, 3, 4):
        for weight in (w, None):
            outs = op(x[:m], weight, 1e-5, Bs, Ss)
            q, a = ops.rmsnorm_and_quantize_i4_gs(x[:m].contiguous(), weight, 1e-5, 128, False)
            for B, S, got in zip(Bs, Ss, outs):
                assert torch.equal(got, ops.gemm_i4_dequant(q.view(m, -1), B, a.view(m, -1), S, 128)), (m, weight is None, B.size(0))


def test_a_norm_weight_off_the_alignment(ops):
    """The one launch needs it aligned; the extension takes two."""
    import flh_amd._ext_ops as extension
    x, _, w, Bs, Ss = make((600, 40), 32, 9)
    moved = torch.cat((w[:1], w))[1:]
    assert moved.data_ptr() % 16 and moved.is_contiguous()
    for m in (1, 3):
        want = extension.rmsnorm_group_quantize_gemm_i4_multi(x[:m], w, 1e-5, Bs, Ss)
        assert all(torch.equal(a, b) for a, b in zip(extension.rmsnorm_group_quantize_gemm_i4_multi(x[:m], moved, 1e-5, Bs, Ss), want))


def test_scales_off_the_alignment(ops):
    x, add, w, Bs, Ss = make((600, 40), 32, 3, offset=1)
    for m in (1, 2, 4):
        total, outs = ops.rmsnorm_rotate_quantize_gemm_i4_multi(x[:m], add[:m].contiguous(), w, 1e-5, Bs, Ss)
        q, a = ops.rmsnorm_rotate_and_quantize_i4(total, w, 1e-5)
        for B, S, got in zip(Bs, Ss, outs):
            assert torch.equal(got, ops.gemm_i4_dequant(q, B, a, S, 128)), m


@pytest.mark.parametrize("value", [0.0, float("inf"), float("nan"), 6e-8, 65504.0])
def test_rows_of_one_value(ops, value):
    """Rows without a maximum, with infinities and NaN, and of subnormal scale quantise as in their own launch."""
    x, _, w, Bs, Ss = make((160,), 32, 5)
    x[1, :] = value
    x[2, 130] = value
    q, a = ops.rotate_and_quantize_i4(x[:4], hadamard="exact")
    want = ops.gemm_i4_dequant(q, Bs[0], a, Ss[0], 128)
    assert torch.equal(ops.rotate_quantize_gemm_i4(x[:4], Bs[0], Ss[0]).view(torch.int16), want.view(torch.int16))
    assert torch.equal(ops.rotate_quantize_gemm_i4(x[1:2], Bs[0], Ss[0]).view(torch.int16), want[1:2].view(torch.int16))
    q, a = ops.rmsnorm_and_quantize_i4_gs(x[:4].contiguous(), w, 1e-5, 128, False)
    want = ops.gemm_i4_dequant(q.view(4, -1), Bs[0], a.view(4, -1), Ss[0], 128)
    got = ops.rmsnorm_group_quantize_gemm_i4_multi(x[:4], w, 1e-5, Bs, Ss)[0]
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
