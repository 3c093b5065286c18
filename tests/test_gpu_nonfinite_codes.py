"""Rows that hold infinities and NaN: every quantiser that writes the 6-bit operand format gives the codes of the nibbles, re-encoded,
and the same scales -- also for values whose quotient is NaN, which the hardware's conversion knows no whole number for."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")


def poisoned(m, k, seed):
    """Rows of every kind, dealt out by index so that each wave and each workgroup has some, and plain rows between them."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(m, k, device="cuda", generator=g).half()
    for i, row in enumerate(range(0, m, 3)):
        kind = i % 10
        if kind == 0:
            x[row, (37 * i) % k] = NAN
        elif kind == 1:
            x[row, (53 * i) % k] = INF if i % 4 else -INF
        elif kind == 2:
            x[row, 5], x[row, k - 9] = INF, -INF
        elif kind == 3:
            x[row] = NAN
        elif kind == 4:
            x[row, 11], x[row, k // 2 + 3] = NAN, INF
        elif kind == 5:
            x[row] = 60000.0                        # sums beyond fp16 in a rotation
        elif kind == 6:
            x[row, 1::2], x[row, ::2] = 65504.0, -65504.0
            x[row, 0] = 65504.0
        elif kind == 7:
            x[row] = (x[row] * 2e-5).half()         # a subnormal scale next to a NaN: clamped quotients
            x[row, 64] = NAN
        elif kind == 8:
            x[row, ::128] = NAN                     # one in every group
        else:
            x[row] = INF
    return x


def same(got, want):
    return torch.equal(got[0], want[0]) and torch.equal(got[1].view(torch.int16), want[1].view(torch.int16))


@pytest.mark.parametrize("hadamard", [True, False])
@pytest.mark.parametrize("m,k", [(9, 128), (64, 1024), (401, 4096), (601, 4096), (2049, 4096)])   # sixteen lanes per group, then four
def test_groups(m, k, hadamard):
    from flh_amd import _ops as ops
    x = poisoned(m, k, m)
    q, s = (ops.hadamard_and_quantize_i4 if hadamard else ops.quant_and_pack_i4)(x.view(-1, 128))
    assert same(ops.group_quantize_f6(x, hadamard), (ops.encode_f6(q.view(m, k // 2)), s.view(m, k // 128)))


@pytest.mark.parametrize("hadamard", [True, False])
def test_long_batches_are_their_pieces(hadamard):
    """Four lanes per group and sixteen: the same codes, whatever becomes of a NaN on its way through the sums."""
    from flh_amd import _ops as ops
    x = poisoned(2049 * 32, 128, 1)
    op = ops.hadamard_and_quantize_i4 if hadamard else ops.quant_and_pack_i4
    pieces = [op(p.clone()) for p in x.split(8192)]
    assert same(op(x), [torch.cat([p[i] for p in pieces]) for i in range(2)])


@pytest.mark.parametrize("m,k", [(64, 1024), (401, 4096), (601, 11008)])
def test_groups_behind_the_norm_and_the_product(m, k):
    from flh_amd import _ops as ops
    x, up = poisoned(m, k, m), torch.randn(m, k, device="cuda").half()
    w = (torch.rand(k, device="cuda") + 0.5).half()
    q, s = ops.rmsnorm_and_quantize_i4_gs(x, w, 1e-5, 128, False)
    assert same(ops.rmsnorm_group_quantize_f6(x, w, 1e-5), (ops.encode_f6(q.view(m, k // 2)), s.view(m, k // 128)))
    q, s = ops.silu_mul_and_quantize_i4_gs(x, up, 128, False)
    assert same(ops.silu_mul_group_quantize_f6(x, up), (ops.encode_f6(q.view(m, k // 2)), s.view(m, k // 128)))


@pytest.mark.parametrize("clip", [1.0, 0.7])
@pytest.mark.parametrize("k,hadamard", [(k, h) for k in (512, 1024, 2048, 4096, 8192) for h in (True, False)] + [(4096, "fast")])
def test_whole_rows(k, hadamard, clip):
    from flh_amd import _ops as ops
    m = 331
    x, add, w = poisoned(m, k, k), torch.randn(m, k, device="cuda").half(), (torch.rand(k, device="cuda") + 0.5).half()
    q, s = ops.rotate_and_quantize_i4(x, hadamard, clip_ratio=clip)
    assert same(ops.rotate_and_quantize_f6(x, hadamard, clip), (ops.encode_f6(q), s))
    if hadamard == "fast":
        return
    q, s = ops.rmsnorm_rotate_and_quantize_i4(x, w, 1e-5, hadamard, clip)
    assert same(ops.rotate_and_quantize_f6(x, hadamard, clip, w, 1e-5), (ops.encode_f6(q), s))
    _, q, s = ops.add_rmsnorm_rotate_and_quantize_i4(x, add, w, 1e-5, hadamard, clip)
    assert same(ops.rotate_and_quantize_f6(x, hadamard, clip, w, 1e-5, add)[1:], (ops.encode_f6(q), s))


@pytest.mark.parametrize("k", [11008, 14336])
def test_dense_factors(k):
    from flh_amd import _ops as ops
    m = 1037                                        # (the kernel of long batches on both sides)
    x = poisoned(m, k, k)
    q, s = ops.rotate_and_quantize_i4(x, "fast")
    assert same(ops.rotate_and_quantize_f6(x, "fast"), (ops.encode_f6(q), s))
