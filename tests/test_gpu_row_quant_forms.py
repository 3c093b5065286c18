"""Every form of the whole-row quantiser whose arithmetic the 6-bit and the nibble output share: the 6-bit codes are those of the
nibbles, re-encoded, for every row length it has, with and without the norm, its weight, the residual addition and the
rotation, clipped and with degenerate rows; rows behind the norm against float32 arithmetic in the order of the reference."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def rows(m, k, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(m, k, device="cuda", generator=g).half()
    x[0] = 0
    x[1] = (torch.randn(k, device="cuda", generator=g) * 2e-5).half()          # a subnormal scale
    x[2] = 0
    x[2, 17] = -1
    x[3, ::2] = 500
    x[4] = -x[5]
    return x


@pytest.mark.parametrize("clip", [1.0, 0.7])
@pytest.mark.parametrize("hadamard", [True, False])
@pytest.mark.parametrize("k", [512, 1024, 2048, 4096, 8192])
def test_six_bit_codes_are_the_nibbles(k, hadamard, clip):
    from flh_amd import _ops as ops
    m = 1037 if k <= 4096 else 131
    x, add, w = rows(m, k, k), rows(m, k, k + 1), (torch.rand(k, device="cuda") + 0.5).half()
    q, s = ops.rotate_and_quantize_i4(x, hadamard, clip_ratio=clip)
    e, t = ops.rotate_and_quantize_f6(x, hadamard, clip)
    assert torch.equal(e, ops.encode_f6(q)) and torch.equal(s, t)
    for weight in (w, None):
        q, s = ops.rmsnorm_rotate_and_quantize_i4(x, weight, 1e-5, hadamard, clip)
        e, t = ops.rotate_and_quantize_f6(x, hadamard, clip, weight, 1e-5)
        assert torch.equal(e, ops.encode_f6(q)) and torch.equal(s, t)
        total, q, s = ops.add_rmsnorm_rotate_and_quantize_i4(x, add, weight, 1e-5, hadamard, clip)
        total6, e, t = ops.rotate_and_quantize_f6(x, hadamard, clip, weight, 1e-5, add)
        assert torch.equal(e, ops.encode_f6(q)) and torch.equal(s, t)
        assert torch.equal(total, x + add) and torch.equal(total6, total)


@pytest.mark.parametrize("weighted", [True, False])
def test_norm_in_float32(weighted):
    """Against the norm as its own launch (whose roundings the parity tests pin), up to the order of the squares' sum: every
    normalised value is within one fp16 step of it."""
    from flh_amd import _ops as ops
    x, w = rows(700, 4096, 3), (torch.rand(4096, device="cuda") + 0.5).half() if weighted else None
    y = ops.rmsnorm_rotate_and_quantize_i4(x, w, 1e-5, False, return_rotated=True)[2]
    want = ops.add_rmsnorm(x, w, 1e-5)
    assert torch.isfinite(y).all() and ((y.float() - want.float()).abs() <= want.float().abs() * 2.0 ** -10 + 2.0 ** -24).all()


@pytest.mark.parametrize("k", [11008, 14336])
def test_dense_rotation_of_rows_one_after_the_other_agrees_with_long_batches(k):
    """One row at a time per workgroup, up to three one after the other (768 rows), against the kernel of long batches: the same bytes on
    both sides of every round of 256 workgroups."""
    from flh_amd import _ops as ops
    x = torch.randn(1300, k, generator=torch.Generator().manual_seed(k)).half()
    x[::97] = 0
    x[5, 3], x[300, 7] = 60000.0, 1e-7
    x = x.cuda()
    q_long, s_long = ops.rotate_and_quantize_i4(x)
    for m in (1, 255, 256, 257, 511, 512, 513, 767, 768, 769, 1023, 1024, 1025):
        print(f"case dense k={k} m={m}", flush=True)
        q, s = ops.rotate_and_quantize_i4(x[1300 - m:].contiguous())
        assert torch.equal(q, q_long[1300 - m:]) and torch.equal(s, s_long[1300 - m:]), m
