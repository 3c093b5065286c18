"""The group quantiser on long batches (four lanes per group of 128): the sizes around the lines from which it is taken, a
last workgroup that is not full, and the rows whose scale is degenerate, against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def rows_of(r, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((r, 128)).astype(np.float16)
    x[:, rng.integers(0, 128, 2)] *= np.float16(20)
    x[5] = 0
    x[6] = (rng.standard_normal(128) * 2e-5).astype(np.float16)        # a subnormal scale: clamped quotients
    x[7] = 0
    x[7, 17] = 1.0
    x[-1] = np.float16(6e-8)                                          # s <= 1e-6
    x[-2, ::2] = np.float16(500)
    return x


@pytest.mark.parametrize("f6", [False, True])
@pytest.mark.parametrize("had", [False, True])
@pytest.mark.parametrize("r", [16383, 16384, 16384 + 37, 49152 + 37, 65536 + 64 * 3 + 1])
def test_long_batches_bit_exact(r, had, f6):
    from flh_amd import _ops
    from oracle import pack, quant
    x = rows_of(r, r + had)
    q_ref, s_ref, _ = quant.kernel_had_and_quant(x, 128, had)
    xd = torch.from_numpy(x).cuda()
    if f6:
        k = 1024 if r % 8 == 0 else 128                               # several slabs, or one
        encoded, s = _ops.group_quantize_f6(xd.view(-1, k), had)
        assert torch.equal(encoded, _ops.encode_f6(torch.from_numpy(pack.pack_i4(q_ref)).cuda().view(-1, k // 2)))
    else:
        q, s = (_ops.hadamard_and_quantize_i4 if had else _ops.quant_and_pack_i4)(xd)
        assert np.array_equal(q.cpu().numpy(), pack.pack_i4(q_ref))
    assert np.array_equal(s.cpu().numpy().view(np.uint16).ravel(), s_ref.view(np.uint16).ravel())
