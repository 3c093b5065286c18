"""Where calls change over to the 6-bit instruction with their weights encoded in the call (group scales on both sides; one scale per
channel), and the encoding of several matrices in one launch."""
import pytest
import torch

from flh_amd.nn import ActQuantizer, LinearFLH

pytestmark = pytest.mark.gpu


def layer(k, n, group):
    src = torch.nn.Linear(k, n, bias=False, device="cuda", dtype=torch.float16)
    return LinearFLH.from_float(src, weight_group_size=group, in_group_size=128, no_hadamard=True)


@pytest.mark.parametrize("k,n,group", [(4096, 4096, 128), (4096, 11008, 128), (11008, 4096, 128), (4096, 4096, -1)])
def test_rows_around_the_line(k, n, group):
    lin, per_token = layer(k, n, group), group < 0
    nibbles = lin._six_bit_rows(group > 0, None, True, not per_token)
    lines = sorted({nibbles, lin._six_bit_rows(group > 0, None, False, not per_token)})
    q = ActQuantizer(bits=4, group_size=128, packed_output=True, per_token=per_token)
    x = torch.randn(lines[-1] + 1, k, device="cuda").half()
    s, z, c = q(x)
    lin.six_bit = "never"
    want = lin(c, s, z, x_is_packed=True)
    lin.six_bit = False
    for m in sorted({l + d for l in lines for d in (-1, 0)}):
        assert torch.equal(lin(c[:m].contiguous(), s[:m].contiguous(), z, x_is_packed=True), want[:m])
        if per_token:
            got = lin.forward_online(x[:m])
            lin.six_bit = "never"
            assert torch.equal(got, lin.forward_online(x[:m]))
            lin.six_bit = False


@pytest.mark.parametrize("rows,k", [((1,), 128), ((31, 33), 384), ((4096, 1024, 1024), 512), ((5, 0, 64, 97), 1664)])
def test_several_matrices_encoded_in_one_launch(rows, k):
    from flh_amd import _ops as ops
    packed = [torch.randint(0, 256, (r, k // 2), dtype=torch.uint8, device="cuda") for r in rows]
    for got, p in zip(ops.encode_f6_many(packed), packed):
        assert torch.equal(got, ops.encode_f6(p))
