"""flh_linear_f16 (the head of a decode step) against float64.  Bound: the products are exact in float32; a float32 sum of K terms
in any order is off by at most K 2^-24 sum |x w|, and the result is rounded to fp16 (2^-11 relative, half the subnormal step)."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lead,n,k", [((1, 1), 64, 128), ((3, 1), 65, 256), ((16,), 1000, 384), ((5, 1), 77, 512), ((16, 1), 4099, 4096),
                                      ((2,), 32000, 640), ((1, 15), 130, 11008)])
def test_linear_f16(lead, n, k):
    from flh_amd import _ops as ops
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    x = torch.randn(*lead, k, device="cuda", generator=gen).half()
    w = torch.randn(n, k, device="cuda", generator=gen).half()
    y = ops.linear_f16(x, w)
    exact = x.double() @ w.double().t()
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    bound = bound + 2.0 ** -11 * (exact.abs() + bound) + 2.0 ** -25
    assert y.shape == (*lead, n) and bool(((y.double() - exact).abs() <= bound).all())
    assert torch.equal(y, ops.linear_f16(x, w))


def test_linear_f16_argument_errors():
    from flh_amd import _ops as ops
    x, w = torch.zeros(17, 128, device="cuda").half(), torch.zeros(8, 128, device="cuda").half()
    with pytest.raises(RuntimeError):
        ops.linear_f16(x, w)
    with pytest.raises(RuntimeError):
        ops.linear_f16(x[:2, :64].contiguous(), w[:, :64].contiguous())
