"""The modules' native calls (linear_i4, linear_online_i4, quantize_groups, quantize_rows) against the general path of the same modules, bit for
bit, over the forms a caller may use, and the row counts around which a layer changes its kernel."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


class General:
    """flh_amd._CUDA without the native calls."""

    def __init__(self, ops):
        self._ops = ops

    def __getattr__(self, name):
        return (lambda *a: None) if name in ("linear_i4", "linear_online_i4", "quantize_groups", "quantize_rows") else getattr(self._ops, name)


@pytest.fixture
def both(monkeypatch):
    import flh_amd

    def run(f):
        got = f()
        with monkeypatch.context() as m:
            m.setattr(flh_amd, "_CUDA", General(flh_amd._CUDA))
            return got, f()
    return run


def layer(k, n, group, bias):
    from flh_amd.nn import LinearFLH
    src = torch.nn.Linear(k, n, bias=bias, device="cuda", dtype=torch.float16)
    return LinearFLH.from_float(src, weight_group_size=group, in_group_size=128, no_hadamard=True)


@pytest.mark.parametrize("group,bias", [(128, False), (128, True), (-1, False), (64, False)])
@pytest.mark.parametrize("lead", [(1,), (3, 5), (130,), (2, 330)])
def test_linear_on_quantised_rows(both, lead, group, bias):
    from flh_amd.nn import ActQuantizer
    torch.manual_seed(sum(lead))
    lin, x = layer(512, 264, group, bias), torch.randn(*lead, 512, device="cuda").half()
    for q in (ActQuantizer(bits=4, group_size=128, packed_output=True), ActQuantizer(bits=4, group_size=128, packed_output=True, use_hadamard=False),
              ActQuantizer(bits=4, packed_output=True, per_token=True),
              ActQuantizer(bits=4, packed_output=True, per_token=True, use_hadamard=False, input_clip_ratio=0.9)):
        if group == 64 and not q.per_token:
            continue
        (s, z, c), (s2, z2, c2) = both(lambda: q(x))
        assert torch.equal(s, s2) and torch.equal(c, c2) and s.shape == s2.shape and c.shape == c2.shape and z is None
        got, want = both(lambda: lin(c, s, z, x_is_packed=True))
        assert got.shape == want.shape == (*lead, 264) and torch.equal(got, want)


@pytest.mark.parametrize("hadamard", [True, "exact", "fast"])
@pytest.mark.parametrize("lead", [(1, 1), (2,), (3,), (70,), (2, 700)])
@pytest.mark.parametrize("group", [128, -1])
def test_online_linear(both, lead, group, hadamard):
    torch.manual_seed(len(lead))
    lin, x = layer(4096, 136, group, False), torch.randn(*lead, 4096, device="cuda").half()
    got, want = both(lambda: lin.forward_online(x, hadamard=hadamard))
    assert got.shape == want.shape == (*lead, 136) and torch.equal(got, want)


def test_strided_input_takes_the_general_path(both):
    lin, x = layer(512, 64, 128, False), torch.randn(8, 1024, device="cuda").half()[:, ::2]
    got, want = both(lambda: lin.forward_online(x))
    assert torch.equal(got, want)


@pytest.mark.parametrize("group", [128, -1])
@pytest.mark.parametrize("n", [256, 4096])
def test_rows_around_the_change_to_the_six_bit_instruction(group, n):
    from flh_amd.nn import ActQuantizer
    lin = layer(512, n, group, False)
    rows = lin._six_bit_rows(group > 0)
    q = ActQuantizer(bits=4, group_size=128, packed_output=True, per_token=group < 0)
    x = torch.randn(rows + 1, 512, device="cuda").half()
    s, z, c = q(x)
    y = lin(c, s, z, x_is_packed=True)
    for m in (rows - 1, rows):
        s, z, c = q(x[:m].contiguous())
        assert torch.equal(lin(c, s, z, x_is_packed=True), y[:m])


@pytest.mark.parametrize("k,hadamard", [(4096, True), (4096, "exact"), (4096, "fast"), (11008, True), (11008, "fast")])
@pytest.mark.parametrize("group,bias", [(128, False), (128, True), (-1, False)])
def test_online_linear_around_the_change_to_the_six_bit_instruction(monkeypatch, k, hadamard, group, bias):
    """The last row count that stays on the int8 kernel and the first whose quantiser writes the 6-bit format, also with a leading
    batch dimension: rotate_and_quantize_i4 + gemm_i4_dequant (+ bias)."""
    import flh_amd
    ops, n = flh_amd._CUDA, 4096
    lin = layer(k, n, group, bias)
    first = lin._six_bit_rows(group > 0)
    assert 600 < first <= 2560
    x = torch.randn(first + 1, k, device="cuda").half()
    q, s = ops.rotate_and_quantize_i4(x, hadamard=hadamard)
    want = ops.gemm_i4_dequant(q, lin.w_packed.view(n, k // 2), s, lin.w_scale.view(n, -1), 128)
    if bias:
        want = want + lin.bias
    calls = []

    class Counted(General):
        def __getattr__(self, name):
            calls.append(name)
            return getattr(self._ops, name)
    monkeypatch.setattr(flh_amd, "_CUDA", Counted(ops))
    for rows in (first - 1, first):
        calls.clear()
        y = lin.forward_online(x[:rows], hadamard=hadamard)
        assert ("rotate_and_quantize_f6" in calls) == (rows == first) and torch.equal(y, want[:rows])
    even = first + first % 2
    assert torch.equal(lin.forward_online(x[:even].view(2, -1, k), hadamard=hadamard), want[:even].view(2, -1, n))
    lin.six_bit = "never"
    calls.clear()
    assert torch.equal(lin.forward_online(x, hadamard=hadamard), want) and "rotate_and_quantize_f6" not in calls


@pytest.mark.parametrize("group", [128, -1])
def test_never_keeps_packed_codes_off_the_six_bit_instruction(monkeypatch, group):
    import flh_amd
    lin = layer(4096, 11008, group, False)
    x = torch.randn(2600, 4096, device="cuda").half()
    q, s = flh_amd._CUDA.rotate_and_quantize_i4(x) if group < 0 else flh_amd._CUDA.hadamard_and_quantize_i4(x.view(-1, 128))
    q, s = q.view(2600, -1), s.view(2600, -1)
    want = lin(q, s, x_is_packed=True)
    lin.six_bit = "never"

    class NoEncoding(General):
        def __getattr__(self, name):
            assert name != "encode_f6"
            return getattr(self._ops, name)
    monkeypatch.setattr(flh_amd, "_CUDA", NoEncoding(flh_amd._CUDA))
    assert torch.equal(lin(q, s, x_is_packed=True), want)
