"""flh_embed_f16 -- a model step's look-ups in one launch -- against the separate torch launches, bit for bit."""
import math

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hadamard", [False, True])
@pytest.mark.parametrize("shape,hidden,t,dim", [((1, 1), 128, 1, 8), ((5, 1), 4096, 1, 128), ((3, 7), 384, 7, 64), ((1, 33), 1152, 33, 128)])
def test_embed_equals_the_separate_launches(shape, hidden, t, dim, hadamard):
    from flh_amd import _ops as ops
    gen = torch.Generator(device="cuda").manual_seed(hidden + t)
    vocab, max_len = 61, 50
    table = (torch.randn(vocab, hidden, device="cuda", generator=gen) * 3).half()
    table[4, :8] = float("inf")
    cos_t, sin_t = (torch.randn(max_len, dim, device="cuda", generator=gen).half() for _ in range(2))
    ids = torch.randint(0, vocab, shape, device="cuda", generator=gen)
    ids.view(-1)[0] = vocab - 1
    positions = torch.randint(0, max_len, (t,), device="cuda", generator=gen)
    out, cos, sin = ops.embed(ids, table, positions, cos_t, sin_t, hadamard=hadamard)
    want = torch.nn.functional.embedding(ids, table)
    if hadamard:
        want = (ops.hadamard_transform_half(want.clone().view(-1, 128)) / math.sqrt(128)).view(want.shape)
    assert out.shape == want.shape and torch.equal(out.nan_to_num(nan=7.0), want.nan_to_num(nan=7.0))
    assert torch.equal(cos, cos_t.index_select(0, positions)) and torch.equal(sin, sin_t.index_select(0, positions))


def test_indices_outside_the_tables_give_nans():
    from flh_amd import _ops as ops
    table, cos_t = torch.ones(9, 128, device="cuda").half(), torch.ones(6, 16, device="cuda").half()
    out, cos, sin = ops.embed(torch.tensor([[8, 9, -1]], device="cuda"), table, torch.tensor([0, 6, -1], device="cuda"), cos_t, cos_t)
    assert out[0, :, 0].isnan().tolist() == [False, True, True] == cos[:, 0].isnan().tolist() == sin[:, 0].isnan().tolist()
