"""Quantisers that encode the weights their codes are to meet in the same launch (ops with `weights`; no reference counterpart:
its GEMM reads nibbles): the bytes of the quantiser and of encode_f6 by themselves, at the edges of the two parts -- no rows, one
row, ragged blocks of either, both group kernels, the rotations that share a launch and those that do not, more values
than one launch takes."""
import pytest
import torch

import flh_amd as P

pytestmark = pytest.mark.gpu


def _weights(k, rows):
    g = torch.Generator(device="cuda").manual_seed(k + sum(rows))
    return [torch.randint(0, 256, (r, k // 2), dtype=torch.uint8, device="cuda", generator=g) for r in rows]


def _x(m, k):
    g = torch.Generator(device="cuda").manual_seed(m)
    return torch.randn(m, k, generator=g, device="cuda", dtype=torch.float16)


def _same(got, parts, weights):
    expect = list(parts) + [P._CUDA.encode_f6(w) for w in weights]
    assert len(got) == len(expect)
    for a, b in zip(got, expect):
        assert torch.equal(a, b)


ROWS = [(1,), (33, 64, 31), (256, 0, 100, 7)]


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("m,k,hadamard", [(0, 256, False), (1, 128, False), (37, 640, False), (513, 4096, False), (2049, 4096, False), (25601, 4096, False),
                                          (65, 640, True)])
def test_groups(m, k, hadamard, rows):
    x, w = _x(m, k), _weights(k, rows)
    _same(P._CUDA.group_quantize_f6(x, hadamard, weights=w), P._CUDA.group_quantize_f6(x, hadamard), w)


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("m,k", [(0, 256), (1, 128), (37, 640), (130, 4096), (3, 16384)])
def test_norm_and_groups(m, k, rows):
    x, w, norm = _x(m, k), _weights(k, rows), _x(1, k)[0]
    _same(P._CUDA.rmsnorm_group_quantize_f6(x, norm, 1e-5, weights=w), P._CUDA.rmsnorm_group_quantize_f6(x, norm, 1e-5), w)


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("m,k,mode,prologue", [(0, 4096, True, "none"), (1, 4096, True, "none"), (37, 4096, True, "norm"),
                                               (130, 4096, True, "add"), (66, 4096, "fast", "add"), (66, 4096, False, "norm"),
                                               (5, 2048, True, "none"), (33, 11008, "fast", "none")])
def test_rotations(m, k, mode, prologue, rows):
    x, w = _x(m, k), _weights(k, rows)
    args = {"none": {}, "norm": dict(eps=1e-5), "add": dict(eps=1e-5, add=x.flip(0).contiguous(), norm_weight=_x(1, k)[0])}[prologue]
    _same(P._CUDA.rotate_and_quantize_f6(x, hadamard=mode, weights=w, **args),
          P._CUDA.rotate_and_quantize_f6(x, hadamard=mode, **args), w)


def test_refusals():
    x = _x(4, 256)
    for bad in ([], _weights(128, (4,)), _weights(256, (1,) * 5)):
        with pytest.raises(RuntimeError):
            P._CUDA.group_quantize_f6(x, False, weights=bad)


@pytest.mark.parametrize("activation,weight_group,inter,rows", [("group", 128, 11008, (256, 257, 513)), ("group", 128, 14336, (384, 385, 896, 897)),
                                                                ("token", 128, 11008, (257, 512, 513)), ("token", 0, 11008, (1792, 1793, 2048, 2049))])
def test_layer_around_the_lines(activation, weight_group, inter, rows):
    """The row counts from which the parts of a layer (7B and 8B shapes) take the 6-bit instruction with weights encoded beside the
    quantiser: the bits of the int8 kernels, and no encoding kept."""
    from flh_amd.quantized_model import W4A4DecoderLayer, rotary_tables
    h, kv = 4096, 4096 if inter == 11008 else 1024
    g = torch.Generator(device="cuda").manual_seed(inter)
    rand = lambda n, k: (torch.randn(n, k, device="cuda", generator=g) / k ** 0.5).half()
    w = {"q_proj": rand(h, h), "k_proj": rand(kv, h), "v_proj": rand(kv, h), "o_proj": rand(h, h), "gate_proj": rand(inter, h),
         "up_proj": rand(inter, h), "down_proj": rand(h, inter)}
    layer = W4A4DecoderLayer.from_float(w, 32, kv // 128, fused=True, activation=activation, weight_group_size=weight_group)
    x = torch.randn(1, rows[-1], h, device="cuda", generator=g).half()
    taken = set()
    for m in rows:
        cos, sin = rotary_tables(torch.arange(m, device="cuda"), 128)
        layer.set_six_bit(False)
        got = layer(x[:, :m].contiguous(), cos, sin)
        layers = [getattr(layer, n) for n in layer.PROJECTIONS]
        assert all(l._w6 is None for l in layers)
        taken.add(tuple(l.wants_six_bit(m, c, activation == "group") for l, c in ((layer.q_proj, h + 2 * kv), (layer.gate_proj, 2 * inter),
                                                                                  (layer.o_proj, h), (layer.down_proj, h))))
        layer.set_six_bit("never")
        want = layer(x[:, :m].contiguous(), cos, sin)
        assert torch.equal(got[0], want[0]) and all(torch.equal(a, b) for a, b in zip(got[1], want[1]))
    assert len(taken) > 1
