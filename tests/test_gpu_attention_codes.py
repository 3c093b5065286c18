"""Decode attention that stores the codes of the group quantiser behind it: the bytes of attention and quantiser in their own
launches, and the decoder layer with and without it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    assert torch.cuda.is_available(), "these tests need the GPU"
    from flh_amd import _ops
    return _ops


# heads per key / value head, and cache lengths of one chunk, a chunk's edge, and more chunks than a pass of the combine kernel
@pytest.mark.parametrize("b,hq,hkv,kv_len", [(1, 32, 8, 1), (2, 8, 8, 64), (3, 16, 8, 65), (5, 8, 1, 777), (1, 4, 4, 4200)])
def test_codes_and_scales(ops, b, hq, hkv, kv_len):
    gen = torch.Generator(device="cuda").manual_seed(kv_len)
    rand = lambda *shape: torch.randn(*shape, device="cuda", generator=gen).half()
    q, k, v = rand(b, hq, 128), rand(b, hkv, 128), rand(b, hkv, 128)
    if kv_len > 64:
        v[0, 0, 5] = 300.0
    keys, values = rand(b, hkv, kv_len + 3, 128), rand(b, hkv, kv_len + 3, 128)
    values[0, 0] *= 1e-7                                   # subnormal scales
    cos, sin = rand(128), rand(128)
    positions = torch.tensor([kv_len - 1], device="cuda")
    twins = [keys.clone(), values.clone()]
    out = ops.decode_attention_rope(q, k, v, cos, sin, positions, keys, values, kv_len)
    codes, scales = ops.quant_and_pack_i4_gs(out.view(-1, 128), 128)
    got_codes, got_scales = ops.decode_attention_rope(q, k, v, cos, sin, positions, *twins, kv_len, quantize=True)
    assert torch.equal(got_codes.view(-1, 64), codes) and torch.equal(got_scales.view(-1), scales.view(-1))
    assert torch.equal(keys, twins[0]) and torch.equal(values, twins[1])


def test_heads_of_64_are_refused(ops):
    z = lambda *shape: torch.zeros(*shape, dtype=torch.float16, device="cuda")
    with pytest.raises(RuntimeError):
        ops.decode_attention_rope(z(1, 4, 64), z(1, 4, 64), z(1, 4, 64), z(64), z(64), torch.zeros(1, dtype=torch.int64, device="cuda"),
                                  z(1, 4, 8, 64), z(1, 4, 8, 64), 1, quantize=True)


@pytest.mark.parametrize("batch", [1, 2, 3, 5, 7, 9])
def test_layer_steps(monkeypatch, batch):
    """A decode step of the group configuration: with norm, quantiser and projections in one launch and the codes out of attention's
    combine, with all of these in launches of their own (the same bits), and module by module (the same attention block; the MLP's
    product of silu and up is torch's there, an exponential's last bit apart)."""
    from flh_amd.quantized_model import StaticKVCache, W4A4DecoderLayer
    from flh_amd.quantized_model.decoder_layer import rotary_tables
    gen = torch.Generator(device="cuda").manual_seed(batch)
    h, inter, kv = 4096, 11008, 1024
    dims = {"q_proj": (h, h), "k_proj": (kv, h), "v_proj": (kv, h), "o_proj": (h, h), "gate_proj": (inter, h), "up_proj": (inter, h),
            "down_proj": (h, inter)}
    weights = {name: (torch.randn(n, k, device="cuda", generator=gen) / k ** 0.5).half() for name, (n, k) in dims.items()}
    weights["input_layernorm"] = (torch.rand(h, device="cuda", generator=gen) + 0.5).half()
    layer = W4A4DecoderLayer.from_float(weights, 32, 8, activation="group")
    x = torch.randn(batch, 1, h, device="cuda", generator=gen).half()

    def step(call):
        cache = StaticKVCache(1, batch, 8, 100, 128, "cuda", q_heads=32)
        cache.keys[0].normal_(generator=torch.Generator(device="cuda").manual_seed(1))
        cache.values[0].normal_(generator=torch.Generator(device="cuda").manual_seed(2))
        cache.kv_len = 80
        positions = cache.advance(1)
        cos, sin = rotary_tables(positions, 128)
        with torch.no_grad():
            y, _ = call(x, cos, sin, cache.layer(0), positions)
        return y, cache.keys[0], cache.values[0]

    # the paths that this is about are the ones that are taken
    assert layer._attention_quantises(batch)
    for pair in ((layer.q_proj, layer.k_proj, layer.v_proj), (layer.gate_proj, layer.up_proj)):
        assert layer._online_rows_apply(pair, batch) == (batch <= 4)
    whole, attention = step(layer), step(layer.attention)
    with monkeypatch.context() as apart:
        apart.setattr(layer, "_attention_quantises", lambda rows: False)
        apart.setattr(layer, "_online_rows_apply", lambda layers, rows: False)
        for got, want in ((whole, step(layer)), (attention, step(layer.attention))):
            assert all(torch.equal(g, w) for g, w in zip(got, want))
    layer.fused = False
    assert all(torch.equal(g, w) for g, w in zip(attention, step(layer.attention)))
    modules = step(layer)
    assert torch.equal(whole[1], modules[1]) and torch.equal(whole[2], modules[2])
    err = (whole[0].float() - modules[0].float()).norm() / modules[0].float().norm()
    assert err < 0.02, err
