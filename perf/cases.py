"""The work that this library is measured by: what its users run, over the range of sizes they run it at.

Four kinds of case, all through the package's public entry points:

  quantize  activations -> int4 codes and scales, ``flh_amd.nn.ActQuantizer``
  linear    quantiser + one W4A4 linear, ``ActQuantizer`` + ``LinearFLH`` or ``LinearFLH.forward_online``
  prefill   a block of new tokens through one decoder layer over a preallocated cache, ``W4A4DecoderLayer``
  decode    one new token per sequence through a stack of layers and the head, the graph that
            ``W4A4LlamaModel.capture_decode_step`` records

A case has either the widths of Llama-2-7B (4096 wide, 32 heads, 11008 in the MLP) or those of Llama-3-8B (4096 wide,
32 query and 8 key / value heads, 14336 in the MLP, 128256 words), and one of the two arrangements of the scales:
"group" (rotation and one scale per 128 channels, weights scaled alike: the reference's own modules and models) and
"token" (the whole row rotated, one scale per token; weights with one scale per output channel or per 128 inputs).
"""
import math

import torch

from flh_amd.nn import ActQuantizer, LinearFLH
from flh_amd.quantized_model import LlamaShape, StaticKVCache, W4A4DecoderLayer, W4A4LlamaModel
from flh_amd.quantized_model.decoder_layer import rotary_tables

DEVICE = "cuda"

# Layers of a decode case.  The stack that users run has 32; the weights of four (450 MB) no longer fit the 256 MB of
# last-level cache either, so every layer's weights come from HBM as they do in the whole stack, and a state is made
# quickly.  The head is there once, as in the whole stack.
DECODE_LAYERS = 4

SHAPES = {"llama2_7b": LlamaShape.llama2_7b, "llama3_8b": LlamaShape.llama3_8b}

# (inputs, outputs) of the linears of both shapes
LINEARS = ((4096, 4096), (4096, 1024), (4096, 11008), (11008, 4096), (4096, 14336), (14336, 4096))


def listed():
    return [
        # the smallest call: one token through an attention projection, as an eager decode loop issues it
        {"name": "linear_1_token", "kind": "linear", "scales": "token", "weight_group": 128, "rows": 1, "k": 4096, "n": 4096},
        # the reference's own modules on a small batch of decoded tokens
        {"name": "linear_16_group", "kind": "linear", "scales": "group", "weight_group": 128, "rows": 16, "k": 4096, "n": 14336},
        # a larger decode batch or a short prompt, ragged: above the sizes of decoding, below those of prefill
        {"name": "linear_45_group", "kind": "linear", "scales": "group", "weight_group": 128, "rows": 45, "k": 11008, "n": 4096},
        # the online-Hadamard linear at the token count of the benchmark
        {"name": "linear_2048_token", "kind": "linear", "scales": "token", "weight_group": 0, "rows": 2048, "k": 4096, "n": 11008},
        # the group quantiser on a long batch (the quantising half of the benchmark, memory-bound)
        {"name": "quantize_16384_group", "kind": "quantize", "scales": "group", "rows": 16384, "k": 4096},
        # one decode step of a chat: one sequence, 2048 cached positions
        {"name": "decode_1x2048_token", "kind": "decode", "shape": "llama3_8b", "scales": "token", "weight_group": 128,
         "batch": 1, "kv_len": 2048},
        # the same for the largest batch of the benchmark
        {"name": "decode_16x2048_token", "kind": "decode", "shape": "llama3_8b", "scales": "token", "weight_group": 128,
         "batch": 16, "kv_len": 2048},
        # a batch in the arrangement of the reference's models, a key / value head per query head, ragged cache length
        {"name": "decode_5x777_group", "kind": "decode", "shape": "llama2_7b", "scales": "group", "weight_group": 128,
         "batch": 5, "kv_len": 777},
        # the benchmark's prefill batch
        {"name": "prefill_8x512_token", "kind": "prefill", "shape": "llama2_7b", "scales": "token", "weight_group": 0,
         "six_bit": False, "batch": 8, "tokens": 512, "past": 0},
        # the next block of a prompt that is fed in pieces, ragged, in the arrangement of the reference's models
        {"name": "prefill_1x1000+531_group", "kind": "prefill", "shape": "llama3_8b", "scales": "group", "weight_group": 128,
         "six_bit": False, "batch": 1, "tokens": 1000, "past": 531},
        # weights held in the 6-bit operand format as well, as a server with memory to spare has them
        {"name": "prefill_1x2048_token_f6", "kind": "prefill", "shape": "llama3_8b", "scales": "token", "weight_group": 128,
         "six_bit": True, "batch": 1, "tokens": 2048, "past": 0},
        # a long document, where attention is a large part of the layer
        {"name": "prefill_1x8192_token", "kind": "prefill", "shape": "llama3_8b", "scales": "token", "weight_group": 128,
         "six_bit": False, "batch": 1, "tokens": 8192, "past": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "decode", "decode", "prefill", "prefill", "quantize"))
    scales = rng.choice(("token", "group"))
    group = 128 if scales == "group" else rng.choice((0, 128))
    if kind == "quantize":
        return {"kind": kind, "scales": scales, "rows": _log_int(rng, 1, 16384), "k": rng.choice((4096, 4096, 11008, 14336))}
    if kind == "linear":
        k, n = rng.choice(LINEARS)
        return {"kind": kind, "scales": scales, "weight_group": group, "rows": _log_int(rng, 1, 2048), "k": k, "n": n}
    shape = rng.choice(tuple(SHAPES))
    if kind == "decode":
        return {"kind": kind, "shape": shape, "scales": scales, "weight_group": group, "batch": _log_int(rng, 1, 16),
                "kv_len": _log_int(rng, 64, 2048)}
    tokens = _log_int(rng, 80, 4096)
    batch = _log_int(rng, 1, max(1, 4096 // tokens))
    past = rng.choice((0, 0, _log_int(rng, 16, 2048)))
    return {"kind": kind, "shape": shape, "scales": scales, "weight_group": group, "six_bit": rng.random() < 0.25,
            "batch": batch, "tokens": tokens, "past": past}


# ---------------------------------------------------------------------------------------------------- inputs
def _activations(shape, gen):
    """fp16 ~ N(0, 1) with 1 % of the channels scaled by 20, as an LLM's hidden states have them."""
    x = torch.randn(shape, device=DEVICE, generator=gen)
    cols = torch.randperm(shape[-1], device=DEVICE, generator=gen)[:max(1, shape[-1] // 100)]
    x[..., cols] *= 20.0
    return x.half()


def _linear(case, gen):
    src = torch.nn.Linear(case["k"], case["n"], bias=False, device=DEVICE, dtype=torch.float16)
    src.weight.data.copy_(torch.randn(case["n"], case["k"], device=DEVICE, generator=gen) / math.sqrt(case["k"]))
    return LinearFLH.from_float(src, weight_group_size=case["weight_group"] or -1, in_group_size=128, no_hadamard=True)


def _layer_weights(s, gen):
    h, i, kv = s.hidden_size, s.intermediate_size, s.num_kv_heads * s.head_dim
    dims = {"q_proj": (h, h), "k_proj": (kv, h), "v_proj": (kv, h), "o_proj": (h, h), "gate_proj": (i, h),
            "up_proj": (i, h), "down_proj": (h, i)}
    w = {name: (torch.randn(n, k, device=DEVICE, generator=gen) / math.sqrt(k)).half() for name, (n, k) in dims.items()}
    for name in ("input_layernorm", "post_attention_layernorm"):
        w[name] = (torch.rand(h, device=DEVICE, generator=gen) + 0.5).half()
    return w


def _fill_cache(cache, slots, gen):
    for t in cache.keys + cache.values:
        t[:, :, :slots].normal_(0.0, 1.0, generator=gen)


def _prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]
    if kind in ("quantize", "linear"):
        state = {"x": _activations((case["rows"], case["k"]), gen)}
        state["quantizer"] = ActQuantizer(bits=4, group_size=128, use_hadamard=True, packed_output=True,
                                          per_token=case["scales"] == "token")
        if kind == "linear":
            state["linear"] = _linear(case, gen)
        return state
    if kind == "decode":
        shape = SHAPES[case["shape"]](DECODE_LAYERS)
        model = W4A4LlamaModel.random_init(shape, activation=case["scales"], weight_group_size=case["weight_group"],
                                           device=DEVICE, seed=seed)
        cache = model.new_cache(case["batch"], case["kv_len"])
        _fill_cache(cache, case["kv_len"] - 1, gen)
        graph, static = model.capture_decode_step(case["batch"], case["kv_len"], cache)
        static["input_ids"].copy_(torch.randint(0, shape.vocab_size, (case["batch"], 1), device=DEVICE, generator=gen))
        return {"model": model, "graph": graph, "static": static}
    shape = SHAPES[case["shape"]](1)
    layer = W4A4DecoderLayer.from_float(_layer_weights(shape, gen), shape.num_heads, shape.num_kv_heads, shape.eps,
                                        weight_group_size=case["weight_group"], activation=case["scales"],
                                        six_bit=case["six_bit"])
    total = case["past"] + case["tokens"]
    cache = StaticKVCache(1, case["batch"], shape.num_kv_heads, total, shape.head_dim, DEVICE, q_heads=shape.num_heads)
    cache.kv_len = case["past"]
    _fill_cache(cache, case["past"], gen)
    positions = cache.advance(case["tokens"])
    cos, sin = rotary_tables(positions, shape.head_dim, shape.rope_theta)
    x = _activations((case["batch"], case["tokens"], shape.hidden_size), gen)
    return {"layer": layer, "x": x, "cos": cos, "sin": sin, "cache": cache, "positions": positions}


def prepare(case, seed):
    with torch.no_grad():
        state = _prepare(case, seed)
    state["case"] = case
    return state


# ---------------------------------------------------------------------------------------------------- the pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        state["graph"].replay()
        out = state["static"]
        return [out["output"], *out["cache"].keys, *out["cache"].values]
    with torch.no_grad():
        if kind == "quantize":
            scales, _, codes = state["quantizer"](state["x"])
            return [codes, scales]
        if kind == "linear":
            if case["scales"] == "token":
                return state["linear"].forward_online(state["x"])
            scales, zeros, codes = state["quantizer"](state["x"])
            return state["linear"](codes, scales, zeros, x_is_packed=True)
        cache = state["cache"]
        y, _ = state["layer"](state["x"], state["cos"], state["sin"], cache.layer(0), state["positions"])
        return [y, cache.keys[0], cache.values[0]]


# ---------------------------------------------------------------------------------------------------- what it cannot do without
def _weight_bytes(n, k, group):
    return n * k / 2 + 2 * n * (k // group if group else 1)


def _layer_linears(s):
    h, i, kv = s.hidden_size, s.intermediate_size, s.num_kv_heads * s.head_dim
    return [(h, h), (kv, h), (kv, h), (h, h), (i, h), (i, h), (h, i)]


def work(case):
    kind = case["kind"]
    if kind == "quantize":
        m, k = case["rows"], case["k"]
        cols = k // 128 if case["scales"] == "group" else 1
        return {"bytes": m * (2 * k + k / 2 + 2 * cols), "flops": m * k * (7 if case["scales"] == "group" else math.log2(k))}
    if kind == "linear":
        m, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": 2 * m * k + _weight_bytes(n, k, case["weight_group"]) + 2 * m * n, "flops": 2 * m * n * k}
    s = SHAPES[case["shape"]](1)
    weights = sum(_weight_bytes(n, k, case["weight_group"]) for n, k in _layer_linears(s))
    products = 2 * sum(n * k for n, k in _layer_linears(s))
    slot = 2 * 2 * s.num_kv_heads * s.head_dim                        # bytes of one position's key and value
    pair = 4 * s.num_heads * s.head_dim                               # operations of one query with one position
    b = case["batch"]
    if kind == "decode":
        length = case["kv_len"]
        layers = DECODE_LAYERS * (weights + b * length * slot)
        head = 2 * s.vocab_size * s.hidden_size + b * 2 * (s.vocab_size + s.hidden_size)
        return {"bytes": layers + head,
                "flops": b * (DECODE_LAYERS * (products + length * pair) + 2 * s.vocab_size * s.hidden_size)}
    t, past = case["tokens"], case["past"]
    if case["six_bit"]:
        weights += sum(n * k / 4 for n, k in _layer_linears(s))        # 6 bits for a code instead of 4
    pairs = t * past + t * (t + 1) / 2
    return {"bytes": weights + b * (4 * t * s.hidden_size + (past + t) * slot),
            "flops": b * (t * products + pairs * pair)}


def tolerance(case):
    """About four times what two correct evaluations at the path's own precision differ by, measured on these cases.

    Codes are rounded: an input that moves by its last bit moves a few codes by a whole step (a relative change e of a row
    moves about 2.5 e of its codes, and the next linear's output by about sqrt(2.5 e) / 2.5), so what follows a second
    quantiser differs by per cents between equally correct evaluations."""
    kind, token = case["kind"], case["scales"] == "token"
    dense = token and case.get("k") in (11008, 14336)        # rows that are rotated by a dense factor as well
    if kind == "quantize":
        if not token:
            return "exact"                                   # every rounding of the fp16 butterflies is specified
        # the float32 butterflies against the matrix cores: < 2e-5 of the codes of a 4096-wide row, 4e-4 of a dense one
        return {"rel": 2e-3, "differ": 2e-3 if dense else 1e-4}
    if kind == "linear":
        # exact codes: the rounding of the result (2.1e-4 against a float64 sum); dense: 0.0095 with the other rotation
        return {"rel": 0.04 if dense else 8.5e-4}
    if kind == "prefill":
        return {"rel": 0.13}                                 # 0.033 against the layer module by module
    return {"rel": 0.4}                                      # 0.099 with attention in float64 (one sequence of 16 diverges)
