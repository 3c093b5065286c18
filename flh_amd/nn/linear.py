"""W4A4 linear layer (reference: flh/nn/linear.py).

Buffers keep the reference's names and layouts: ``w_packed`` uint8 flat [N*K/2] (low nibble
= even input channel), ``w_scale`` [N, K/group] (or [N, 1] when group_size <= 0),
``w_zero`` uint8 (always 0: symmetric), optional ``bias``.  ``forward`` is one call of the
int4 GEMM + dequant kernel.  Unlike the reference's forward (flh/nn/linear.py:125-133, which
never adds it) the bias is added when the layer has one.
"""
import torch

import flh_amd as _pkg
from . import quantization as _quant
from ..functional.quantization import unpack_i4


class LinearFLH(torch.nn.Module):
    def __init__(self, in_features, out_features, bias=False, dtype=torch.float16, device="cpu",
                 dual_hadamard=False, in_group_size=None, out_group_size=None, no_hadamard=False, group_size=128):
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        self.dual_hadamard = dual_hadamard
        self.in_group_size = in_group_size
        self.out_group_size = out_group_size
        self.weight_group_size = group_size
        self.no_hadamard = no_hadamard
        n_groups = -(-in_features // group_size) if group_size > 0 else 1
        self.register_buffer("w_packed", torch.zeros((out_features * in_features + 1) // 2, dtype=torch.uint8, device=device))
        self.register_buffer("w_scale", torch.zeros(out_features, n_groups, dtype=dtype, device=device))
        self.register_buffer("w_zero", torch.zeros(out_features, n_groups, dtype=torch.uint8, device=device))
        if bias:
            self.register_buffer("bias", torch.zeros(out_features, dtype=dtype, device=device))
        else:
            self.bias = None
        # Prefill-sized calls run on the 6-bit matrix instruction where that is faster (extension; same bits, no unpack in the
        # loop).  Its operands are re-encoded at 6 bits per code, 0.75 byte per weight next to the 0.5 of `w_packed`.
        # False (default): nothing is kept; a long call (_six_bit_rows) encodes its weights into a buffer that goes back with
        # it.  "never": not even that, for callers without that memory to spare.  True: the layer keeps the encoding (2.5 x
        # the weight memory) and every call of at least `six_bit_min_rows` rows uses it.  "auto" (or None): kept for weights
        # with a scale per group of 128.
        # `prepare_six_bit()` builds the kept encoding at once (a loader calls it); otherwise it is built on first use.  It is
        # rebuilt whenever `w_packed` has been written to or replaced (in-place copies, load_state_dict, .to(device)): keyed
        # on the buffer's storage address and version counter.
        self.six_bit = False
        self.six_bit_min_rows = 256
        self._w6 = None
        self._w6_key = None

    def drop_six_bit_weights(self):
        self._w6 = self._w6_key = None

    # A call that encodes its weights for the 6-bit instruction first is faster from these rows on (one scale per channel;
    # group-scaled weights with a scale per token; group scales on both sides) if it also has more 128 x 128 tiles than
    # _transient_tiles -- less fills the chip with neither kernel, and the passes over the operands are all that differs.
    # Packed codes, which the call encodes as well, need more.  us, int8 / 6-bit with the weights encoded (codes from the
    # quantiser in the 6-bit format, which costs it 1-3 us more) / packed codes encoded as well, rows x channels, K = 4096 unless stated:
    #   one scale per channel: 2048 x 4096 34.5 / 34.9 / 40.7, 3000 x 4096 49 / 43 / 52, 2400 x 11008 109 / 82 / 90; 2048 x 11008
    #   89 / 79 / 87 in
    #   a graph, 84 / 84 as separate calls, and a layer of 1400 tokens whose gate and up change over is slower, 380 / 409
    #   a scale per token: 640 x 4096 25.7 / 28.5 / 28.4, 1280 x 4096 45 / 35 / 42, 1000 x 14336 95 / 70 / 79, 640 x 4096 of K =
    #   11008 63 / 54 / 58
    #   group scales: 640 x 4096 27 / 30 / 30, 1000 x 4096 28 / 33 / 33, 640 x 11008 52 / 51 / 55, 800 x 11008 74 / 68 / 70, 1000 x
    #   14336 98 / 76 / 84,
    #   512 x 4096 of K = 11008 60 / 54 / 57;
    #   320 x 11008 52 / 43 / 46, but the host's part of the encoding makes a layer of 300 or 450 tokens slower (245 / 262; 500: 271 / 263)
    TRANSIENT_ROWS = (2560, 641)
    TRANSIENT_ROWS_GROUPS = 513
    # The same lines where a decoder layer's quantiser writes the codes in the 6-bit format and encodes the weights in its own launch:
    # (rows from which, 128 x 128 tiles that a K up to 8192 needs more of, a longer one).  Effect of the change on a layer of 200 to
    # 570 us (8B / 7B shapes; qkv 6144 / 12288 channels, gate + up 28672 / 22016, o and down 4096), us by rows:
    #   group scales: qkv 257 .. 384 -1 .. +2 (144 tiles) / -10 (288), 700 -16 / -7; gate + up 257 .. 384 -2 .. +1 / -6, 385 .. 512 -16 ..
    #     -20 / -6; down 257 .. 512 -9 .. -11 / -4 .. -5 (96 and 128 tiles); o 257 .. 384 +2 .. +5, 800 -4 / +3, 900 .. 1024 (256) -3 .. -5
    #   a scale per token: qkv 257 .. 384 -1 / -8, 513 -4 / -7; gate + up 257 .. 384 -1 .. -4 / -6, 385 .. 640 -9 .. -15 / -5 .. -14;
    #     down (a rotation that shares no launch) 257 .. 512 0 .. +4, 513 .. 640 (160) -6 .. -10
    #   one scale per channel: gate + up 1024 +4 / +4, 1200 +8, 2048 -21 / -33; down 2048 (512) 0, 2100 .. 2400 -14 .. -24; qkv 1400 .. 2400
    #     0 / -3; o 2100 .. 2400 -4 .. -7.  1400 .. 1792 gate + up go by the clock: 0 .. -18 / -2 .. -16 where calls have followed each other
    #     long enough for the power limit, which the int8 instruction meets first, +12 .. +23 / +15 .. +23 in short runs, +8 at 1513 / 7B
    #     with the inputs of successive calls different.  The line is 22016 channels': their eighth 256 rows, from 1793 on, cost int8 another
    #     round of tiles (the launch with its quantiser, 1792 / 1793 rows: int8 141 / 162, 6-bit 134 / 138); 28672 have it at 2049 (int8 190 /
    #     197, at 2049 224; 6-bit 173 / 177, 187), q / k / v beyond 2048 rows (6144 59 / 59 up to there, 70 / 65 beyond; 12288 98 / 100, 121 /
    #     113).  What it does to the whole layer of 1793 .. 2048 tokens, long runs / short ones / one input again and again: 22016 -3 .. -8 /
    #     -17 .. -20 / 0 .. -3 of 440, 28672 +5 .. -2 / -2 .. -10 / +9 .. +13 of 460; of 2100, 28672 -46 / -50 / -42 of 570
    # 256 rows and fewer have smaller int8 tiles: a layer of 256 tokens 164 us, of 257 214.  Up to 384 rows the encoding of more than
    # 24576 channels takes what the faster instruction gives (hidden 8192, gate + up 57344, 257 rows: 547 -> 559 with them).  Hidden sizes
    # below 4096 keep the lines above: their layers wait for the host, which has more to do here (hidden 2048, 400 tokens 154 / 164).  So
    # does whole-row rotation at K = 8192, whose layers were not timed, and a linear that quantises for itself (forward_online), which asks
    # without columns: its lines are those of an encoding in a launch of its own.
    # The whole layer, us: 257 tokens 220 -> 200 and 214 -> 204 (7B, 8B), 400 231 -> 215 and 247 -> 218; a scale per token 640 tokens
    # 274 -> 250 and 293 -> 280; one scale per channel 2100 tokens 555 -> 516 and 574 -> 520; hidden 5120, 400 tokens 329 -> 294.
    BESIDE_QUANTISER = ((1793, 512, 512), (257, 255, 128), (257, 255, 95))
    _LEAST_ROWS = BESIDE_QUANTISER[-1][0]          # the first of all these lines
    _NO_ROWS = 1 << 62                             # more rows than any call has

    def _transient_tiles(self, grouped, nibbles, groups=False):
        long_k = self.in_features > 8192
        if grouped and groups:
            return (128 if nibbles else 95) if long_k else 256
        if grouped:
            return 191 if long_k else 256
        return 1280 if nibbles and not long_k else 512

    def _keeps_six_bit(self, grouped):
        return self.six_bit is True or (self.six_bit not in (False, "never") and grouped)

    def _six_bit_rows(self, grouped, columns=None, nibbles=False, groups=False):
        """Rows from which a launch over `columns` channels (this layer's, unless it shares the launch) takes the 6-bit
        instruction.  nibbles: its activations come as packed codes, to be encoded as well; groups: with a scale per group of 128.
        Given `columns` and no nibbles, the quantiser encodes the weights (as wants_six_bit says)."""
        if self.six_bit is not False:
            if self.six_bit == "never":
                return self._NO_ROWS
            if self._keeps_six_bit(grouped):
                return self.six_bit_min_rows
        groups = grouped and groups
        tiles = -(-(columns or self.out_features) // 128)
        if columns and not nibbles and (self.in_features >= 4096 if groups else self.in_features in (4096, 11008, 14336)):
            first, *needs = self.BESIDE_QUANTISER[2 if groups else grouped]
            return max(first, 385 if tiles > 192 else 0, 128 * (needs[self.in_features > 8192] // tiles) + 1)
        first = self.TRANSIENT_ROWS_GROUPS if groups else self.TRANSIENT_ROWS[grouped]
        return max(first, 128 * (self._transient_tiles(grouped, nibbles, groups) // tiles) + 1)

    def prepare_six_bit(self):
        """Build the 6-bit encoding of the weights now if this layer's setting keeps one (at load time, rather than inside
        the first long call)."""
        if self.wants_six_bit(self.six_bit_min_rows) and self._keeps_six_bit(self.w_scale.view(self.out_features, -1).size(1) > 1):
            self._six_bit_weights()

    def _six_bit_weights(self):
        if not self._keeps_six_bit(self.w_scale.numel() > self.out_features):
            return _pkg._CUDA.encode_f6_many([self.w_packed.view(self.out_features, self.in_features // 2)])[0]
        key = (self.w_packed.data_ptr(), self.w_packed._version, self.w_packed.device)
        if self._w6 is None or self._w6_key != key:
            self._w6 = _pkg._CUDA.encode_f6(self.w_packed.view(self.out_features, self.in_features // 2))
            self._w6_key = key
        return self._w6

    @staticmethod
    def _weights_to_encode(layers):
        """The packed weights of layers that share their activations and keep no 6-bit encoding, for one launch to encode; None
        where one of them keeps its own."""
        if len(layers) <= 4 and all(type(l) is LinearFLH and l.in_features == layers[0].in_features
                                    and not l._keeps_six_bit(l.w_scale.numel() > l.out_features) for l in layers):
            return [l.w_packed.view(l.out_features, l.in_features // 2) for l in layers]
        return None

    @staticmethod
    def _beside_quantiser(layers):
        """Arguments of the quantiser in front of `layers` that has it encode their weights as well, if they are to be encoded."""
        packed = LinearFLH._weights_to_encode(layers)
        return {} if packed is None or not packed[0].is_cuda else {"weights": packed}

    @staticmethod
    def _six_bit_weights_of(layers):
        """[l._six_bit_weights() for l in layers], encodings that are not kept built in one launch."""
        packed = LinearFLH._weights_to_encode(layers) if len(layers) > 1 else None
        return [l._six_bit_weights() for l in layers] if packed is None else _pkg._CUDA.encode_f6_many(packed)

    @staticmethod
    def _six_bit_operands(layers, rows, encoded, w6):
        """(codes, [weights]) of `layers` in the 6-bit format, from codes that are `encoded` already or packed ones; w6: the weights'
        encodings, if there are any.  Packed codes and weights that have to be encoded share a launch (us a call, two launches
        -> one: 600 x 4096 codes, 11008 channels 52.8 -> 51.0, 513 x 11008, 4096 channels 58.4 -> 55.4, 4096 x 4096, 11008 channels with one
        scale each 122.3 -> 118.7)."""
        rows = rows.contiguous()
        if not encoded and w6 is None and len(layers) < 4:
            packed = LinearFLH._weights_to_encode(layers)
            if packed is not None:
                rows, *w6 = _pkg._CUDA.encode_f6_many([rows, *packed])
                return rows, w6
        return rows if encoded else _pkg._CUDA.encode_f6(rows), w6 or LinearFLH._six_bit_weights_of(layers)

    _SIX_BIT_MAX_ROWS = ((1 << 32) - 1) // 96       # rows of either operand that the 6-bit launches index; more go to int8

    def wants_six_bit(self, n_rows, columns=None, groups=False):
        """Whether a call with `n_rows` rows quantised per token (or, `groups`, per group of 128) takes the 6-bit matrix
        instruction (a producer can then write the activations in that format directly, rotate_and_quantize_f6).
        `columns`: channels of the whole launch, from a caller whose quantiser is given the weights to encode (_beside_quantiser); the
        lines of BESIDE_QUANTISER are a decoder layer's."""
        if self._below_six_bit(n_rows) or self.in_features % 128 or not self.w_packed.is_cuda:
            return False
        cols = self.w_scale.numel() // self.out_features
        if cols != 1 and not (cols == self.in_features // 128 and self.weight_group_size == 128):
            return False
        return self._six_bit_rows(cols != 1, columns, False, groups) <= n_rows <= self._SIX_BIT_MAX_ROWS

    def _below_six_bit(self, n_rows):
        """Whether `n_rows` rows are fewer than this layer takes to the 6-bit instruction in any launch."""
        return (n_rows < (self._LEAST_ROWS if self.in_features >= 4096 else self.TRANSIENT_ROWS_GROUPS)
                and (self.six_bit is False or n_rows < self.six_bit_min_rows))

    def _six_bit_applies(self, rows, a_scale, w_scale, group, columns=None):
        n = rows.size(0)
        if self._below_six_bit(n) or not rows.is_cuda or self.in_features % 128:
            return False
        per_row = a_scale.size(1) == 1 and w_scale.size(1) == 1
        grouped = group == 128 and w_scale.size(1) == self.in_features // 128 and a_scale.size(1) in (1, w_scale.size(1))
        return ((grouped or per_row)
                and self._six_bit_rows(not per_row, columns, True, a_scale.size(1) > 1) <= n <= self._SIX_BIT_MAX_ROWS)

    def _group(self):
        return self.weight_group_size if self.weight_group_size > 0 else (self.in_group_size or 128)

    def _few_rows(self, w_scale, nibbles=False, groups=False):
        """Rows below which no call of this layer (on packed codes, if `nibbles`) takes the 6-bit instruction."""
        return self._six_bit_rows(w_scale.numel() > self.out_features, None, nibbles, groups)

    # ------------------------------------------------------------------ kernels
    def forward(self, x, a_scale=None, a_zero=None, x_is_packed=False, is_symmetric=None, residual=None, w6=None):
        """x: packed int4 activations [..., K/2] uint8; a_scale [..., K/in_group] or [..., 1]
        fp16 (as returned by ActQuantizer).  Returns fp16 [..., N].  `residual` (extension; fp16 [..., N]): returns
        residual + forward(x, ...) from the same launch -- the layer output rounded to fp16 as always, then one fp16
        addition in the GEMM's epilogue instead of a separate pass over both tensors.  `w6` (extension, here and in
        forward_many and forward_swiglu): with activations in the 6-bit format, the encodings of the weights, a list in the order of
        the layers, where the quantiser's launch has made them (`weights` of rotate_and_quantize_f6 and its like)."""
        if residual is None and a_scale is not None and w6 is None:
            w, w_scale = self._buffers.get("w_packed"), self._buffers.get("w_scale")
            if w is not None and w_scale is not None:
                k, least = self.in_features, self.TRANSIENT_ROWS_GROUPS
                few = (least if self.six_bit is False and 2 * x.numel() < least * k      # below every line: asked for no further
                       else self._few_rows(w_scale, True, a_scale.size(-1) > 1))
                y = _pkg._CUDA.linear_i4(x, a_scale, w, w_scale, k, self.out_features, self._group(), few)
                if y is not None:
                    return y if self.bias is None else y + self.bias
        lead = x.shape[:-1]
        if residual is not None and self.bias is not None:
            return residual + self.forward(x, a_scale, a_zero, x_is_packed, is_symmetric, w6=w6)
        res = None if residual is None else residual.reshape(-1, self.out_features)
        rows = x.view(-1, x.size(-1))
        w_scale = self.w_scale.view(self.out_features, -1)
        group = self.weight_group_size if self.weight_group_size > 0 else (self.in_group_size or 128)
        a_rows = a_scale.reshape(rows.size(0), -1)
        encoded = rows.size(1) * 4 == self.in_features * 3      # activations already in the 6-bit format
        if encoded or self._six_bit_applies(rows, a_rows, w_scale, group):
            ops = _pkg._CUDA
            a6, (w6,) = self._six_bit_operands((self,), rows, encoded, w6)
            if encoded and not ((w_scale.size(1) == 1 and a_rows.size(1) == 1) or
                                (group == 128 and w_scale.size(1) == self.in_features // 128)):
                raise ValueError("6-bit activations need per-token x per-channel scales or group-of-128 weight scales")
            if res is not None:
                y = ops.gemm_f6_dequant_add(a6, w6, a_rows.contiguous(), w_scale, res.contiguous())
            elif w_scale.size(1) == 1:
                y = ops.gemm_f6_dequant_o16(a6, w6, a_rows.contiguous(), w_scale)
            else:
                y = ops.gemm_f6_dequant_o16_gs(a6, w6, a_rows.contiguous(), w_scale)
            if self.bias is not None:
                y = y + self.bias
            return y.view(*lead, self.out_features)
        if res is not None:
            y = _pkg._CUDA.gemm_i4_dequant_add(rows, self.w_packed.view(self.out_features, self.in_features // 2),
                                               a_rows, w_scale, res.contiguous(), group)
            return y.view(*lead, self.out_features)
        y = _pkg._CUDA.gemm_i4_dequant(rows, self.w_packed.view(self.out_features, self.in_features // 2),
                                       a_scale.reshape(rows.size(0), -1), w_scale, group)
        if self.bias is not None:
            y = y + self.bias
        return y.view(*lead, self.out_features)

    @staticmethod
    def forward_many(layers, x, a_scale, w6=None):
        """[layer(x, a_scale, x_is_packed=True) for layer in layers] in one GEMM launch: for projections that share
        their quantised input (q / k / v, gate / up; at most four), each with its own weights where they are.
        Same bits as the separate calls."""
        first = layers[0]
        lead = x.shape[:-1]
        rows = x.view(-1, x.size(-1))
        group = first.weight_group_size if first.weight_group_size > 0 else (first.in_group_size or 128)
        for layer in layers:
            if layer.in_features != first.in_features or layer.w_scale.shape[1:] != first.w_scale.shape[1:]:
                raise ValueError("forward_many: the layers must share in_features and the weight-scale layout")
        ops = _pkg._CUDA
        a_rows = a_scale.reshape(rows.size(0), -1)
        w_scales = [l.w_scale.view(l.out_features, -1) for l in layers]
        encoded = rows.size(1) * 4 == first.in_features * 3      # activations already in the 6-bit format
        columns = sum(l.out_features for l in layers)
        if encoded or all(l._six_bit_applies(rows, a_rows, ws, group, columns) for l, ws in zip(layers, w_scales)):
            # every layer takes the 6-bit matrix instruction here: one launch there as well
            ys = ops.gemm_f6_dequant_multi(*LinearFLH._six_bit_operands(layers, rows, encoded, w6), a_rows.contiguous(), w_scales)
        else:
            ys = ops.gemm_i4_dequant_multi(rows, [l.w_packed.view(l.out_features, l.in_features // 2) for l in layers],
                                           a_rows, w_scales, group)
        return [(y if l.bias is None else y + l.bias).view(*lead, l.out_features) for y, l in zip(ys, layers)]

    @staticmethod
    def forward_swiglu(gate_layer, up_layer, x, a_scale, w6=None):
        """act_fn(gate_layer(x)) * up_layer(x) of a SwiGLU MLP (flh/quantized_model/modeling_llama.py:522-526) in one
        GEMM launch that stores only the product: x packed codes [..., K/2], a_scale as for forward.  The two
        projections are rounded to fp16 as their own calls would store them, then combined as torch's fp16 silu and
        multiply do (the device's exponential: the fp16 result can differ from torch's in its last bit in a few values
        per thousand)."""
        if (gate_layer.in_features != up_layer.in_features or gate_layer.out_features != up_layer.out_features
                or gate_layer.w_scale.shape != up_layer.w_scale.shape):
            raise ValueError("forward_swiglu: gate and up must have the same shape and weight-scale layout")
        if gate_layer.bias is not None or up_layer.bias is not None:
            raise ValueError("forward_swiglu: layers with a bias take the separate calls")
        lead = x.shape[:-1]
        rows = x.view(-1, x.size(-1))
        n, k = gate_layer.out_features, gate_layer.in_features
        group = gate_layer.weight_group_size if gate_layer.weight_group_size > 0 else (gate_layer.in_group_size or 128)
        a_rows = a_scale.reshape(rows.size(0), -1)
        encoded = rows.size(1) * 4 == k * 3                     # activations already in the 6-bit format
        both = (gate_layer, up_layer)
        if encoded or not any(l._below_six_bit(rows.size(0)) for l in both) and all(
                l._six_bit_applies(rows, a_rows, l.w_scale.view(n, -1), group, 2 * n) for l in both):
            ops = _pkg._CUDA
            a6, weights = LinearFLH._six_bit_operands(both, rows, encoded, w6)
            y = ops.gemm_f6_swiglu(a6, *weights, a_rows.contiguous(),
                                   gate_layer.w_scale.view(n, -1), up_layer.w_scale.view(n, -1))
            return y.view(*lead, n)
        y = _pkg._CUDA.gemm_i4_swiglu(rows, gate_layer.w_packed.view(n, k // 2), up_layer.w_packed.view(n, k // 2),
                                      a_rows, gate_layer.w_scale.view(n, -1),
                                      up_layer.w_scale.view(n, -1), group)
        return y.view(*lead, n)

    _ONLINE_MODES = {"exact": 1, "fast": 2}        # FLH_HAD_F32, FLH_HAD_MFMA

    def forward_online(self, x, hadamard=True):
        """fp16 activations [..., K] -> fp16 [..., N] with the activation side done here: whole-row rotation
        (`hadamard`: as in rotate_and_quantize_i4), one symmetric int4 scale per token, then the GEMM -- the
        online-Hadamard linear of the reference's benchmarks (benchmark/nn/benchmark_linear_flh.py:139-222), which
        has no module of its own there.  One token of K = 4096 (up to 32768 channels; two up to 16384) with
        the bit-exact rotation takes the single-launch decode path; the outputs are the same bits either way."""
        ops = _pkg._CUDA
        buf, mode = self._buffers, -1 if hadamard is True else self._ONLINE_MODES.get(hadamard)
        if mode is not None and buf.get("w_packed") is not None and buf.get("w_scale") is not None:
            k, least = self.in_features, self.TRANSIENT_ROWS_GROUPS
            few = least if self.six_bit is False and x.numel() < least * k else self._few_rows(buf["w_scale"])
            y = ops.linear_online_i4(x, buf["w_packed"], buf["w_scale"], k, self.out_features, self._group(), mode, few)
            if y is not None:
                return y if self.bias is None else y + self.bias
        lead = x.shape[:-1]
        rows = x.reshape(-1, x.size(-1)).contiguous()
        w = self.w_packed.view(self.out_features, self.in_features // 2)
        w_scale = self.w_scale.view(self.out_features, -1)
        group = self.weight_group_size if self.weight_group_size > 0 else (self.in_group_size or 128)
        fusable = ((rows.size(0) == 1 and self.out_features <= 32768 or rows.size(0) == 2 and self.out_features <= 16384)
                   and self.in_features == 4096 and hadamard in (True, "exact")
                   and (w_scale.size(1) == 1 or (group == 128 and w_scale.size(1) == 32)))
        if fusable:
            y = ops.rotate_quantize_gemm_i4(rows, w, w_scale)
        elif (rows.size(0) >= self.TRANSIENT_ROWS_GROUPS and self.in_features in (4096, 11008, 14336)
              and self.wants_six_bit(rows.size(0))) and (
                hadamard in (True, "fast") or (hadamard == "exact" and self.in_features == 4096)):
            # long calls: the quantiser writes the 6-bit operand format
            q, s, *w6 = ops.rotate_and_quantize_f6(rows, hadamard=hadamard, **self._beside_quantiser((self,)))
            return self.forward(q, s, x_is_packed=True, **({"w6": w6} if w6 else {})).view(*lead, self.out_features)
        else:
            q, s = ops.rotate_and_quantize_i4(rows, hadamard=hadamard)
            y = ops.gemm_i4_dequant(q, w, s, w_scale, group)
        if self.bias is not None:
            y = y + self.bias
        return y.view(*lead, self.out_features)

    # ------------------------------------------------------------------ torch arithmetic
    def _unpack_weights(self):
        """Dequantised weight [N, K] in the scale's dtype (flh/nn/linear.py:37-86)."""
        n, k = self.out_features, self.in_features
        w_int = unpack_i4(self.w_packed[: n * k // 2].view(n, k // 2)).float()
        g = self.weight_group_size
        if g > 0:
            wg = w_int.view(n, k // g, g) - self.w_zero.float().unsqueeze(-1)
            return (wg * self.w_scale.unsqueeze(-1)).view(n, k).to(self.w_scale.dtype)
        return ((w_int - self.w_zero.float()) * self.w_scale).to(self.w_scale.dtype)

    def _unpack_activation_4bit(self, x_packed, a_scale, a_zero, is_symmetric=None):
        """Packed codes -> dequantised float activations (flh/nn/linear.py:287-364)."""
        if is_symmetric is None:
            is_symmetric = not (a_zero is not None and torch.any(a_zero != 0))
        if is_symmetric:
            x_int = unpack_i4(x_packed).float()
        else:
            x_int = torch.stack((x_packed & 0x0F, x_packed >> 4), dim=-1).reshape(*x_packed.shape[:-1], -1).float()
        if a_scale is None:
            return x_int
        zp = a_zero if a_zero is not None else 0
        if self.in_group_size and self.in_group_size > 0 and a_scale.shape[-1] != 1:
            g = self.in_group_size
            v = x_int.view(*x_int.shape[:-1], -1, g)
            if torch.is_tensor(zp):
                zp = zp.view(*v.shape[:-1], 1)
            return ((v - zp) * a_scale.view(*v.shape[:-1], 1)).view_as(x_int)
        return (x_int - zp) * a_scale

    def forward_torch(self, x, a_scale=None, a_zero=None, x_is_packed=False, is_symmetric=None):
        if x_is_packed:
            x = self._unpack_activation_4bit(x, a_scale, a_zero, is_symmetric)
        elif a_scale is not None:
            zp = a_zero if a_zero is not None else 0
            x = (x - zp) * a_scale
        weight = self._unpack_weights()
        return torch.nn.functional.linear(x.to(weight.dtype), weight, self.bias)

    def get_weight(self, dtype=None):
        w = self._unpack_weights()
        return w if dtype is None else w.to(dtype)

    # ------------------------------------------------------------------ weight preparation
    def _pack_weights(self, w_int, scale, zero):
        """Store codes [N, K] (values in [-8, 7]) and their scales (flh/nn/linear.py:88-123)."""
        self.w_scale.copy_(scale.reshape(self.w_scale.shape))
        self.w_zero.copy_(zero.reshape(self.w_zero.shape).clamp(0, 15).to(torch.uint8))
        q = torch.clamp(w_int.flatten(), -8, 7).to(torch.int16) & 0xF
        if q.numel() % 2:
            q = torch.cat((q, q.new_zeros(1)))
        q = q.view(-1, 2)
        self.w_packed.copy_((q[:, 0] | (q[:, 1] << 4)).to(torch.uint8))

    def _quantize_and_store(self, W, bits, group_size, sym, clip_ratio):
        # fp16 weights that already sit on the GPU take the HIP quantise-and-pack kernel (same scales and
        # codes as the tensor arithmetic below: scale = fp16(max|w| / 7) per group or per row, codes =
        # clamp(rint(w / scale)); an all-zero group gets scale 1 where that arithmetic yields NaN)
        k = W.shape[-1]
        g = group_size if group_size and group_size > 0 else 0
        if (W.is_cuda and W.dtype == torch.float16 and W.dim() == 2 and bits == 4 and sym and clip_ratio >= 1.0
                and k % 16 == 0 and (g == 0 or (k % g == 0 and g % 2 == 0)) and self.w_scale.numel() == W.shape[0] * (k // g if g else 1)):
            q, s = _pkg._CUDA.rotate_and_quantize_i4(W.contiguous(), hadamard=False, scale_group=g)
            self.w_packed.copy_(q.reshape(self.w_packed.shape))
            self.w_scale.copy_(s.reshape(self.w_scale.shape))
            self.w_zero.zero_()
            return
        wq = _quant.WeightQuantizer(bits=bits, group_size=group_size, sym=sym, channel_wise=(group_size == -1),
                                    use_hadamard=False, clip_ratio=clip_ratio)
        wq.calibrate(W)
        if bits < 16 and torch.isnan(wq.scale).any():
            print(f"WARNING: NaN detected in quantization scale for layer {self.out_features}x{self.in_features}")
            return
        scale, zp, w_int = wq.quantize(W)
        if scale.dim() == 1:  # per tensor
            scale = scale.expand(self.out_features, 1)
            zp = zp.expand(self.out_features, 1)
        self._pack_weights(w_int, scale, zp)

    def set_weight(self, weight):
        """Quantise a float weight [N, K] (RTN, symmetric 4 bit, this layer's group size)."""
        self._quantize_and_store(weight, 4, self.weight_group_size, True, 1.0)

    @staticmethod
    def from_float(module, weight_bits=4, weight_group_size=128, weight_sym=True, dual_hadamard=False,
                   in_group_size=None, out_group_size=None, clip_ratio=1.0, no_hadamard=False):
        """Build from an nn.Linear (flh/nn/linear.py:190-285): optionally rotate the weight by
        the (grouped) normalised Hadamard matrix on the input side -- and on the output side,
        with the bias, when dual_hadamard -- then quantise and pack."""
        layer = LinearFLH(module.in_features, module.out_features, bias=module.bias is not None,
                          dtype=module.weight.dtype, device=module.weight.device, dual_hadamard=dual_hadamard,
                          in_group_size=in_group_size, out_group_size=out_group_size, group_size=weight_group_size)
        W = module.weight.data.clone()
        if layer.bias is not None:
            layer.bias.copy_(module.bias.data)
        if not no_hadamard:
            rot = _quant.fast_hadamard_transform
            if dual_hadamard:
                W = rot(W, group_size=in_group_size, use_cuda=False)
                W = rot(W.T, group_size=out_group_size, use_cuda=False).T
                if layer.bias is not None:
                    layer.bias.copy_(rot(layer.bias.unsqueeze(0), group_size=out_group_size).squeeze(0))
            else:
                W = rot(W, group_size=in_group_size)
        if torch.isnan(W).any():
            print(f"WARNING: NaN detected in weights after Hadamard for layer {module.out_features}x{module.in_features}")
            return layer
        layer._quantize_and_store(W.contiguous(), weight_bits, weight_group_size, weight_sym, clip_ratio)
        return layer
