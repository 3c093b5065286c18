"""Activation / weight quantisers and the torch Hadamard helpers
(reference: flh/nn/quantization.py).

``ActQuantizer.forward`` runs the HIP kernels; ``forward_origin`` is the torch arithmetic
the reference defines next to it.  Beyond the reference, ``ActQuantizer(per_token=True)``
selects the whole-row online rotation with one scale per token (the QuaRot-style path of
fake_quant/quant_utils.py:94-128 + flh/functional/hadamard.py:92-113), which the reference
offers only in torch.
"""
import math

import numpy as np

import torch

import flh_amd as _pkg

# float32(1 / sqrt(128)): torch's GPU kernel for "half tensor / python scalar" multiplies by this reciprocal
_INV_SQRT_128 = float(np.float32(1.0) / np.float32(math.sqrt(128)))


def _fwht_f64(x64, width):
    """float64 butterflies over every contiguous block of `width`, ascending strides."""
    n = x64.shape[-1]
    lead = x64.shape[:-1]
    stride = 1
    while stride < width:
        v = x64.reshape(*lead, n // (2 * stride), 2, stride)
        a, b = v[..., 0, :], v[..., 1, :]
        x64 = torch.stack((a + b, a - b), dim=-2).reshape(*lead, n)
        stride *= 2
    return x64


def had_transform(X: torch.Tensor, transpose=False):
    """Normalised FWHT of the whole last dimension (a power of two), evaluated in float64;
    returns float64 (flh/nn/quantization.py:42-74)."""
    n = X.shape[-1]
    if (n & (n - 1)) != 0:
        raise ValueError(f"n must be a power of 2 for Hadamard transform, got {n}")
    return _fwht_f64(X.to(torch.float64), n) / math.sqrt(float(n))


def had_transform_group(X: torch.Tensor, transpose=False, group_size: int = 128):
    """Independent normalised FWHT of each contiguous group; falls back to the whole row
    when the group does not divide it (flh/nn/quantization.py:77-113)."""
    n = X.shape[-1]
    if n % group_size != 0:
        return had_transform(X, transpose)
    return _fwht_f64(X.to(torch.float64), group_size) / math.sqrt(float(group_size))


def fast_hadamard_transform(x, group_size=None, normalize=True, use_cuda=True):
    """flh/nn/quantization.py:116-138.  fp16 tensors on the GPU take the 128-group kernel
    (as in the reference, whatever `group_size` says); everything else the float64 torch
    path, cast back to the input dtype."""
    if use_cuda and x.dtype == torch.float16 and x.device.type == "cuda":
        y = _pkg._CUDA.hadamard_transform_half(x.clone().view(-1, 128)) / math.sqrt(128)
        return y.view(x.shape)
    if group_size is not None and group_size > 0:
        out = had_transform_group(x, group_size=group_size)
    else:
        out = had_transform(x)
    return out if x.dtype == torch.float64 else out.to(x.dtype)


def _pack_nibbles(x_int, signed=True):
    """Codes (any dtype holding integers) -> uint8, low nibble = even element."""
    shape = x_int.shape
    q = x_int.flatten().to(torch.int8)
    q = torch.clamp(q, -8, 7) if signed else torch.clamp(q, 0, 15)
    if q.numel() % 2:
        q = torch.cat((q, q.new_zeros(1)))
    pair = q.view(-1, 2)
    packed = ((pair[:, 0] & 0x0F) | ((pair[:, 1] & 0x0F) << 4)).to(torch.uint8)
    if len(shape) <= 1:
        return packed
    return packed.view(*shape[:-1], (shape[-1] + 1) // 2)


class ActQuantizer(torch.nn.Module):
    def __init__(self, bits=8, group_size=-1, sym=True, input_clip_ratio=1.0, use_hadamard=True,
                 packed_output=False, per_token=False):
        super().__init__()
        self.bits = bits
        self.group_size = group_size
        self.sym = sym
        self.input_clip_ratio = input_clip_ratio
        self.use_hadamard = use_hadamard
        self.packed_output = packed_output
        self.per_token = per_token
        if self.packed_output and self.bits != 4:
            raise ValueError("Packed output is only supported for 4-bit quantization")

    def forward(self, x):
        """x [..., K] fp16 on the GPU -> (scale, None, packed codes [..., K/2]).

        Default (as the reference, flh/nn/quantization.py:156-162): every 128 consecutive
        values form a group: unnormalised fp16 FWHT-128 (when use_hadamard) + int4
        quantisation and the division of the scales by sqrt(128) in one kernel; scale shape
        [..., K/128].  per_token=True: normalised rotation of the whole row in float32 and
        one scale per row, shape [..., 1]."""
        if self.per_token:
            mode = -1 if self.use_hadamard is True else 0 if self.use_hadamard is False else None
            r = _pkg._CUDA.quantize_rows(x, mode, self.input_clip_ratio) if mode is not None else None
        else:
            # (the reference's "scales / sqrt(128)" rides on the same launch, see below)
            r = _pkg._CUDA.quantize_groups(x, bool(self.use_hadamard), _INV_SQRT_128 if self.use_hadamard else 1.0)
        if r:
            return r[0], None, r[1]
        lead, k = x.shape[:-1], x.shape[-1]
        if self.per_token:
            q, s = _pkg._CUDA.rotate_and_quantize_i4(x.reshape(-1, k), hadamard=self.use_hadamard,
                                                     clip_ratio=self.input_clip_ratio)
            return s.view(*lead, 1), None, q.view(*lead, k // 2)
        if self.use_hadamard:
            # the reference's "scales / sqrt(128)" (a second kernel there) rides on the same launch
            q, s = _pkg._CUDA.hadamard_and_quantize_i4(x.view(-1, 128), scale_mul=_INV_SQRT_128)
        else:
            q, s = _pkg._CUDA.quant_and_pack_i4(x.view(-1, 128))
        return s.view(*lead, k // 128), None, q.view(*lead, k // 2)

    def forward_origin(self, x):
        """The torch arithmetic of the reference (flh/nn/quantization.py:163-241)."""
        y = fast_hadamard_transform(x, group_size=self.group_size, normalize=True) if self.use_hadamard else x
        if self.bits >= 16:
            return None, None, y
        if self.input_clip_ratio < 1.0:
            bound = y.abs().amax(dim=-1, keepdim=True) * self.input_clip_ratio
            y = torch.clamp(y, -bound, bound)
        g = self.group_size
        grouped = g is not None and g > 0 and y.size(-1) % g == 0
        v = y.view(*y.shape[:-1], y.size(-1) // g, g) if grouped else y
        if self.sym:
            qmax = 2 ** (self.bits - 1) - 1
            scale = torch.clamp(v.abs().amax(dim=-1, keepdim=True) / qmax, min=1e-8)
            zero = torch.zeros_like(scale)
            q = (v / scale).round().clamp(-qmax - 1, qmax)
        else:
            hi, lo = v.amax(dim=-1, keepdim=True), v.amin(dim=-1, keepdim=True)
            qmax = 2 ** self.bits - 1
            scale = (hi - lo) / (qmax + 1e-8)
            scale = torch.where(scale == 0, torch.ones_like(scale), scale)
            zero = -lo / scale
            q = ((v - lo) / scale).round().clamp(0, qmax)
        if grouped:
            scale = scale.view(*y.shape[:-1], -1)
            zero = zero.view(*y.shape[:-1], -1)
        q = q.view(y.shape).to(y.dtype)
        if self.packed_output:
            return scale, zero, _pack_nibbles(q, signed=self.sym)
        return scale, zero, q

    # kept under the reference's name for callers that use it directly
    def _pack_4bit_to_uint8(self, x_int):
        return _pack_nibbles(x_int, signed=self.sym)


class WeightQuantizer(torch.nn.Module):
    """Round-to-nearest weight quantiser (flh/nn/quantization.py:294-484): per tensor, per
    output channel or per group of input channels; symmetric or asymmetric."""

    def __init__(self, bits=4, group_size=-1, sym=True, channel_wise=True, use_hadamard=True, clip_ratio=1.0):
        super().__init__()
        self.bits = bits
        self.group_size = group_size
        self.sym = sym
        self.channel_wise = channel_wise
        self.use_hadamard = use_hadamard
        self.clip_ratio = clip_ratio
        self.register_buffer("scale", None)
        self.register_buffer("zero_point", None)
        self.calibrated = False

    def _prepare(self, weight):
        w = fast_hadamard_transform(weight, group_size=self.group_size, normalize=True) if self.use_hadamard else weight
        return self._clip_weight(w)

    def _view(self, w):
        """weight viewed so that the last axis is one quantisation unit."""
        if self.group_size > 0:
            if w.shape[1] % self.group_size:
                raise ValueError(f"in_features ({w.shape[1]}) must be divisible by group_size ({self.group_size})")
            return w.view(w.shape[0], -1, self.group_size)
        if self.channel_wise:
            return w.view(w.shape[0], 1, -1)
        return w.reshape(1, 1, -1)

    def _clip_weight(self, w):
        if self.clip_ratio >= 1.0:
            return w
        v = self._view(w) if (self.group_size <= 0 or w.shape[1] % self.group_size == 0) else w.view(w.shape[0], 1, -1)
        bound = v.abs().amax(dim=-1, keepdim=True) * self.clip_ratio
        return torch.clamp(v, -bound, bound).view(w.shape)

    def calibrate(self, weight):
        if self.bits >= 16:
            self.calibrated = True
            return
        with torch.no_grad():
            v = self._view(self._prepare(weight))
            if self.sym:
                qmax = 2 ** (self.bits - 1) - 1
                scale = torch.clamp(v.abs().amax(dim=-1) / qmax, min=1e-8)
                zero = torch.zeros_like(scale)
            else:
                hi, lo = v.amax(dim=-1), v.amin(dim=-1)
                scale = torch.clamp((hi - lo) / (2 ** self.bits - 1), min=1e-8)
                zero = -lo / scale
            if self.group_size <= 0 and not self.channel_wise:
                scale, zero = scale.view(1), zero.view(1)
            self.scale, self.zero_point = scale, zero
        self.calibrated = True

    def quantize(self, weight):
        w = self._prepare(weight)
        if self.bits >= 16:
            return None, None, w
        if not self.calibrated:
            raise RuntimeError("WeightQuantizer must be calibrated before quantization")
        qmin, qmax = (-2 ** (self.bits - 1), 2 ** (self.bits - 1) - 1) if self.sym else (0, 2 ** self.bits - 1)
        v = self._view(w)
        s = self.scale.reshape(v.shape[0], v.shape[1], 1)
        q = v / s
        if not self.sym:
            q = q + self.zero_point.reshape(v.shape[0], v.shape[1], 1)
        return self.scale, self.zero_point, q.round().clamp(qmin, qmax).view(w.shape).to(w.dtype)

    def forward(self, weight):
        if not self.calibrated:
            self.calibrate(weight)
        return self.quantize(weight)


Quantizer = ActQuantizer
