"""bf16 convolutions on fp16 MIOpen kernels (tbf16/conv.py of the reference).

The weight gets one exact power-of-two scale per output channel and the input one
per sample (a convolution mixes positions, so rows cannot be scaled separately);
the convolution runs in fp16 with fp32 accumulation and the scales are undone in
one pass that writes bf16. The weight conversion is lossless; the input's is
lossless for every element within 2^14 of its sample's max (smaller ones become
fp16 subnormals, far below the output's bf16 rounding).

On MI355X a 2-D convolution of some size runs whole on this library's kernels
(tbf16_conv2d: per-sample maxima, one scaled channels-last copy of the input, an
implicit GEMM that writes bf16 from its fp32 sums). For the others the passes around the
convolution are HIP kernels (tbf16_conv_input: per-sample max, exponent and scaled fp16
copy; tbf16_conv_epilogue: both scales and the bias in one bf16-writing pass) and the
fp16 convolution is MIOpen's, through torch. 1x1 convolutions (stride 1, no padding,
one group) are per-pixel linear layers and go through scaled_linear, which scales
each pixel separately. Inference only: inputs that need gradients, or are not
bf16, run the native convolution on the dequantized weight (conv.py:34-38).
Converted modules get the class TBF16<their class>, the buffers weight16 and
weight_scale and the method dequantized_weight(), as in the reference.
"""
import ctypes
import functools
from typing import NamedTuple

import torch
import torch.nn as nn
import torch.nn.functional as F

from ._ext import launch, lib, ptr
from .ops import _dev_check, _target_exp, prepare_weight, scaled_linear

_CONV = {1: F.conv1d, 2: F.conv2d, 3: F.conv3d}
_CHANNELS_LAST = {2: torch.channels_last, 3: torch.channels_last_3d}


def _sample_major(x: torch.Tensor, nd: int) -> torch.Tensor:
    """x itself when each sample is one dense run of memory (contiguous, or
    channels-last for 2-D/3-D) starting 16-byte aligned, else a copy that is."""
    dense = x.is_contiguous() or (nd in _CHANNELS_LAST and x.is_contiguous(memory_format=_CHANNELS_LAST[nd]))
    if not dense:
        x = x.contiguous()
    return x if x.data_ptr() % 16 == 0 else x.clone()


def scale_input(x: torch.Tensor, t: int):
    """bf16 (B, C, *spatial) -> (int32 (B,) exponents e, fp16 x * 2^-e in x's layout).
    e = frexp(max |x[b]|) - t, so the scaled max lies in [2^(t-1), 2^t) (conv.py:49-54).
    Empty samples take amax = 1 as the reference's where(amax > 0, amax, 1) does."""
    _dev_check(x)
    if x.dtype != torch.bfloat16:
        raise TypeError(f"tbf16.conv.scale_input: expected bf16, got {x.dtype}")
    nd = x.dim() - 2
    x = _sample_major(x, nd)
    B = x.shape[0]
    n = x[0].numel() if B else 0
    exps = torch.empty((B,), device=x.device, dtype=torch.int32)
    x16 = torch.empty_like(x, dtype=torch.float16)
    if B and n:
        wsb = lib().tbf16_conv_input_ws_bytes(B, n)
        ws = torch.empty(max(wsb, 16), device=x.device, dtype=torch.uint8)
        launch("tbf16_conv_input", x, ptr(x), B, n, int(t), ptr(exps), ptr(x16), ptr(ws), ws.numel())
    elif B:
        exps.fill_(1 - int(t))
    return exps, x16


def unscale_output(y16: torch.Tensor, exps: torch.Tensor, w_sinv: torch.Tensor, bias=None) -> torch.Tensor:
    """fp16 (B, O, *spatial) -> bf16 y16 * 2^e[b] * w_sinv[o] + bias[o] (conv.py:56-60)."""
    _dev_check(y16, exps, w_sinv, bias)
    if y16.dtype != torch.float16 or exps.dtype != torch.int32 or exps.numel() != y16.shape[0]:
        raise TypeError("tbf16.conv.unscale_output: expected fp16 y16 and int32 exponents, one per sample")
    exps = exps.contiguous()
    nd = y16.dim() - 2
    y16 = _sample_major(y16, nd)
    cl = 0 if y16.is_contiguous() else 1
    B, O = y16.shape[:2]
    P = y16[0, 0].numel() if B and O else 0
    out = torch.empty_like(y16, dtype=torch.bfloat16)
    ws = w_sinv.float().contiguous()
    b = None if bias is None else bias.detach().float().contiguous()
    if out.numel():
        launch("tbf16_conv_epilogue", y16, ptr(y16), B, O, P, cl, ptr(exps), ptr(ws), ptr(b), ptr(out))
    return out


class ConvPlan(NamedTuple):
    """What convert_conv decided for one convolution."""
    target_exp: int   # the input's per-sample target exponent (_target_exp of the weight's fan-in)
    pointwise: bool   # 1x1, stride 1, unpadded, ungrouped: a per-pixel linear layer


def _pointwise(conv: nn.Module) -> bool:
    pad = conv.padding
    unpadded = pad == "valid" or (not isinstance(pad, str) and not any(pad))
    return unpadded and conv.groups == 1 and set(conv.kernel_size) == {1} and set(conv.stride) == {1}


def _pair(v) -> ctypes.Array:
    return (ctypes.c_int64 * 2)(*v)


# Multiply-adds below which the fp16 convolution stays the library's.
_NATIVE_MIN_MACS = 1 << 29
# Bytes of a padded input copy that are taken whatever the channels. Of 491 convolutions of
# 3 to 96 channels (3x3, strided 3x3, 5x5, strided 7x7; 128 to 1024 pixels a side; both
# layouts), native against library, this takes 298, none more than 4% slower and the median
# half the time (16 -> 64 at 256 x 256: 28 us against 55). At 32 MiB they begin to lose (16 -> 16
# at 512 x 512: 70 us against 55; 8 -> 8 at 1024 x 1024: 222 against 98).
_NATIVE_MAX_PADDED = 28 << 20
# Products spent on padding that the native kernel is given, after what the library path
# costs more: per output pixel its own slower products (1.5 for each real one), im2col (as 32
# products a value) and the fp16 output (256 a value). Of 720 convolutions of 2 to 48 channels
# (taps 2x2 to 11x11, 24 to 768 outputs, copies to 60 MiB) this leaves 372, the worst 19%
# slower than the library, 7 by more than 5%; without it 3 -> 320 at 460 x 460, 11 x 11, takes
# 944 us against 243, 8 -> 320 at 464 x 464, 7 x 7, twice the library's time.
_NATIVE_MAX_WASTE = 8_000_000_000


def _native_layout(conv: nn.Module, x: torch.Tensor, padding, bias):
    """0 (contiguous) or 1 (channels last) when the native 2-D convolution takes this
    call, else None: one group, zero padding given in numbers, a bf16 bias, an input
    dense in exactly one of the two layouts, as many channels as the weight has, the weight
    still fp16 (the library's convolution refuses any other).
    Small convolutions (_NATIVE_MIN_MACS) keep the library's fp16 convolution and its
    fp16 rounding: their results are pinned bit for bit to the reference's formula on
    that call. The native kernel is the faster one there too (64 -> 64 at 16 x 16: 22 us
    against 51)."""
    w16 = conv.weight16  # (a module's buffers are slow to look up)
    if (x.dim() != 4 or w16.dim() != 4 or conv.groups != 1 or isinstance(padding, str) or x.data_ptr() % 16
            or w16.dtype != torch.float16 or not w16.is_contiguous()
            or (bias is not None and bias.dtype != torch.bfloat16)):
        return None
    B, C, H, W = x.shape
    O, Cw, KH, KW = w16.shape
    nchw, nhwc = x.is_contiguous(), x.is_contiguous(memory_format=torch.channels_last)
    if C != Cw or nchw == nhwc or (nhwc and C % 8):
        return None
    ph, pw = (padding, padding) if isinstance(padding, int) else padding
    sh, sw = conv.stride
    pixels = B * H * W // (sh * sw)  # the output's, up to its edges
    if pixels * C * O * KH * KW < _NATIVE_MIN_MACS:
        return None
    # The kernels' copy of the input has its channels padded to a multiple of 64: it is the
    # memory of the call, and with few channels its products are most of the time. It is
    # taken where it is small or no larger than the two fp16 tensors around the library's
    # convolution, and the products with zeros are few enough.
    padded = B * (H + 2 * ph) * (W + 2 * pw) * (C + -C % 64)
    taps = KH * KW
    if pixels * ((O + -O % 64) * taps * (C + -C % 64 - 2.5 * C) - 32 * taps * C - 256 * O) > _NATIVE_MAX_WASTE:
        return None
    small = 2 * padded <= _NATIVE_MAX_PADDED
    return int(nhwc) if small or (C >= 16 and padded <= B * C * H * W + pixels * O) else None


def _conv2d_native(conv: nn.Module, x: torch.Tensor, padding, bias, layout: int):
    """The whole scaled convolution on the library's own kernels, or None for sizes they
    do not take."""
    B, C, H, W = x.shape
    w16, scale = conv.weight16, conv.weight_scale
    O, Cw, KH, KW = w16.shape
    pad = (padding, padding) if isinstance(padding, int) else padding
    stride, dilation = conv.stride, conv.dilation
    geom = (_pair(stride), _pair(pad), _pair(dilation))
    wsb = lib().tbf16_conv2d_ws_bytes(B, C, H, W, O, KH, KW, *geom)
    if wsb == 0:
        return None
    _dev_check(x, w16, scale, bias)
    Ho = (H + 2 * pad[0] - dilation[0] * (KH - 1) - 1) // stride[0] + 1
    Wo = (W + 2 * pad[1] - dilation[1] * (KW - 1) - 1) // stride[1] + 1
    y = torch.empty((B, O, Ho, Wo), device=x.device, dtype=torch.bfloat16,
                    memory_format=torch.channels_last if layout else torch.contiguous_format)
    ws = torch.empty(wsb, device=x.device, dtype=torch.uint8)
    b = None if bias is None else bias.detach().contiguous()
    s = scale.float().contiguous()
    launch("tbf16_conv2d", x, ptr(x), B, C, H, W, layout, int(conv._tbf16_plan.target_exp), ptr(w16), O, Cw, KH, KW,
           *geom, ptr(s), ptr(b), ptr(y), ptr(ws), wsb)
    return y


def _run_scaled(conv: nn.Module, x: torch.Tensor, bias) -> torch.Tensor:
    """The scaled fp16 convolution of a batched bf16 input (tbf16/conv.py:39-60)."""
    plan = conv._tbf16_plan
    if plan.pointwise:
        O = conv.out_channels
        return scaled_linear(x.movedim(1, -1), conv.weight16.view(O, -1), conv.weight_scale, bias).movedim(-1, 1)
    padding = conv.padding
    if conv.padding_mode != "zeros":  # reflect / replicate / circular: pad first, convolve unpadded
        x = F.pad(x, conv._reversed_padding_repeated_twice, mode=conv.padding_mode)
        padding = 0
    layout = _native_layout(conv, x, padding, bias)
    if layout is not None:
        y = _conv2d_native(conv, x, padding, bias, layout)
        if y is not None:
            return y
    exps, x16 = scale_input(x, plan.target_exp)
    y16 = _CONV[x.dim() - 2](x16, conv.weight16, None, conv.stride, padding, conv.dilation, conv.groups)
    return unscale_output(y16, exps, conv.weight_scale, bias)


class ScaledConvMixin:
    """First base of every converted convolution class TBF16<Conv class>
    (tbf16/conv.py:63-78). It overrides only _conv_forward, so a subclass whose own
    forward ends in super().forward (diffusers' causal 3-D convolutions) keeps
    working; the class it was made from stays a base, so isinstance checks hold."""

    def dequantized_weight(self) -> torch.Tensor:
        """The bf16 weight, rebuilt exactly from weight16 and weight_scale."""
        ws = self.weight_scale.reshape((-1,) + (1,) * (self.weight16.dim() - 1))
        return (self.weight16.float() * ws).to(torch.bfloat16)

    def _conv_forward(self, x, weight, bias):
        # `weight` is the removed parameter (None): the weight lives in weight16
        if x.dtype != torch.bfloat16 or (torch.is_grad_enabled() and x.requires_grad):
            # not bf16, or a gradient is wanted: the native convolution on the rebuilt weight
            b = None if bias is None else bias.to(x.dtype)
            return super()._conv_forward(x, self.dequantized_weight().to(x.dtype), b)
        if x.dim() == self.weight16.dim() - 1:  # unbatched input: one sample
            return _run_scaled(self, x.unsqueeze(0), bias).squeeze(0)
        return _run_scaled(self, x, bias)


@functools.lru_cache(maxsize=None)
def _scaled_class(cls: type) -> type:
    """TBF16<cls.__name__>: cls with ScaledConvMixin in front (one class per cls)."""
    return type(f"TBF16{cls.__name__}", (ScaledConvMixin, cls), {})


def convertible(m: nn.Module) -> bool:
    """A bf16 nn.Conv1d/2d/3d (or subclass) on the GPU that is not converted yet
    (tbf16/conv.py:81-83)."""
    w = getattr(m, "weight", None)
    return (isinstance(m, (nn.Conv1d, nn.Conv2d, nn.Conv3d)) and not isinstance(m, ScaledConvMixin)
            and isinstance(w, torch.Tensor) and w.dtype == torch.bfloat16 and w.is_cuda)


def convert_conv(conv: nn.Module):
    """Convert one bf16 nn.Conv{1,2,3}d (or subclass) in place and return it
    (tbf16/conv.py:86-103). The `weight` parameter becomes None; buffers weight16
    (fp16, the weight's shape) and weight_scale (fp32, one per output channel) hold
    it, and .dequantized_weight() rebuilds the bf16 tensor."""
    w = conv.weight.detach()
    O = w.shape[0]
    w16, ws = prepare_weight(w.reshape(O, -1))
    plan = ConvPlan(_target_exp(w[0].numel()), _pointwise(conv))
    conv.weight = None
    conv.register_buffer("weight16", w16.contiguous().view(w.shape))
    conv.register_buffer("weight_scale", ws)
    conv._tbf16_plan = plan
    conv.__class__ = _scaled_class(type(conv))
    return conv
