"""Packed main weight for the fused NHWC kernel.

The fused kernel reads the weight in the layout dcn_pack_weight produces (MFMA-fragment
blocks for fp16 / bf16, [Cout][kh][kw][C] for fp32). The weight is packed on every call,
as the reference flattens its weight on every call (dcn_split_nhwc.py:143,
fused_tl.py:399): one small kernel (a few microseconds for a 256 x 256 x 3 x 3 weight)
beside the convolution, and no cached copy that a write through ``weight.data``, an EMA
swap or another kernel could leave stale.
"""
from __future__ import annotations

import torch


def _ext():
    import _modulated_deform_conv_ext as ext
    return ext


def pack_weight(weight: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    """Pack weight [Cout, C, kh, kw] converted to `dtype`."""
    return _ext().dcn_pack_weight(weight.detach().to(dtype).contiguous())


def split_applies(x, channels, channels_out, taps):
    """fp32 shapes of the split kernel: whole 32-channel K steps, at most 9 taps, and buffers
    under 2 GiB."""
    lim = 2 ** 31 - 256
    return (x.dtype == torch.float32 and channels % 32 == 0 and taps <= 9
            and 4 * x.numel() <= lim
            and 6.5 * (channels_out + 15) * channels * taps <= lim)


def fused_conv(x, offset, mask, weight, bias, sizes, out, relu=False):
    """The fused deformable forward into out, with the weight packed for the kernel that takes
    the shape. sizes = (B, C, H, W, Ho, Wo, Cout, kh, kw, ph, pw, sh, sw, dh, dw); offset 2T
    with a mask, or the 3T y (then mask is ignored). relu: fp32 shapes of the split kernel only
    (returns whether it was applied).

    fp32: C % 32 == 0 runs on the bf16 matrix cores (dcn_fused_fwd_nhwc_f32), other channel
    counts on the fp32 ones."""
    ext = _ext()
    if split_applies(x, sizes[1], sizes[6], sizes[7] * sizes[8]):
        split = ext.dcn_split_weight(weight.detach().to(x.dtype).contiguous())
        ext.dcn_fused_fwd_nhwc_f32(x, offset, mask, split, bias, *sizes, out, relu)
        return relu
    ext.dcn_fused_fwd_nhwc(x, offset, mask, pack_weight(weight, x.dtype), bias, *sizes, out)
    return False


def columns_grad_f32(dout, weight):
    """The columns' gradient [M, T*C] = dout [M, Cout] @ W, fp32, W [Cout, C, kh, kw] with its
    columns in (tap, C) order."""
    ext = _ext()
    cout, c, kh, kw = weight.shape
    lim = 2 ** 31 - 256
    if (c % 16 == 0 and cout % 32 == 0 and kh * kw <= 9 and 4 * dout.numel() <= lim
            and 6.5 * weight.numel() <= lim):
        dcol = dout.new_empty(dout.size(0), kh * kw * c)
        ext.gemm_f32(dout, ext.dcn_split_weight(weight.contiguous(), True), kh * kw * c, dcol)
        return dcol
    return torch.mm(dout, weight.permute(0, 2, 3, 1).reshape(cout, kh * kw * c))


def weight_grad(cols, dout, weight, out_dtype):
    """The weight's gradient [Cout, C, kh, kw] from the columns [M, T*C] and dout [M, Cout],
    summed in fp32 and rounded once to out_dtype."""
    cout, c, kh, kw = weight.shape
    if out_dtype != torch.float64:
        grad = _ext().dcn_weight_grad(cols, dout, kh, kw, out_dtype)
        if grad is not None:
            return grad
    acc = cols.dtype if cols.dtype == torch.float64 else torch.float32
    grad = torch.mm(dout.t().to(acc), cols.to(acc)).view(cout, kh, kw, c)
    return grad.permute(0, 3, 1, 2).contiguous().to(out_dtype)
