"""Weights and gradients of the layers: packing for the fused NHWC kernel, and the gradient
products of the backward passes.

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
