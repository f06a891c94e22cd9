"""Autograd for the DiNAT all-in-one operators.

The reference's public ``na{1,2}d_qk_rpb`` / ``na{1,2}d_av_fused`` are
forward-only; its Metal backward lives in separate functions
(``extras/allin1/functional_metal.py:1206-1918``: dq, dk, drpb and dattn,
dvalue).  Here both directions are joined in ``torch.autograd.Function`` s
whose backward calls the library's deterministic kernels: operators with
their nodes in C++ (``csrc/na_torch.cpp``), or the same as Python Functions
where the operator library is not built, for arguments it does not take and
under ``python_autograd()``.
"""

from __future__ import annotations

import torch

from .._core import _lib, hip
from . import fused as _fused


class _QKRPB(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, rpb, kernel_size, dilation, scale, heads_first):
        ctx.save_for_backward(q, k)
        ctx.args = (kernel_size, dilation, scale, heads_first)
        ctx.rpb_dtype = None if rpb is None else rpb.dtype
        return hip.rpb_qk_forward(q, k, rpb, kernel_size, dilation, scale, heads_first)

    @staticmethod
    def backward(ctx, d_logits):
        q, k = ctx.saved_tensors
        need_q, need_k, need_rpb = ctx.needs_input_grad[:3]
        dq, dk, drpb = hip.rpb_qk_backward(q, k, d_logits, *ctx.args, need_q=need_q,
                                           need_k=need_k,
                                           need_rpb=need_rpb and ctx.rpb_dtype is not None)
        if dk is not None and dk.dtype != k.dtype:
            dk = dk.to(k.dtype)
        if drpb is not None and drpb.dtype != ctx.rpb_dtype:
            drpb = drpb.to(ctx.rpb_dtype)
        return dq, dk, drpb, None, None, None, None


class _AVRPB(torch.autograd.Function):
    @staticmethod
    def forward(ctx, attn, v, kernel_size, dilation, heads_first, out_dtype):
        ctx.save_for_backward(attn, v)
        ctx.args = (kernel_size, dilation, heads_first)
        return hip.rpb_av_forward(attn, v, kernel_size, dilation, heads_first, out_dtype)

    @staticmethod
    def backward(ctx, d_out):
        attn, v = ctx.saved_tensors
        need_a, need_v = ctx.needs_input_grad[:2]
        da, dv = hip.rpb_av_backward(attn, v, d_out, *ctx.args, need_attn=need_a, need_v=need_v)
        if da is not None and da.dtype != attn.dtype:
            da = da.to(attn.dtype)
        return da, dv, None, None, None, None


def _op(name, a, b, kernel_size, dilation):
    """(operator, kernel and dilation per axis), or None."""
    rank = a.dim() - 3
    if _fused._py_autograd or rank not in (1, 2):
        return None
    op = _lib.node_op(name, a, b)
    if op is None:
        return None
    return (op, hip._per_axis(kernel_size, rank), hip._per_axis(dilation, rank))


def _axes(v):
    """An int, or a per-axis tuple of ints (non-square windows)."""
    return tuple(int(x) for x in v) if isinstance(v, (tuple, list)) else int(v)


def qk_rpb_with_grad(q, k, rpb, kernel_size, dilation, scale=None, heads_first=False):
    """float32 logits of the fused QK + RPB op, differentiable in q, k, rpb.
    kernel_size / dilation: an int or one value per axis."""
    op = _op("rpb_qk", q, k, kernel_size, dilation)
    if op is not None and q.shape == k.shape:
        heads = q.shape[1 if heads_first else -2]
        if rpb is None or (rpb.device == q.device and rpb.is_floating_point()
                           and tuple(rpb.shape) == (heads, *(2 * x - 1 for x in op[1]))):
            return op[0](q, k, rpb, op[1], op[2], 0.0 if scale is None else float(scale),
                         scale is not None, bool(heads_first), _lib.stream_of(q))
    return _QKRPB.apply(q, k, rpb, _axes(kernel_size), _axes(dilation), scale,
                        bool(heads_first))


def av_rpb_with_grad(attn, v, kernel_size, dilation, heads_first=False,
                     out_dtype=torch.float32):
    """AV op output, differentiable in attn and v."""
    op = _op("rpb_av", v, attn, kernel_size, dilation)
    if (op is not None and out_dtype in (torch.float32, v.dtype)
            and tuple(attn.shape) == hip._slots_shape(v, op[1], heads_first)):
        return op[0](attn, v, op[1], op[2], bool(heads_first), out_dtype == torch.float32,
                     _lib.stream_of(v))
    return _AVRPB.apply(attn, v, _axes(kernel_size), _axes(dilation), bool(heads_first),
                        out_dtype)


__all__ = ["qk_rpb_with_grad", "av_rpb_with_grad"]
