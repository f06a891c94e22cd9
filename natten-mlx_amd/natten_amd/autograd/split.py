"""Autograd for the split QK / AV ops (reference ``autograd/split.py``).

With the built-in ``hip`` backend both are operators with their autograd
nodes in C++ (``csrc/na_torch.cpp``); ``_QK`` / ``_AV`` below are the same ops
as Python Functions over the backend's hooks, for other registered backends,
where the operator library is not built, and under ``python_autograd()``.
"""

from __future__ import annotations

import torch

from .._core import _lib, ops
from .._core import hip as _hip
from . import fused as _fused

_QK_FWD = {1: ops.na1d_qk_forward, 2: ops.na2d_qk_forward, 3: ops.na3d_qk_forward}
_QK_BWD = {1: ops.na1d_qk_backward, 2: ops.na2d_qk_backward, 3: ops.na3d_qk_backward}
_AV_FWD = {1: ops.na1d_av_forward, 2: ops.na2d_av_forward, 3: ops.na3d_av_forward}
_AV_BWD = {1: ops.na1d_av_backward, 2: ops.na2d_av_backward, 3: ops.na3d_av_backward}


class _QK(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, kernel_size, stride, dilation, is_causal, scale):
        rank = q.dim() - 3
        ctx.save_for_backward(q, k)
        ctx.args = (kernel_size, stride, dilation, is_causal, scale)
        return _QK_FWD[rank](q, k, kernel_size, stride, dilation, is_causal, scale)

    @staticmethod
    def backward(ctx, grad_attn):
        q, k = ctx.saved_tensors
        rank = q.dim() - 3
        dq, dk = _QK_BWD[rank](q, k, grad_attn, *ctx.args)
        return dq, dk, None, None, None, None, None


class _AV(torch.autograd.Function):
    @staticmethod
    def forward(ctx, attn, v, kernel_size, stride, dilation, is_causal):
        rank = v.dim() - 3
        ctx.save_for_backward(attn, v)
        ctx.args = (kernel_size, stride, dilation, is_causal)
        return _AV_FWD[rank](attn, v, kernel_size, stride, dilation, is_causal)

    @staticmethod
    def backward(ctx, grad_out):
        attn, v = ctx.saved_tensors
        rank = v.dim() - 3
        dattn, dv = _AV_BWD[rank](attn, v, grad_out, *ctx.args)
        return dattn, dv, None, None, None, None


def _op(name, a, b):
    if _fused._py_autograd or ops.backend_module() is not _hip:
        return None
    return _lib.node_op(name, a, b)


def _qk(q, k, kernel_size, stride, dilation, is_causal, scale):
    op = _op("qk", q, k)
    if op is not None:
        flags = ((_lib.NA_FLAG_GENERIC if _hip._force_generic else 0)
                 | (_lib.NA_FLAG_NO_LEAN if _hip._no_lean else 0))
        return op(q, k, kernel_size, stride, dilation, [int(bool(c)) for c in is_causal],
                  _hip._scale(scale, q.shape[-1]), flags, _lib.stream_of(q))
    return _QK.apply(q, k, tuple(kernel_size), tuple(stride), tuple(dilation),
                     tuple(bool(c) for c in is_causal), scale)


def _av(attn, v, kernel_size, stride, dilation, is_causal):
    op = _op("av", attn, v)
    if op is not None:
        _hip._check_attn_shape(attn, v, kernel_size, stride)
        return op(attn, v, kernel_size, stride, dilation, [int(bool(c)) for c in is_causal],
                  _lib.stream_of(v))
    return _AV.apply(attn, v, tuple(kernel_size), tuple(stride), tuple(dilation),
                     tuple(bool(c) for c in is_causal))


na1d_qk_with_grad = na2d_qk_with_grad = na3d_qk_with_grad = _qk
na1d_av_with_grad = na2d_av_with_grad = na3d_av_with_grad = _av
