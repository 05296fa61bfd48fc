"""Depthwise conv1d candidate for the F.conv1d contest.

Interface of the reference's depthwise_conv1d_ops (amd_tuned_torch/depthwise_conv1d_ops.py:
95-247): `available`, `maybe_contiguous`, `_out_len`, the torch.library ops
`amd_tuned_torch::depthwise_conv1d_forward/backward` with fake (meta) implementations,
`conv1d_forward`/`conv1d_backward`, `DepthwiseConv1dFn` and `depthwise_conv1d_candidate`.
The forward runs this package's gfx950 kernels (fp32 accumulation): the (B, C, L) layout
for any width K <= 64, the (B, L, C) layout (weight [K, C]) through the channels-last kernel
for K <= 8, stock F.conv1d on the transposed view beyond that; the reference's kernel only
accepted odd K (conv1d.h:76).  The backward is native too
(`_native.dwconv1d_backward`: du through the forward kernel with reversed weights, dweight /
dbias through one streaming reduction kernel) where it applies -- K <= 5 for the weight
gradient, padding <= K-1 for du -- and stock aten.convolution_backward for the rest.
"""
from __future__ import annotations

from typing import Any, Optional, Tuple

import torch

from . import _native
from . import autograd_state
from . import compile_ops

KMAX = 64
PADMAX = 64


def available() -> bool:
    return _native.available()


def maybe_contiguous(x: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    """Copy only when the last dimension is not unit-stride (depthwise_conv1d_ops.py:104-109)."""
    return x.contiguous() if x is not None and x.stride(-1) != 1 else x


def _out_len(length: int, padding: int, width: int) -> int:
    """l_out = l + 2 * padding - k + 1 (depthwise_conv1d_ops.py:112-118)."""
    return length + 2 * padding - width + 1


def _stock_forward_blh(input_, weight, bias, padding: int):
    """BLH forward through stock F.conv1d on the transposed view (shapes the kernel declines)."""
    K, C = weight.shape
    w = weight.t().unsqueeze(1)
    if w.dtype != input_.dtype:
        w = w.to(input_.dtype)
    b = bias.to(input_.dtype) if bias is not None else None
    # the original F.conv1d: the patched one would route this channel-last view back here
    from . import miopen_fallback
    conv1d = miopen_fallback._original_conv1d or torch.nn.functional.conv1d
    y = conv1d(input_.transpose(1, 2), w, b, 1, padding, 1, C)
    return y.transpose(1, 2).contiguous()


def _forward(input_, weight, bias, padding: int, is_bhl: bool):
    if is_bhl:
        return _native.conv1d_forward(input_, weight, bias, padding, True)
    try:
        return _native.conv1d_forward(input_, weight, bias, padding, False)
    except _native.Unsupported:
        return _stock_forward_blh(input_, weight, bias, padding)


def _stock_backward(dout, input_, weight, bias, padding: int, is_bhl: bool, needs=(True, True, True)):
    if not is_bhl:
        # (B, L, C) tensors through the (B, C, L) op on transposed views; weight [K, C]
        K, C = weight.shape
        du, dw, db = torch.ops.aten.convolution_backward(
            dout.transpose(1, 2), input_.transpose(1, 2), weight.t().unsqueeze(1).to(input_.dtype), [C], [1],
            [padding], [1], False, [0], C, list(needs))
        return (None if du is None else du.transpose(1, 2).contiguous(),
                None if dw is None else dw.reshape(C, K).t().contiguous().to(weight.dtype),
                None if db is None else db.to(dout.dtype))
    C, K = weight.shape
    du, dw, db = torch.ops.aten.convolution_backward(
        dout.contiguous(), input_, weight.unsqueeze(1), [C], [1], [padding], [1], False, [0], C,
        list(needs))
    return (du, None if dw is None else dw.reshape(C, K).to(weight.dtype),
            None if db is None else db.to(dout.dtype))


def _backward(dout, input_, weight, bias, padding: int, is_bhl: bool):
    """(du, dweight, dbias) of conv1d_forward (conv1d_bwd_hip_bhl.hip:78-116 semantics:
    dweight in weight's dtype, dbias in dout's dtype): each part native where the library
    serves it, the rest stock."""
    du = dw = db = None
    if not is_bhl and input_.is_cuda and _native.available():
        # (B, L, C) layout, weight [K, C]: du, dweight and dbias in one pass over x and dout
        # where the fused kernel takes the shape (K 2..4); else du through the channels-last
        # forward kernel on dout with the taps reversed and dweight / dbias through its
        # channels-last reduction
        K = weight.shape[0]
        wf = weight if weight.dtype in (torch.float32, input_.dtype) else weight.float()
        if dout.stride(-1) == 1 and input_.stride(-1) == 1:
            try:
                du, dw32, db32 = _native.dwconv1d_cl_bwd(input_, dout, wf.t(), padding)
                return du, dw32.t().contiguous().to(weight.dtype), db32.to(dout.dtype)
            except _native.Unsupported:
                pass
        try:
            if padding <= K - 1:
                du = _native.dwconv1d_cl(dout, wf.t().flip(-1), None, K - 1 - padding, input_.shape[1])
        except _native.Unsupported:
            du = None
        try:
            dw32, db32 = _native.dwconv1d_cl_bwd_weight(input_, dout, K, padding)
            dw, db = dw32.t().contiguous().to(weight.dtype), db32.to(dout.dtype)
        except _native.Unsupported:
            dw = db = None
    elif input_.is_cuda and _native.available():
        dout = dout.contiguous()
        K = weight.shape[-1]
        try:  # du, dw and db together (one pass over x and dout where the fused kernel applies);
            # dw / db come back None when only du is native (K > 5)
            du, dw32, db32 = _native.dwconv1d_backward(dout, input_, weight, padding, (True, True, True))
            if dw32 is not None:
                dw, db = dw32.to(weight.dtype), db32.to(dout.dtype)
        except _native.Unsupported:
            du = dw = db = None
        if du is None:
            try:
                _, dw32, db32 = _native.dwconv1d_backward(dout, input_, weight, padding, (False, True, True))
                dw, db = dw32.to(weight.dtype), db32.to(dout.dtype)
            except _native.Unsupported:
                dw = db = None
    if du is None or dw is None:
        su, sw, sb = _stock_backward(dout, input_, weight, bias, padding, is_bhl,
                                     (du is None, dw is None, dw is None))
        du = su if du is None else du
        if dw is None:
            dw, db = sw, sb
    return du, dw, db


def _already_registered(name: str) -> bool:
    return hasattr(torch.ops, "amd_tuned_torch") and hasattr(torch.ops.amd_tuned_torch, name)


if hasattr(torch.library, "custom_op") and not _already_registered("depthwise_conv1d_forward"):

    @torch.library.custom_op("amd_tuned_torch::depthwise_conv1d_forward", mutates_args=())
    def _fwd_op(input_: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, padding: int,
                is_bhl: bool) -> torch.Tensor:
        return _forward(input_, weight, bias, padding, is_bhl)

    @_fwd_op.register_fake
    def _fwd_fake(input_, weight, bias, padding, is_bhl):
        del bias
        if is_bhl:
            b, d, length = input_.shape
            return input_.new_empty(b, d, _out_len(length, padding, weight.shape[1]))
        b, length, d = input_.shape
        return input_.new_empty(b, _out_len(length, padding, weight.shape[0]), d)

    @torch.library.custom_op("amd_tuned_torch::depthwise_conv1d_backward", mutates_args=())
    def _bwd_op(dout: torch.Tensor, input_: torch.Tensor, weight: torch.Tensor,
                bias: torch.Tensor, padding: int, is_bhl: bool
                ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
        du, dw, db = _backward(dout, input_, weight, bias, padding, is_bhl)
        return du.contiguous(), dw.contiguous(), db.contiguous()

    @_bwd_op.register_fake
    def _bwd_fake(dout, input_, weight, bias, padding, is_bhl):
        # du/dweight take input/weight's shape and dtype; dbias takes bias's shape and
        # dout's dtype (depthwise_conv1d_ops.py:173-187)
        return input_.new_empty(input_.shape), weight.new_empty(weight.shape), dout.new_empty(bias.shape)

    _fwd_impl = torch.ops.amd_tuned_torch.depthwise_conv1d_forward
    _bwd_impl = torch.ops.amd_tuned_torch.depthwise_conv1d_backward
elif _already_registered("depthwise_conv1d_forward"):
    _fwd_impl = torch.ops.amd_tuned_torch.depthwise_conv1d_forward
    _bwd_impl = torch.ops.amd_tuned_torch.depthwise_conv1d_backward
else:
    def _fwd_impl(input_, weight, bias, padding, is_bhl):
        return _forward(input_, weight, bias, padding, is_bhl)

    def _bwd_impl(dout, input_, weight, bias, padding, is_bhl):
        return _backward(dout, input_, weight, bias, padding, is_bhl)


def conv1d_forward(input: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, padding: int,
                   is_bhl: bool = True) -> torch.Tensor:
    """`weight` is the squeezed [C, K] kernel, `bias` is required ([C])."""
    input, weight, bias = maybe_contiguous(input), maybe_contiguous(weight), maybe_contiguous(bias)
    return _fwd_impl(input, weight, bias, padding, is_bhl)


def conv1d_backward(dout, input, weight, bias, padding: int, is_bhl: bool = True):
    dout, input, weight, bias = (maybe_contiguous(dout), maybe_contiguous(input),
                                 maybe_contiguous(weight), maybe_contiguous(bias))
    return _bwd_impl(dout, input, weight, bias, padding, is_bhl)


class DepthwiseConv1dFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, input, weight, bias, padding, is_bhl):
        ctx.padding, ctx.is_bhl = padding, is_bhl
        ctx.save_for_backward(input, weight, bias)
        return conv1d_forward(input, weight, bias, padding, is_bhl)

    @staticmethod
    def backward(ctx, dout):
        input, weight, bias = ctx.saved_tensors
        if not compile_ops.is_compiling() and autograd_state.graph_wanted(dout, input, weight):
            # differentiable themselves, in the wider of the types (fp32 weights enter unrounded)
            acc = torch.promote_types(input.dtype, weight.dtype)
            du, dw, db = _stock_backward(dout.to(acc), input.to(acc), weight.to(acc), bias, ctx.padding, ctx.is_bhl)
            return du.to(input.dtype), dw.to(weight.dtype), db.to(bias.dtype), None, None
        du, dw, db = conv1d_backward(dout, input, weight, bias, ctx.padding, ctx.is_bhl)
        return du, dw, db, None, None


def depthwise_conv1d_candidate(input: torch.Tensor, weight: torch.Tensor,
                               bias: Optional[torch.Tensor], stride: Any, padding: Any,
                               dilation: Any, groups: int) -> torch.Tensor:
    """Candidate with F.conv1d's calling convention (un-squeezed [C, 1, K] weight, optional
    bias); the caller has already checked stride == dilation == 1, groups == C."""
    channels = weight.shape[0]
    squeezed = weight.squeeze(1)
    if bias is None:
        bias = torch.zeros(channels, device=input.device, dtype=weight.dtype)
    pad = padding[0] if isinstance(padding, (tuple, list)) else padding
    return DepthwiseConv1dFn.apply(input, squeezed, bias, pad, True)
