"""Causal depthwise conv1d + SiLU on the HIP engine: the producer of the scan's input.

Counterpart of models/mamba.py:101-107 (F.pad / state concat, F.conv1d with groups=D, SiLU,
and the conv-state update of :104-106).  ``x`` is the (B, L, D) view the in_proj split gives
(no transposes or copies are needed); the output is (B, L, D) contiguous, which the fused scan
reads directly.  Training uses ``causal_conv1d`` (differentiable in x, weight and bias); the
recurrent decode step passes a ``state`` (B, D, W-1) that is read and then updated in place.
"""

import torch

from . import _abi
from .hip_scan import _require_gpu


def _weight2d(weight):
    """nn.Conv1d's (D, 1, W) weight, or a (D, W) tensor, as (D, W)."""
    return weight.reshape(weight.shape[0], weight.shape[-1]) if weight.dim() == 3 else weight


def conv_forward(x, w2, bias, activation):
    """One ssm_conv_fwd launch: (B, L, D) out for x, weight (D, W) and bias in the state type."""
    return _abi.host().conv_forward(x, w2, bias, activation, None)


def conv_backward(x, w2, bias, dout, activation, dx=None):
    """One ssm_conv_bwd launch: (dx, dweight, dbias).  dx may be given (a (B, L, D) view into a
    caller's buffer); it is allocated otherwise."""
    return _abi.host().conv_backward(x, w2, bias, dout, activation, dx)


class CausalConv1dFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias, activation):
        ct = torch.promote_types(x.dtype, torch.float32)
        w2 = weight if weight.dtype == ct else weight.to(ct)
        bv = bias if bias is None or bias.dtype == ct else bias.to(ct)
        out = conv_forward(x, w2, bv, activation)
        ctx.save_for_backward(x, w2, bv)
        ctx.activation = activation
        ctx.wdtype = weight.dtype
        ctx.bdtype = None if bias is None else bias.dtype
        return out

    @staticmethod
    def backward(ctx, dout):
        x, w2, bv = ctx.saved_tensors
        dx, dw, db = conv_backward(x, w2, bv, dout, ctx.activation)
        if dw.dtype != ctx.wdtype:
            dw = dw.to(ctx.wdtype)
        return dx, dw, db if db is None or db.dtype == ctx.bdtype else db.to(ctx.bdtype), None


def causal_conv1d(x, weight, bias=None, state=None, activation=True):
    """out = silu(conv1d(pad_left(x), weight, bias, groups=D)) over time, as (B, L, D).

    x (B, L, D); weight (D, W) or nn.Conv1d's (D, 1, W); bias (D,) or None.  With ``state``
    (B, D, W-1) the previous inputs replace the zero padding and ``state`` is overwritten with
    the last W-1 inputs (models/mamba.py:104-106); that path is not differentiable."""
    _require_gpu(x, weight, bias, state)
    if x.dim() != 3:
        raise ValueError(f"x must be (B, L, D), got {tuple(x.shape)}")
    w2 = _weight2d(weight)
    Bsz, L, D = x.shape
    if w2.shape[0] != D:
        raise ValueError(f"weight must have {D} channels, got {tuple(weight.shape)}")
    if bias is not None and tuple(bias.shape) != (D,):
        raise ValueError(f"bias must be ({D},), got {tuple(bias.shape)}")
    if state is None:
        return CausalConv1dFn.apply(x, w2, bias, bool(activation))
    W = w2.shape[1]
    if tuple(state.shape) != (Bsz, D, W - 1) or state.dtype != x.dtype:
        raise ValueError(f"state must be ({Bsz}, {D}, {W - 1}) of {x.dtype}, got {tuple(state.shape)} {state.dtype}")
    ct = torch.promote_types(x.dtype, torch.float32)
    w2c, bv = w2.detach().to(ct), None if bias is None else bias.detach().to(ct)
    return _abi.host().conv_forward(x, w2c, bv, bool(activation), state)
