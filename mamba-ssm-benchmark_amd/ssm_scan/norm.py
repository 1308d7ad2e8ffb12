"""RMSNorm on the HIP engine: the LM's pre-norms (models/common.py:8-16).

``rms_norm(x, weight, eps)`` computes ``(x * rsqrt(mean(x^2, -1) + eps)) * weight`` in one
launch forward and two backward (the row kernel and the weight-gradient sum), in place of the
six forward and about ten backward torch kernels of the composed expression.  float32 rows of
up to 1024 elements with a float32 weight run on the kernels.  Other inputs keep the
reference's torch expression on the GPU, which gives what the reference gives: a bf16
residual stream under autocast (its product with the float32 weight promotes), float64 rows
(the reference normalizes them in float32, `x.float()`), wider rows.  The C ABI also takes
float64 rows, computed in float64 throughout.
"""

import torch

from . import _abi
from .hip_scan import _require_gpu

MAX_DIM = 1024


class RMSNormFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, eps):
        out, x2, w, rstd = _abi.host().norm_forward(x, weight, float(eps))
        ctx.save_for_backward(x2, w, rstd)
        ctx.eps = float(eps)
        return out

    @staticmethod
    def backward(ctx, dout):
        dx, dw = _abi.host().norm_backward(*ctx.saved_tensors, dout, ctx.eps)
        return dx, dw, None


def rms_norm_reference(x, weight, eps):
    """models/common.py:14-16 as torch ops (any dtype)."""
    xf = x.float()
    return (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)).to(x.dtype) * weight


def rms_norm(x, weight, eps=1e-5):
    """models/common.py:14-16.  The kernels run for float32 x and weight and a last dimension
    <= 1024; otherwise the reference's torch expression runs on the GPU."""
    _require_gpu(x, weight)
    if tuple(weight.shape) != (x.shape[-1],):  # the kernels read dim weights
        raise ValueError(f"weight must be ({x.shape[-1]},), got {tuple(weight.shape)}")
    if (x.dtype == torch.float32 and weight.dtype == torch.float32 and 0 < x.shape[-1] <= MAX_DIM
            and x.numel() > 0):
        return RMSNormFn.apply(x, weight, eps)
    return rms_norm_reference(x, weight, eps)
