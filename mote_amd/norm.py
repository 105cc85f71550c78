"""Fused residual add + RMSNorm on MI355X (mote/model/norm.py:26-59 of the reference).

`RMSNorm` keeps the reference's constructor, parameter and call signature:
forward(x, residual=None, prenorm=False, residual_in_fp32=True) adds the residual (in fp32 when
residual_in_fp32), normalises in fp32 and returns y in the dtype of x, and with prenorm also the new
residual stream (fp32 when residual_in_fp32). Underneath are the custom ops `mote::add_rms_norm` /
`mote::add_rms_norm_bwd` over the C ABI (mote_add_rms_norm_fwd / _bwd): one HIP launch forward, two
backward (the weight gradient is summed in a fixed order, so every gradient is reproducible). There is
no CPU path: CPU tensors raise.
"""

from __future__ import annotations

from typing import Optional, Tuple

import torch
import torch.nn as nn

from . import _lib as L


def _sum_dtype(x: torch.Tensor, residual: Optional[torch.Tensor], prenorm: bool, residual_in_fp32: bool):
    """dtype of the summed stream s (norm.py:50-55): fp32 when residual_in_fp32 and a residual is
    added or prenorm; otherwise x + residual in torch's promotion, or x itself."""
    if residual is not None:
        return torch.float32 if residual_in_fp32 else torch.promote_types(x.dtype, residual.dtype)
    if residual_in_fp32 and prenorm:
        return torch.float32
    return x.dtype


@torch.library.custom_op("mote::add_rms_norm", mutates_args=())
def _add_rms_norm(x: torch.Tensor, weight: torch.Tensor, residual: Optional[torch.Tensor], eps: float, prenorm: bool,
                  residual_in_fp32: bool) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    if not x.is_cuda:
        raise RuntimeError("mote::add_rms_norm needs the HIP library and an MI355X")
    # s is x itself when it is not materialised: an empty tensor stands in (outputs may not alias x)
    sdt = _sum_dtype(x, residual, prenorm, residual_in_fp32)
    return L.native().add_rms_norm(x, weight, residual, eps, sdt, L.stream_of(x))


@_add_rms_norm.register_fake
def _add_rms_norm_fake(x, weight, residual, eps, prenorm, residual_in_fp32):
    rows = x.numel() // x.shape[-1]
    sdt = _sum_dtype(x, residual, prenorm, residual_in_fp32)
    s = x.new_empty(x.shape, dtype=sdt) if (residual is not None or sdt != x.dtype) else x.new_empty(0)
    return x.new_empty(x.shape), s, x.new_empty((rows,), dtype=torch.float32)


@torch.library.custom_op("mote::add_rms_norm_bwd", mutates_args=())
def _add_rms_norm_bwd(dy: torch.Tensor, dres_out: Optional[torch.Tensor], s: torch.Tensor, rstd: torch.Tensor,
                      weight: torch.Tensor, x_dtype: torch.dtype, has_res: bool, res_dtype: torch.dtype
                      ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """(dx, dresidual, dweight); dresidual is empty when has_res is false."""
    return L.native().add_rms_norm_bwd(dy, dres_out, s, rstd, weight, x_dtype, has_res, res_dtype, L.stream_of(s))


@_add_rms_norm_bwd.register_fake
def _add_rms_norm_bwd_fake(dy, dres_out, s, rstd, weight, x_dtype, has_res, res_dtype):
    return (s.new_empty(s.shape, dtype=x_dtype), s.new_empty(s.shape if has_res else 0, dtype=res_dtype),
            s.new_empty((s.shape[-1],), dtype=torch.float32))


def _setup(ctx, inputs, output):
    x, weight, residual, eps, prenorm, residual_in_fp32 = inputs
    _y, s, rstd = output
    ctx.s_is_x = s.shape != x.shape          # the empty stand-in: s is x itself
    ctx.save_for_backward(x if ctx.s_is_x else s, rstd, weight)
    ctx.x_dtype = x.dtype
    ctx.has_res = residual is not None
    ctx.res_dtype = residual.dtype if residual is not None else x.dtype
    ctx.w_dtype = weight.dtype
    # no zero tensors for rstd, or for the stream when it is not differentiated
    ctx.set_materialize_grads(False)


def _backward(ctx, dy, ds_out, _drstd):
    s, rstd, weight = ctx.saved_tensors
    if dy is None:
        dy = torch.zeros_like(s, dtype=ctx.x_dtype)
    if ctx.s_is_x or (ds_out is not None and ds_out.shape != s.shape):
        ds_out = None                       # the returned stream is x itself: autograd routes its gradient
    dx, dres, dw = _add_rms_norm_bwd(dy, ds_out, s, rstd, weight, ctx.x_dtype, ctx.has_res, ctx.res_dtype)
    return dx, dw.to(ctx.w_dtype), (dres if ctx.has_res else None), None, None, None


_add_rms_norm.register_autograd(_backward, setup_context=_setup)


def add_rms_norm(x: torch.Tensor, weight: torch.Tensor, residual: Optional[torch.Tensor] = None, eps: float = 1e-5,
                 prenorm: bool = False, residual_in_fp32: bool = True):
    """Functional form of RMSNorm.forward (norm.py:36-59)."""
    y, s, _ = _add_rms_norm(x, weight, residual, float(eps), bool(prenorm), bool(residual_in_fp32))
    if not prenorm:
        return y
    return y, (s if s.shape == x.shape else x)


class RMSNorm(nn.Module):
    """RMSNorm(dim, eps=1e-5) with the fused-residual call of mote/model/norm.py:26-59."""

    def __init__(self, dim: int, eps: float = 1e-5, device=None, dtype=None):
        super().__init__()
        self.eps = eps
        self.weight = nn.Parameter(torch.ones(dim, device=device, dtype=dtype))

    def forward(self, x: torch.Tensor, residual: Optional[torch.Tensor] = None, prenorm: bool = False,
                residual_in_fp32: bool = True):
        return add_rms_norm(x, self.weight, residual, self.eps, prenorm, residual_in_fp32)
