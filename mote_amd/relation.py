"""FullRelation on MI355X — the Relation token mixer behind mote/model/relation.py's interface.

Same constructor, parameter names and construction order (relation.py:97-157), same forward
signature and return convention (relation.py:184-268). What runs underneath:

    p1, p2, I~ = mote::qkv_rope(x, [w1; w2; wi])  HIP: one launch for the projections with QK-Norm and
                                                 RoPE on p1/p2 and Givens on I~ in the epilogue
                                                 (bf16, dh 64 / 96 / 128, and 48 without QK-Norm);
                                                 otherwise one hipBLASLt GEMM and mote::rope_givens
    Y, g = mote::relation_fwd(p1, P2, I~)        HIP: the fused Relation core (any T, decode too)
    out = wo(Y [* sigmoid(wg x)])                 Y is token-major already, so no transpose copy

There is no materialized path: `USE_FLASH = False` raises, and so does a CPU tensor. The
materialized restatement lives in the test oracle.
"""

from __future__ import annotations

import math
from typing import Optional, Tuple

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _lib as L
from .arena import ArenaLayer
from .flash_relation import HAS_HIP, HAS_TRITON, flash_relation  # noqa: F401  (re-exported names)

RelationCache = Tuple[torch.Tensor, torch.Tensor]  # (P2 [B,H,S,dh], I~ [B,H,S,dh]) or an ArenaLayer
USE_FLASH = True   # the HIP path; the reference's materialized alternative is not part of this package
FLASH_MIN_T = 16   # kept for callers that read it; the HIP kernels serve every T, T = 1 included


def rope_inv_freq(dim: int, theta: float, device=None) -> torch.Tensor:
    """fp32 [dim/2] table 1 / theta^(2k/dim), computed with the same fp32 ops as relation.py:39 so
    the kernels' angles float(pos) * inv_freq[k] round exactly like the reference's tables. Built on
    the CPU and then moved: a last-ulp difference of the device's pow would grow by the position
    (one ulp of the angle at pos ~ 1000 is ~6e-5 rad)."""
    k2 = torch.arange(0, dim, 2, dtype=torch.float32)
    return (1.0 / (theta ** (k2 / dim))).to(device)


# ---- torch-level RoPE helpers (the names mote/model/relation.py:37-68 exports) ------------------
# The module's own forward runs RoPE inside the HIP prologue kernels; these helpers are for callers
# that rotate rows themselves (mote/infer/graph.py:39, 158-164). They round where the kernels round:
# tables cast to the operand dtype, then every product and sum in that dtype.
def _rope_cos_sin(positions: torch.Tensor, dim: int, theta: float, dtype: torch.dtype) -> Tuple[torch.Tensor, torch.Tensor]:
    """positions [T] (integers) -> cos, sin [T, dim] in `dtype`: fp32 angles pos * inv_freq, the
    half-table repeated for the rotate-half convention (relation.py:37-42)."""
    inv = rope_inv_freq(dim, theta, positions.device)
    ang = positions.to(torch.float32)[:, None] * inv[None, :]
    ang = torch.cat([ang, ang], dim=-1)
    return ang.cos().to(dtype), ang.sin().to(dtype)


_ROPE_CPU_TABLES: "dict" = {}


def rope_tables(S: int, T: int, dim: int, theta: float, dtype: torch.dtype, device=None) -> Tuple[torch.Tensor, torch.Tensor]:
    """cos / sin for absolute positions S .. S+T-1, memoised per (S, T, dim, theta, dtype, device),
    at most 32 entries (relation.py:45-58)."""
    key = (int(S), int(T), int(dim), float(theta), dtype, str(torch.device(device) if device is not None else "cpu"))
    hit = _ROPE_CPU_TABLES.get(key)
    if hit is None:
        if len(_ROPE_CPU_TABLES) >= 32:
            _ROPE_CPU_TABLES.clear()
        hit = _rope_cos_sin(torch.arange(S, S + T, device=device), dim, theta, dtype)
        _ROPE_CPU_TABLES[key] = hit
    return hit


def _rotate_half(x: torch.Tensor) -> torch.Tensor:
    """(x1, x2) -> (-x2, x1) over the two halves of the last axis (relation.py:61-63)."""
    half = x.shape[-1] // 2
    return torch.cat([-x[..., half:], x[..., :half]], dim=-1)


def _apply_rope(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    """x [B, H, T, dh] rotated by tables [T, dh]: x cos + rotate_half(x) sin (relation.py:66-68)."""
    return x * cos[None, None] + _rotate_half(x) * sin[None, None]


# ---- mote::rope_givens ---------------------------------------------------------------------------
@torch.library.custom_op("mote::rope_givens", mutates_args=())
def _rope_givens(qkv: torch.Tensor, inv_freq: Optional[torch.Tensor], theta: Optional[torch.Tensor], n_heads: int,
                 parity: int, pos0: int) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    if not qkv.is_cuda:
        raise RuntimeError("mote::rope_givens needs the HIP library and an MI355X")
    return L.native().rope_givens(qkv, inv_freq, theta, n_heads, parity, pos0, L.stream_of(qkv))


@_rope_givens.register_fake
def _rope_givens_fake(qkv, inv_freq, theta, n_heads, parity, pos0):
    B, T, D3 = qkv.shape
    H = n_heads
    D = D3 // (3 * H)
    mk = lambda: qkv.new_empty((B, T, H, D)).transpose(1, 2)
    return mk(), mk(), mk()


@torch.library.custom_op("mote::rope_givens_bwd", mutates_args=())
def _rope_givens_bwd(dp1: torch.Tensor, dp2: torch.Tensor, dinfo: torch.Tensor, qkv: torch.Tensor,
                     inv_freq: Optional[torch.Tensor], theta: Optional[torch.Tensor], n_heads: int, parity: int,
                     pos0: int, info_only: bool = False) -> Tuple[torch.Tensor, torch.Tensor]:
    """(dqkv [B, T, 3 H dh], dtheta). qkv is the projection output, or with info_only its I~ part
    alone ([B, T, H dh]): the backward reads only the I~ columns (for dtheta)."""
    return L.native().rope_givens_bwd(dp1, dp2, dinfo, qkv, inv_freq, theta, n_heads, parity, pos0, info_only,
                                      L.stream_of(qkv))


@_rope_givens_bwd.register_fake
def _rope_givens_bwd_fake(dp1, dp2, dinfo, qkv, inv_freq, theta, n_heads, parity, pos0, info_only=False):
    B, T, Dx = qkv.shape
    D3 = 3 * Dx if info_only else Dx
    return qkv.new_empty((B, T, D3)), qkv.new_empty((max(n_heads // 2, 1),), dtype=torch.float32)


def _rg_setup(ctx, inputs, output):
    qkv, inv_freq, theta, n_heads, parity, pos0 = inputs
    ctx.save_for_backward(qkv, inv_freq, theta)
    ctx.has_theta = theta is not None
    ctx.n_heads, ctx.parity, ctx.pos0 = n_heads, parity, pos0
    ctx.set_materialize_grads(False)  # the backward takes a missing gradient as zeros


def _rg_backward(ctx, dp1, dp2, dinfo):
    qkv, inv_freq, theta = ctx.saved_tensors
    B, T, D3 = qkv.shape
    H = ctx.n_heads
    D = D3 // (3 * H)
    z = lambda: torch.zeros(B, H, T, D, device=qkv.device, dtype=qkv.dtype)
    dp1 = z() if dp1 is None else dp1
    dp2 = z() if dp2 is None else dp2
    dinfo = z() if dinfo is None else dinfo
    dqkv, dtheta = _rope_givens_bwd(dp1, dp2, dinfo, qkv, inv_freq, theta, H, ctx.parity, ctx.pos0)
    return dqkv, None, (dtheta[: H // 2] if ctx.has_theta else None), None, None, None


_rope_givens.register_autograd(_rg_backward, setup_context=_rg_setup)


def rope_givens(qkv: torch.Tensor, n_heads: int, inv_freq: Optional[torch.Tensor], theta: Optional[torch.Tensor],
                layer_idx: int, pos0: int = 0):
    """[B, T, 3*H*dh] projections -> (p1, p2, I~) as [B, H, T, dh] views: RoPE at positions
    pos0.. on p1/p2 (relation.py:211-214), Givens on I~ (relation.py:215). Differentiable in qkv
    and theta."""
    return _rope_givens(qkv, inv_freq, theta, int(n_heads), int(layer_idx) % 2, int(pos0))


# ---- mote::qkv_rope (fused projection prologue) ----------------------------------------------------
USE_FUSED_PROLOGUE = True   # bf16 activations, head dim 64 / 96 / 128 (with or without QK-Norm): one
                            # launch for the projections, QK-Norm and RoPE / Givens, at every row count;
                            # the unfused path serves everything else. Against hipBLASLt's product plus
                            # the RoPE kernel at width 768 it measured 28.6 / 34.8 us at 4,964 rows
                            # (dh 96) and 365 / 414, 369 / 403, 407 / 406 us at 79,424 rows (dh 96,
                            # 128, 64).


# cos / sin tables of the fused prologue, memoised per (device, stream, inv_freq, T, pos0) the way
# the reference memoises its RoPE tables (at most 32 entries, relation.py:45-58): every layer of a
# step asks for the same positions. Keyed by stream as well, so a table is only reused behind the
# launch that wrote it. A graph capture reuses a table written before the capture began (on the
# capture stream) and pins it, since the graph keeps its address; a table missing at capture time
# is computed inside the graph on every replay and not memoised (its memory belongs to the graph).
_ROPE_TABLES: "dict" = {}          # key -> (inv_freq, its version, table)
_ROPE_TABLES_PINNED: "dict" = {}   # tables a captured graph reads, kept for the life of the process
_ROPE_TABLES_MAX = 32


def _rope_table_ws(T: int, D: int, pos0: int, x: torch.Tensor, inv: Optional[torch.Tensor],
                   cacheable: bool) -> Tuple[torch.Tensor, int, Optional[tuple]]:
    """Workspace for mote_qkv_rope_fwd (mote_qkv_rope_workspace: a 32-bit cos / sin pair per position and
    frequency), whether it already holds the table (table_ready), and what _rope_table_keep takes once a
    launch has filled it (None: not to be kept). `cacheable`: inv is the caller's own frequency tensor
    (not a converted temporary)."""
    n = max(T * (D // 2) * 4 if inv is not None else 0, 16)
    if inv is None or not cacheable:
        return torch.empty(n, device=x.device, dtype=torch.uint8), 0, None
    key = (x.device, L.stream_of(x), inv.data_ptr(), T, pos0, D)
    hit = _ROPE_TABLES.get(key)
    # the entry holds the frequency tensor itself: its memory cannot be recycled for another tensor
    # while the entry lives, and an in-place change of it shows in its version counter
    valid = hit is not None and hit[0] is inv and hit[1] == inv._version
    if torch.cuda.is_current_stream_capturing():
        if valid:
            _ROPE_TABLES_PINNED[hit[2].data_ptr()] = hit[2]
            return hit[2], 1, None
        return torch.empty(n, device=x.device, dtype=torch.uint8), 0, None
    if valid:
        return hit[2], 1, None
    ws = torch.empty(n, device=x.device, dtype=torch.uint8)
    # a call without rows launches nothing, so it leaves the table unwritten
    return ws, 0, (key, inv, inv._version, ws) if x.numel() else None


def _rope_table_keep(key, inv, version, ws):
    """Memoise a table whose launch was accepted: a refused call must not leave an unwritten one behind."""
    if key not in _ROPE_TABLES and len(_ROPE_TABLES) >= _ROPE_TABLES_MAX:
        _ROPE_TABLES.pop(next(iter(_ROPE_TABLES)), None)  # a pinned table stays alive through the pin
    _ROPE_TABLES[key] = (inv, version, ws)


def _qkv_rope_launch(x, w, inv_freq, theta, n_heads, parity, pos0, keep_info, norm_w1, norm_w2, norm_eps, into=None):
    """The prologue's launch for a stacked bf16 weight or a tuple of the three; `into`: (P2, I~) views
    [B, H, T, dh] to write instead of new tensors."""
    if not x.is_cuda:
        raise RuntimeError("mote::qkv_rope needs the HIP library and an MI355X")
    T, K = x.shape[1:]
    D = K // n_heads
    if (norm_w1 is None) != (norm_w2 is None):
        raise ValueError("mote::qkv_rope: QK-Norm needs both gains")
    if norm_w1 is not None and (norm_w1.numel() != D or norm_w2.numel() != D):
        raise ValueError("mote::qkv_rope: QK-Norm gains must have head-dim elements")
    # the kernel reads 16-byte chunks: contiguous copies of operands that are not, or start off a chunk
    x, *ws = (t if t.data_ptr() % 16 == 0 else t.clone()
              for t in (t.contiguous() for t in (x, *(w if isinstance(w, tuple) else (w,)))))
    # the caller's own frequency tensor (not a converted temporary) can key a memoised table
    own = inv_freq is not None and inv_freq.device == x.device and inv_freq.dtype == torch.float32 and inv_freq.is_contiguous()
    inv = inv_freq if inv_freq is None or own else inv_freq.to(device=x.device, dtype=torch.float32).contiguous()
    table, ready, fresh = _rope_table_ws(T, D, pos0, x, inv, own)
    p2, info = into if into is not None else (None, None)
    out = L.native().qkv_rope(x, ws, inv, theta, n_heads, parity, pos0, keep_info, norm_w1, norm_w2, norm_eps, table,
                              bool(ready), p2, info, L.stream_of(x))
    if fresh is not None:
        _rope_table_keep(*fresh)
    return out


@torch.library.custom_op("mote::qkv_rope", mutates_args=())
def _qkv_rope(x: torch.Tensor, w: torch.Tensor, inv_freq: Optional[torch.Tensor], theta: Optional[torch.Tensor],
              n_heads: int, parity: int, pos0: int, keep_info: bool, norm_w1: Optional[torch.Tensor] = None,
              norm_w2: Optional[torch.Tensor] = None, norm_eps: float = 1e-5
              ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    """(p1, p2, I~) as [B, H, T, dh] views of x [w1; w2; wi]^T after (QK-Norm,) RoPE / Givens, and for
    the backward (keep_info): the I~ projections before the rotation ([B, T, H dh]) and, with QK-Norm,
    the p1 | p2 projections before the norm ([B, T, 2 H dh]); empty otherwise."""
    return _qkv_rope_launch(x, w, inv_freq, theta, n_heads, parity, pos0, keep_info, norm_w1, norm_w2, norm_eps)


@_qkv_rope.register_fake
def _qkv_rope_fake(x, w, inv_freq, theta, n_heads, parity, pos0, keep_info, norm_w1=None, norm_w2=None, norm_eps=1e-5):
    B, T, K = x.shape
    D = K // n_heads
    mk = lambda: x.new_empty((B, T, n_heads, D)).transpose(1, 2)
    norm = norm_w1 is not None
    return (mk(), mk(), mk(), (x.new_empty((B, T, K)) if keep_info else x.new_empty(0)),
            (x.new_empty((B, T, 2 * K)) if (keep_info and norm) else x.new_empty(0)))


def _qr_setup(ctx, inputs, output):
    x, w, inv_freq, theta, n_heads, parity, pos0, keep_info, norm_w1, norm_w2, norm_eps = inputs
    ctx.save_for_backward(x, w, inv_freq, theta, output[3], norm_w1, norm_w2, output[4])
    ctx.has_theta = theta is not None
    ctx.norm = norm_w1 is not None
    ctx.keep = keep_info
    ctx.n_heads, ctx.parity, ctx.pos0, ctx.eps = n_heads, parity, pos0, norm_eps
    ctx.set_materialize_grads(False)  # the kept projections have no gradient: no zero tensors for them


@torch.library.custom_op("mote::head_rms_norm_bwd_", mutates_args=("dqkv",))
def _head_norm_bwd_(dqkv: torch.Tensor, qkraw: torch.Tensor, gain1: torch.Tensor, gain2: torch.Tensor, eps: float,
                    n_heads: int) -> Tuple[torch.Tensor, torch.Tensor]:
    """Backward of QK-Norm (relation.py:71-94) on p1 | p2 of the prologue, in place: the first 2 H dh
    columns of dqkv [B, T, 3 H dh] (gradients of the normalised projections) become the gradients
    of the raw projections qkraw [B, T, 2 H dh]; returns the two gains' gradients (fp32). One launch
    of mote_head_rms_norm_bwd (per head row g = dy gain, r = rsqrt(mean(x^2) + eps):
    dx = r g - r^3 x mean(g x), dgain = sum of dy x r)."""
    if not dqkv.is_cuda:
        raise RuntimeError("mote::head_rms_norm_bwd_ needs the HIP library and an MI355X")
    B, T, K3 = dqkv.shape
    K = K3 // 3
    D = K // n_heads
    if B * T == 0:
        z = torch.zeros(D, device=dqkv.device, dtype=torch.float32)
        return z, z.clone()
    if dqkv.stride(2) != 1 or qkraw.stride(2) != 1 or (B > 1 and (dqkv.stride(0) != T * dqkv.stride(1) or
                                                               qkraw.stride(0) != T * qkraw.stride(1))):
        raise ValueError("mote::head_rms_norm_bwd_: token rows must be back to back with unit column stride")
    g1 = gain1.detach().to(device=dqkv.device, dtype=torch.float32).contiguous()
    g2 = gain2.detach().to(device=dqkv.device, dtype=torch.float32).contiguous()
    dg1 = torch.empty(D, device=dqkv.device, dtype=torch.float32)
    dg2 = torch.empty(D, device=dqkv.device, dtype=torch.float32)
    a = L.HeadNormBwdArgs()
    a.dtype, a.rows, a.parts, a.H, a.D, a.eps = L.dtype_code(dqkv), B * T, 2, int(n_heads), D, float(eps)
    a.x, a.x_sr = qkraw.data_ptr(), qkraw.stride(1)
    a.dy, a.dy_sr = dqkv.data_ptr(), dqkv.stride(1)
    a.dx, a.dx_sr = dqkv.data_ptr(), dqkv.stride(1)
    a.gain0, a.gain1, a.dgain0, a.dgain1 = g1.data_ptr(), g2.data_ptr(), dg1.data_ptr(), dg2.data_ptr()
    ws = torch.empty(max(int(L.lib().mote_head_rms_norm_bwd_workspace(a)), 16), device=dqkv.device, dtype=torch.uint8)
    a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
    L.check(L.lib().mote_head_rms_norm_bwd(a, L.stream_of(dqkv)), "mote_head_rms_norm_bwd")
    return dg1, dg2


@_head_norm_bwd_.register_fake
def _head_norm_bwd_fake(dqkv, qkraw, gain1, gain2, eps, n_heads):
    D = dqkv.shape[-1] // 3 // n_heads
    return dqkv.new_empty(D, dtype=torch.float32), dqkv.new_empty(D, dtype=torch.float32)


# ---- mote::wgrad (weight gradient of the projections) -------------------------------------------
USE_WGRAD = True  # bf16 rows, both widths multiples of 64: mote_linear_wgrad; else the GEMM library


@torch.library.custom_op("mote::wgrad", mutates_args=())
def _wgrad(a: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """bf16 dW [N, K] = a^T x for a [M, N], x [M, K], fp32 sums, N and K multiples of 128: mote::linear_wgrad
    under its earlier name."""
    if not a.is_cuda:
        raise RuntimeError("mote::wgrad needs the HIP library and an MI355X")
    if a.dtype != torch.bfloat16 or a.shape[1] % 128 or x.shape[1] % 128:
        raise RuntimeError(f"mote::wgrad: {a.dtype} [M, {a.shape[1]}] and [M, {x.shape[1]}] (bf16, widths multiples of 128)")
    return L.native().linear_wgrad(a, x, a.dtype, L.stream_of(a))


@_wgrad.register_fake
def _wgrad_fake(a, x):
    return a.new_empty((a.shape[1], x.shape[1]))


@torch.library.custom_op("mote::linear_wgrad", mutates_args=())
def _linear_wgrad(a: torch.Tensor, x: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    """dW [N, K] = a^T x in `dtype` (bf16, or the fp32 sums unrounded) for bf16 a [M, N], x [M, K] with N
    and K multiples of 64 (operands whose rows are not apart, unit-stride and 16-byte aligned are copied first)."""
    if not a.is_cuda:
        raise RuntimeError("mote::linear_wgrad needs the HIP library and an MI355X")
    return L.native().linear_wgrad(a, x, dtype, L.stream_of(a))


@_linear_wgrad.register_fake
def _linear_wgrad_fake(a, x, dtype):
    return a.new_empty((a.shape[1], x.shape[1]), dtype=dtype)


def _wgrad_serves(a_dtype: torch.dtype, x_dtype: torch.dtype, N: int, K: int) -> bool:
    """bf16 operands, both widths multiples of 64 (the kernel's smallest tile of dW), any number of rows.
    Widths that are not multiples of 128 are faster here from one row on (576 x 192: 3.6 us here and 4.5 on
    the library, whose reduction runs over the token rows, at 1 row, 6.6 and 13.1 at 1000, 18 and 110 at
    19,856). Multiples of 128 are within a microsecond up to 256 rows and faster here from about 2500 (2304 x 768:
    5.9 and 5.8 us at 1 row, 25.7 and 33.3 at 3000), but slower in between, where two to four splits of the rows
    are summed by a second launch (1000 rows: 24.2 and 15.5, or 24.4 and 19.4 with the cast to fp32; 512 x 512:
    10.6 and 13.1): they stay here, since the library's fp32 gradient would be rounded to bf16 first."""
    return USE_WGRAD and a_dtype == torch.bfloat16 and x_dtype == torch.bfloat16 and N % 64 == 0 and K % 64 == 0


def _transformed() -> bool:
    """Whether a functional transform (vmap, grad, jvp; batched gradients too) or a forward-mode level is
    active: products then stay with torch, since mote_linear_wgrad's function and op have neither rule."""
    return not torch.compiler.is_compiling() and (torch._C._are_functorch_transforms_active()
                                                  or torch.autograd.forward_ad._current_level >= 0)


def weight_grad(a: torch.Tensor, x: torch.Tensor, dtype: Optional[torch.dtype] = None) -> torch.Tensor:
    """a^T x over the token rows of a [..., N] and x [..., K]: the weight gradient of y = x W^T, in a's
    dtype or `dtype` (fp32: the sums unrounded). mote_linear_wgrad for bf16 on the GPU with N, K
    multiples of 64; the GEMM library otherwise."""
    N, K = a.shape[-1], x.shape[-1]
    a2, x2 = a.reshape(-1, N), x.reshape(-1, K)
    dtype = a2.dtype if dtype is None else dtype
    # under create_graph the product has to be differentiable itself
    if a2.is_cuda and _wgrad_serves(a2.dtype, x2.dtype, N, K) and not torch.is_grad_enabled() and not _transformed():
        return _linear_wgrad(a2, x2, dtype)
    return torch.matmul(a2.t(), x2).to(dtype)


class _LinearWgrad(torch.autograd.Function):
    """y = x W^T on the GEMM library for bf16 x and wb, W in bf16 (W itself, or its cast by the caller);
    backward dx = dy W on the library and dW = dy^T x on mote_linear_wgrad, in W's own dtype straight to W
    (the library runs that product with its reduction over the token rows). Only wb is saved: a later
    in-place update of fp32 W leaves the graph usable, as with F.linear of the cast. Under create_graph the
    gradient goes to wb, through the cast."""

    @staticmethod
    def forward(ctx, x, w, wb):
        ctx.save_for_backward(x, wb)
        ctx.w_dtype = w.dtype
        return F.linear(x, wb)

    @staticmethod
    def backward(ctx, dy):
        x, wb = ctx.saved_tensors
        dx = torch.matmul(dy, wb) if ctx.needs_input_grad[0] else None
        if torch.is_grad_enabled():
            return dx, None, (weight_grad(dy, x) if ctx.needs_input_grad[2] else None)
        return dx, (weight_grad(dy, x, ctx.w_dtype) if ctx.needs_input_grad[1] else None), None


def linear_wgrad(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """F.linear(x, w) whose weight gradient runs on mote_linear_wgrad: bf16 x and w on the GPU (or bf16
    autocast, which casts both as F.linear would) with both widths multiples of 64; F.linear otherwise."""
    wb = w
    if torch.is_autocast_enabled() and torch.get_autocast_dtype("cuda") == torch.bfloat16 and x.is_cuda:
        x, wb = x.to(torch.bfloat16), w.to(torch.bfloat16)  # (F.linear itself would not cast fp64)
    # without a backward the function would only cost host time: 2 us with the checks before it, which a short
    # extension feels (311 rows after 4096 cached ones: 126.8 us a call with them, 116.5 so)
    if torch.is_grad_enabled() and x.is_cuda and w.is_cuda and _wgrad_serves(x.dtype, wb.dtype, *w.shape) and not _transformed():
        # fp32 weights take dW from the function itself, others through their cast
        return _LinearWgrad.apply(x, w if w.dtype == torch.float32 else wb, wb)
    return F.linear(x, wb)


def _qr_grads(ctx, dp1, dp2, dinfo, wdtype, need_w):
    """(dx, dW of the stacked weight in wdtype, dtheta, the gains' gradients) of the fused prologue; dx and,
    without need_w, dW are None where nothing takes them (the products are most of this backward)."""
    x, w, inv_freq, theta, iraw, norm_w1, norm_w2, qkraw = ctx.saved_tensors
    if (ctx.has_theta or ctx.norm) and not ctx.keep:
        raise RuntimeError("mote::qkv_rope: the backward needs keep_info=True with theta or QK-Norm")
    B, T, K = x.shape
    H = ctx.n_heads
    D = K // H
    z = lambda: torch.zeros(B, H, T, D, device=x.device, dtype=x.dtype)
    dp1 = z() if dp1 is None else dp1
    dp2 = z() if dp2 is None else dp2
    dinfo = z() if dinfo is None else dinfo
    src = iraw if ctx.keep else x.new_empty(B, T, K)  # read only for dtheta
    dqkv, dtheta = _rope_givens_bwd(dp1, dp2, dinfo, src, inv_freq, theta, H, ctx.parity, ctx.pos0, True)
    dn1 = dn2 = None
    if ctx.norm:  # gradients of the normalised p1 / p2 back through QK-Norm, in place in dqkv
        dn1, dn2 = _head_norm_bwd_(dqkv, qkraw, norm_w1, norm_w2, ctx.eps, H)
        dn1, dn2 = dn1.to(norm_w1.dtype), dn2.to(norm_w2.dtype)
    dx = torch.matmul(dqkv, w) if ctx.needs_input_grad[0] else None   # [B, T, 3K] x [3K, K]
    dw = weight_grad(dqkv, x, wdtype) if need_w else None             # [3K, K]
    return dx, dw, (dtheta[: H // 2] if ctx.has_theta else None), dn1, dn2


def _qr_backward(ctx, dp1, dp2, dinfo, _diraw, _dqkraw):
    dx, dw, dtheta, dn1, dn2 = _qr_grads(ctx, dp1, dp2, dinfo, None, ctx.needs_input_grad[1])
    return dx, dw, None, dtheta, None, None, None, None, dn1, dn2, None


_qkv_rope.register_autograd(_qr_backward, setup_context=_qr_setup)


# ---- the prologue from the layer's own three weights -----------------------------------------------
def _packed(x: torch.Tensor, w1: torch.Tensor, w2: torch.Tensor, wi: torch.Tensor) -> torch.Tensor:
    """The bf16 stack [w1; w2; wi]: fp32 weights rounded and stacked in one launch, others by torch."""
    if not w1.shape == w2.shape == wi.shape or any(t.device != x.device for t in (w1, w2, wi)):
        raise RuntimeError("mote::qkv_rope_master: the three weights must be of one shape, on x's device")
    if not all(t.dtype == torch.float32 for t in (w1, w2, wi)) or w1.numel() % 8:
        return torch.cat([w1, w2, wi], dim=0).to(torch.bfloat16)
    ws = [t if t.data_ptr() % 16 == 0 else t.clone() for t in (w1.contiguous(), w2.contiguous(), wi.contiguous())]
    N, K = w1.shape
    w = torch.empty(3 * N, K, device=x.device, dtype=torch.bfloat16)
    a = L.PackWeightsArgs()
    a.n, a.out = N * K, w.data_ptr()
    a.w0, a.w1, a.w2 = (t.data_ptr() for t in ws)
    L.check(L.lib().mote_pack_weights(a, L.stream_of(x)), "mote_pack_weights")
    return w


def _bf16_parts(x, w1, w2, wi, keep: bool):
    """(the three bf16 weights, their stack when it was made): bf16 weights are read where they are
    unless the backward needs the stack (its dx is one product with it)."""
    if keep or any(t.dtype != torch.bfloat16 for t in (w1, w2, wi)):
        w = _packed(x, w1, w2, wi)
        return tuple(w.chunk(3)), w
    return (w1, w2, wi), x.new_empty(0)


@torch.library.custom_op("mote::qkv_rope_master", mutates_args=())
def _qkv_rope_master(x: torch.Tensor, w1: torch.Tensor, w2: torch.Tensor, wi: torch.Tensor,
                     inv_freq: Optional[torch.Tensor], theta: Optional[torch.Tensor], n_heads: int, parity: int,
                     pos0: int, keep_info: bool, train: bool, norm_w1: Optional[torch.Tensor] = None,
                     norm_w2: Optional[torch.Tensor] = None, norm_eps: float = 1e-5
                     ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    """mote::qkv_rope from the layer's weights [H dh, H dh] (fp32 or bf16); with `train` the sixth output is
    their bf16 stack, kept for the backward's dx (empty otherwise). dh 48 is served too (no QK-Norm)."""
    if not x.is_cuda:
        raise RuntimeError("mote::qkv_rope_master needs the HIP library and an MI355X")
    ws, stack = _bf16_parts(x, w1, w2, wi, train)
    return (*_qkv_rope_launch(x, ws, inv_freq, theta, n_heads, parity, pos0, keep_info, norm_w1, norm_w2, norm_eps), stack)


@_qkv_rope_master.register_fake
def _qkv_rope_master_fake(x, w1, w2, wi, inv_freq, theta, n_heads, parity, pos0, keep_info, train, norm_w1=None,
                          norm_w2=None, norm_eps=1e-5):
    w = x.new_empty((3 * w1.shape[0], w1.shape[1]))
    bf16 = all(t.dtype == torch.bfloat16 for t in (w1, w2, wi))
    return (*_qkv_rope_fake(x, w, inv_freq, theta, n_heads, parity, pos0, keep_info, norm_w1, norm_w2, norm_eps),
            x.new_empty(0) if bf16 and not train else w)


def _qrm_setup(ctx, inputs, output):
    x, w1, _w2, _wi, inv_freq, theta, n_heads, parity, pos0, keep_info, train, *norm = inputs
    _qr_setup(ctx, (x, output[5], inv_freq, theta, n_heads, parity, pos0, keep_info, *norm), output)
    ctx.w_dtypes = tuple(t.dtype for t in inputs[1:4])
    ctx.train = train


def _qrm_backward(ctx, dp1, dp2, dinfo, _diraw, _dqkraw, _dw):
    if not ctx.train:
        raise RuntimeError("mote::qkv_rope_master: the backward needs train=True")
    wdtype = torch.float32 if torch.float32 in ctx.w_dtypes else None
    dx, dw, dtheta, dn1, dn2 = _qr_grads(ctx, dp1, dp2, dinfo, wdtype, any(ctx.needs_input_grad[1:4]))
    dws = (None,) * 3 if dw is None else (d.to(t) for d, t in zip(dw.chunk(3), ctx.w_dtypes))
    return (dx, *dws, None, dtheta, None, None, None, None, None, dn1, dn2, None)


_qkv_rope_master.register_autograd(_qrm_backward, setup_context=_qrm_setup)


@torch.library.custom_op("mote::qkv_rope_into", mutates_args=("p2", "info"))
def _qkv_rope_into(x: torch.Tensor, w1: torch.Tensor, w2: torch.Tensor, wi: torch.Tensor, inv_freq: Optional[torch.Tensor],
                   theta: Optional[torch.Tensor], n_heads: int, parity: int, pos0: int, p2: torch.Tensor,
                   info: torch.Tensor, norm_w1: Optional[torch.Tensor] = None, norm_w2: Optional[torch.Tensor] = None,
                   norm_eps: float = 1e-5) -> torch.Tensor:
    """mote::qkv_rope_master without a backward, P2 and I~ written into the given bf16 [B, H, T, dh] views
    (a cache's new rows); returns p1."""
    if not x.is_cuda:
        raise RuntimeError("mote::qkv_rope_into needs the HIP library and an MI355X")
    ws, _ = _bf16_parts(x, w1, w2, wi, False)
    return _qkv_rope_launch(x, ws, inv_freq, theta, n_heads, parity, pos0, False, norm_w1, norm_w2, norm_eps, (p2, info))[0]


@_qkv_rope_into.register_fake
def _qkv_rope_into_fake(x, w1, w2, wi, inv_freq, theta, n_heads, parity, pos0, p2, info, norm_w1=None, norm_w2=None,
                        norm_eps=1e-5):
    B, T, K = x.shape
    return x.new_empty((B, T, n_heads, K // n_heads)).transpose(1, 2)


def qkv_rope(x: torch.Tensor, w: torch.Tensor, n_heads: int, inv_freq: Optional[torch.Tensor],
             theta: Optional[torch.Tensor], layer_idx: int, pos0: int = 0,
             norm: Optional[Tuple[torch.Tensor, torch.Tensor, float]] = None):
    """The fused prologue: bf16 x [B, T, H dh] and w = [w1; w2; wi] [3 H dh, H dh] -> (p1, p2, I~),
    the same as rope_givens(F.linear(x, w), ...) (relation.py:199-215); `norm` = (p1 gain, p2 gain,
    eps) applies QK-Norm to p1 / p2 first (relation.py:208-210). Differentiable in x, w, theta and
    the gains. w may also be the tuple of the three weights, fp32 or bf16 (mote::qkv_rope_master)."""
    n1, n2, eps = norm if norm is not None else (None, None, 1e-5)
    train = torch.is_grad_enabled()
    keep = train and (theta is not None or norm is not None)
    head = (inv_freq, theta, int(n_heads), int(layer_idx) % 2, int(pos0), keep)
    if isinstance(w, tuple):
        return _qkv_rope_master(x, *w, *head, train, n1, n2, float(eps))[:3]
    return _qkv_rope(x, w, *head, n1, n2, float(eps))[:3]


# ---- mote::out_gate (the output gate of _out) ----------------------------------------------------
@torch.library.custom_op("mote::out_gate", mutates_args=())
def _out_gate(x: torch.Tensor, wg: torch.Tensor, y: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """bf16 (z, s): z = y * sigmoid(x wg^T) and s = the sigmoid, [B, T, D] (relation.py:179-181)."""
    if not x.is_cuda:
        raise RuntimeError("mote::out_gate needs the HIP library and an MI355X")
    B, T, D = x.shape
    x2 = x.reshape(B * T, D).contiguous()
    y2 = y.reshape(B * T, D).contiguous()
    wc = wg.contiguous()
    z = torch.empty(B, T, D, device=x.device, dtype=x.dtype)
    s = torch.empty(B, T, D, device=x.device, dtype=x.dtype)
    a = L.GateProductArgs()
    a.B, a.T, a.D = 1, B * T, D
    a.x, a.x_sr = x2.data_ptr(), x2.stride(0)
    a.w, a.w_sr = wc.data_ptr(), wc.stride(0)
    a.y, a.y_sr = y2.data_ptr(), y2.stride(0)
    a.z, a.s, a.z_sr = z.data_ptr(), s.data_ptr(), D
    L.check(L.lib().mote_gate_product(a, L.stream_of(x)), "mote_gate_product")
    return z, s


@_out_gate.register_fake
def _out_gate_fake(x, wg, y):
    return x.new_empty(x.shape), x.new_empty(x.shape)


def _og_setup(ctx, inputs, output):
    x, wg, y = inputs
    ctx.save_for_backward(x, wg, y, output[1])
    ctx.set_materialize_grads(False)  # s has no gradient: no zero tensor for it


@torch.library.custom_op("mote::gate_bwd", mutates_args=())
def _gate_bwd(dz: torch.Tensor, y: torch.Tensor, s: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """bf16 (dy, dg) = (dz s, dz y s (1 - s)) of equally shaped bf16 tensors whose last axis is a multiple
    of 8, contiguous results."""
    if not dz.shape == y.shape == s.shape or any(t.dtype != torch.bfloat16 or t.device != dz.device for t in (dz, y, s)):
        raise RuntimeError("mote::gate_bwd takes bf16 dz, y and s of one shape on one device")
    if not dz.is_cuda:
        raise RuntimeError("mote::gate_bwd needs the HIP library and an MI355X")
    # the kernel walks flat memory in 16-byte chunks: copies of views in another order or off a chunk
    dz, y, s = (t if t.data_ptr() % 16 == 0 else t.clone() for t in (t.contiguous() for t in (dz, y, s)))
    dy, dg = torch.empty_like(y), torch.empty_like(y)
    a = L.GateBwdArgs()
    a.dtype, a.n = L.dtype_code(dz), dz.numel()
    a.dz, a.y, a.s, a.dy, a.dg = dz.data_ptr(), y.data_ptr(), s.data_ptr(), dy.data_ptr(), dg.data_ptr()
    L.check(L.lib().mote_gate_bwd(a, L.stream_of(dz)), "mote_gate_bwd")
    return dy, dg


@_gate_bwd.register_fake
def _gate_bwd_fake(dz, y, s):
    return dz.new_empty(dz.shape), dz.new_empty(dz.shape)


def _og_backward(ctx, dz, _ds):
    """z = y s, s = sigmoid(g), g = x wg^T: dy = dz s, dg = dz y s (1 - s), dx = dg wg, dwg = dg^T x."""
    x, wg, y, s = ctx.saved_tensors
    dz = torch.zeros_like(y) if dz is None else dz
    if torch.is_grad_enabled():  # create_graph: as torch ops, which can be differentiated again
        dzf, sf = dz.float(), s.float()
        dy, dg = (dzf * sf).to(y.dtype), (dzf * y.float() * sf * (1.0 - sf)).to(x.dtype)
    else:
        dy, dg = _gate_bwd(dz, y, s)
    dx = torch.matmul(dg, wg)
    dwg = weight_grad(dg, x)
    return dx, dwg, dy


_out_gate.register_autograd(_og_backward, setup_context=_og_setup)
USE_FUSED_GATE = True  # bf16 and a width that is a multiple of 128: the gate product kernel


def out_gate(x: torch.Tensor, wg: torch.Tensor, y: torch.Tensor) -> torch.Tensor:
    """y * sigmoid(x wg^T) in one launch (bf16 x, wg, y [B, T, D]); differentiable in all three."""
    return _out_gate(x, wg, y)[0]


class HeadRMSNorm(nn.Module):
    """QK-Norm over the head dim with a learnable gain (relation.py:71-94); fp32 math."""

    def __init__(self, dim: int, eps: float = 1e-5, device=None, dtype=None):
        super().__init__()
        self.eps = eps
        self.weight = nn.Parameter(torch.ones(dim, device=device, dtype=dtype))

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        xf = x.float()
        y = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + self.eps)
        return (y * self.weight.float()).to(x.dtype)


class FullRelation(nn.Module):
    def __init__(self, d_model: int, n_heads: int, layer_idx: int, tau_s: float = 2.0, lambda_init: float = 0.5,
                 rope_theta: float = 10000.0, givens: bool = True, qk_norm: bool = False, out_gate: bool = False,
                 rope: bool = True, device=None, dtype=None):
        super().__init__()
        assert d_model % n_heads == 0, "d_model must be divisible by n_heads"
        assert n_heads % 2 == 0, "Givens pairing needs an even number of heads"
        fk = {"device": device, "dtype": dtype}
        self.d_model, self.n_heads, self.d_head = d_model, n_heads, d_model // n_heads
        assert self.d_head % 2 == 0, "head dim must be even for RoPE"
        self.layer_idx = layer_idx
        self.tau_s = tau_s
        self.rope_theta = rope_theta
        self.use_givens = givens
        self.telemetry: Optional[dict] = None
        self.qk_norm = qk_norm
        if qk_norm:
            self.p1_norm = HeadRMSNorm(self.d_head, **fk)
            self.p2_norm = HeadRMSNorm(self.d_head, **fk)
        self.w1 = nn.Linear(d_model, d_model, bias=False, **fk)
        self.w2 = nn.Linear(d_model, d_model, bias=False, **fk)
        self.wi = nn.Linear(d_model, d_model, bias=False, **fk)
        self.wo = nn.Linear(d_model, d_model, bias=False, **fk)
        self.out_gate = out_gate
        if out_gate:
            self.wg = nn.Linear(d_model, d_model, bias=False, **fk)
        self.use_rope = rope
        self.lam = nn.Parameter(torch.tensor(float(lambda_init), dtype=torch.float32, device=device))
        self.lam._no_weight_decay = True
        if givens:
            self.theta = nn.Parameter(torch.zeros(n_heads // 2, dtype=torch.float32, device=device))
            self.theta._no_weight_decay = True
            if layer_idx % 2 == 0:
                a = torch.arange(0, n_heads, 2)
                b = torch.arange(1, n_heads, 2)
            else:
                a = torch.arange(1, n_heads, 2)
                b = (torch.arange(2, n_heads + 1, 2)) % n_heads
            self.register_buffer("pair_a", a, persistent=False)
            self.register_buffer("pair_b", b, persistent=False)
        self.register_buffer("inv_freq", rope_inv_freq(self.d_head, rope_theta, device), persistent=False)

    def _apply(self, fn, recurse=True):
        # `.to(dtype)`, `.half()`, `.bfloat16()` would round the RoPE frequencies (an angle error of
        # radians at positions in the thousands); the reference recomputes them in fp32 on every call
        # (relation.py:39). Keep the buffer fp32 on whatever device the parameters moved to.
        super()._apply(fn, recurse)
        self._buffers["inv_freq"] = rope_inv_freq(self.d_head, self.rope_theta, self.lam.device)
        return self

    def _givens(self, info: torch.Tensor) -> torch.Tensor:
        """Givens mixing of head pairs for callers that rotate rows themselves (relation.py:160-174,
        graph.py:165): info [B, H, T, dh]; pairs (0,1),(2,3),... on even layers, (1,2),...,(H-1,0) on
        odd ones; (a, b) -> (c a - s b, s a + c b) with c, s = cos / sin(theta) in info's dtype. The
        module's forward applies the same rotation inside its HIP prologue kernels."""
        if not self.use_givens:
            return info
        H = info.shape[1]
        c = torch.cos(self.theta).to(info.dtype)[None, :, None, None]
        s = torch.sin(self.theta).to(info.dtype)[None, :, None, None]
        first = torch.arange(self.layer_idx % 2, H, 2, device=info.device)
        second = (first + 1) % H
        ia, ib = info.index_select(1, first), info.index_select(1, second)
        out = torch.empty_like(info)
        out.index_copy_(1, first, c * ia - s * ib)
        out.index_copy_(1, second, s * ia + c * ib)
        return out

    # ------------------------------------------------------------------------------------------
    def _check_width(self, x: torch.Tensor) -> None:
        """The prologue's kernels take the head dim from x, so its width has to be the layer's."""
        if x.dim() != 3 or x.shape[-1] != self.d_model:
            raise RuntimeError(f"FullRelation takes x [B, T, {self.d_model}], got {list(x.shape)}")

    def _fused_prologue(self, bf16: bool) -> bool:
        """Whether the one-launch prologue serves this layer: bf16 activations, a width of whole 64-column
        stages, head dim 64 / 96 / 128, or 48 without QK-Norm (the 192-wide layer, 19,856 rows: product
        and RoPE kernel 20.7 + 13.7 us apart, 20.0 fused)."""
        if not USE_FUSED_PROLOGUE or not bf16:
            return False
        if self.d_head == 48:
            return self.d_model % 64 == 0 and not self.qk_norm
        return self.d_head in (64, 96, 128) and self.d_model % 32 == 0

    def heads(self, x: torch.Tensor, S: int):
        """Projections -> (QK-Norm) -> RoPE / Givens: (p1, p2, I~) as [B, H, T, dh] views."""
        self._check_width(x)
        B, T, D = x.shape
        H, dh = self.n_heads, self.d_head
        ws = (self.w1.weight, self.w2.weight, self.wi.weight)
        inv = self.inv_freq if self.use_rope else None
        theta = self.theta if self.use_givens else None
        bf16 = x.dtype == torch.bfloat16 or (torch.is_autocast_enabled() and
                                             torch.get_autocast_dtype("cuda") == torch.bfloat16)
        if self._fused_prologue(bf16):
            norm = (self.p1_norm.weight, self.p2_norm.weight, self.p1_norm.eps) if self.qk_norm else None
            # fp32 master weights: stacked and rounded in one launch, their gradients written in fp32
            # (three launches fewer than a concatenation, a cast and the cast of dW back); bf16
            # weights: read where they are when there is no backward
            return qkv_rope(x.to(torch.bfloat16), ws, H, inv, theta, self.layer_idx, S, norm)
        qkv = linear_wgrad(x, torch.cat(ws, dim=0))
        if self.qk_norm:
            q, k, v = qkv.split(D, dim=-1)
            q = self.p1_norm(q.reshape(B, T, H, dh)).reshape(B, T, D)
            k = self.p2_norm(k.reshape(B, T, H, dh)).reshape(B, T, D)
            qkv = torch.cat([q, k, v], dim=-1)
        return rope_givens(qkv, H, inv, theta, self.layer_idx, S)

    def _heads_into(self, x: torch.Tensor, S: int, cache: ArenaLayer) -> Optional[torch.Tensor]:
        """heads() with P2 and I~ written straight into the arena's rows [S, S + T) by the prologue's launch
        (two copies fewer): p1, or None where that does not apply (a backward is wanted, another dtype or
        batch, a width the fused prologue does not serve, a traced call)."""
        self._check_width(x)
        B, T, _ = x.shape
        arena = cache.arena
        bf16 = x.dtype == torch.bfloat16 or (torch.is_autocast_enabled() and
                                             torch.get_autocast_dtype("cuda") == torch.bfloat16)
        if (torch.is_grad_enabled() or torch.compiler.is_compiling() or not self._fused_prologue(bf16) or T == 0
                or arena.dtype != torch.bfloat16 or arena.batch != B or arena.n_heads != self.n_heads
                or arena.d_head != self.d_head or arena.store.device != x.device or S + T > arena.capacity):
            return None
        p2, info = (t[:, :, S: S + T] for t in (arena.p2(cache.layer), arena.info(cache.layer)))
        if any(t.data_ptr() % 16 or t.stride(3) != 1 or any(st % 8 for st in t.stride()[:3]) for t in (p2, info)):
            return None
        n1, n2, eps = (self.p1_norm.weight, self.p2_norm.weight, self.p1_norm.eps) if self.qk_norm else (None, None, 1e-5)
        return _qkv_rope_into(x.to(torch.bfloat16), self.w1.weight, self.w2.weight, self.wi.weight,
                              self.inv_freq if self.use_rope else None, self.theta if self.use_givens else None,
                              self.n_heads, self.layer_idx % 2, S, p2, info, n1, n2, float(eps))

    def _out(self, y: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
        """[B, H, T, dh] -> [B, T, D] -> optional output gate -> wo (relation.py:176-182)."""
        B, H, T, dh = y.shape
        y = y.transpose(1, 2).reshape(B, T, H * dh)
        if self.out_gate:
            bf16 = y.dtype == torch.bfloat16 and (x.dtype == torch.bfloat16 or torch.is_autocast_enabled())
            if USE_FUSED_GATE and bf16 and y.is_cuda and (H * dh) % 128 == 0:
                y = out_gate(x.to(torch.bfloat16), self.wg.weight.to(torch.bfloat16), y)
            else:
                y = y * torch.sigmoid(self.wg(x))
        return linear_wgrad(y, self.wo.weight)

    def forward(self, x: torch.Tensor, cache: Optional[RelationCache] = None, return_cache: bool = False,
                return_gates: bool = False):
        """x: [B, T, D]. With a cache, x holds the new T positions appended after S cached ones.
        Returns out [B, T, D], then (in this order, when asked) the updated cache and the exchange
        mass g [B, H, T] (relation.py:184-268)."""
        if not USE_FLASH:
            raise RuntimeError("mote_amd.relation has only the HIP path (USE_FLASH = False is not supported)")
        self._check_width(x)
        if not x.is_cuda:
            raise RuntimeError("FullRelation needs the HIP library and an MI355X (x is on the CPU)")
        B, T, D = x.shape
        arena = isinstance(cache, ArenaLayer)
        S = cache.n if arena else (0 if cache is None else cache[0].shape[2])
        p1 = self._heads_into(x, S, cache) if arena else None
        if p1 is None:
            p1, p2, info = self.heads(x, S)
            if arena:
                cache.write(p2, info)
        if arena:
            p2_all, info_all = cache.views(S + T)
        elif cache is not None:
            p2_all = torch.cat([cache[0], p2], dim=2)
            info_all = torch.cat([cache[1], info], dim=2)
        else:
            p2_all, info_all = p2, info
        new_cache = cache if arena else (p2_all, info_all)
        if p2_all.dtype != p1.dtype:  # an arena kept in another dtype than the activations
            p1 = p1.to(p2_all.dtype)
        y, g = flash_relation(p1, p2_all, info_all, self.lam, self.tau_s, q_start=S)
        if y.dtype != x.dtype and not torch.is_autocast_enabled():
            y = y.to(x.dtype)  # an arena in a narrower dtype than an fp32 module
        out = self._out(y, x)
        extras = []
        if return_cache:
            extras.append(new_cache)
        if self.telemetry is not None:
            self.telemetry["exchange_mass"] = float(g[0, :, -1].detach().mean())
        if return_gates:
            extras.append(g)
        return (out, *extras) if extras else out
