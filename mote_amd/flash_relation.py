"""FlashRelation on MI355X — the fused Relation core behind Mote's call signatures.

Mirrors mote/model/flash_relation.py: the same public function `flash_relation`, the same
`torch.library` custom ops `mote::relation_fwd` / `mote::relation_bwd` (schemas of
flash_relation.py:620-641, with fake implementations and autograd, so `torch.compile(fullgraph=True)`
traces through them), the same `DETERMINISTIC` switch (MOTE_DETERMINISTIC_RELATION,
flash_relation.py:51). The kernels are the hand-written HIP ones in libmote_relation.so; there is no
other implementation behind these names, and calling them without the library or without a GPU
raises.

Additions with no counterpart in the reference:
* `flash_relation_varlen` / `mote::relation_fwd_varlen`: packed sequences with `cu_seqlens` (the
  reference pads to a bucket instead, mote/model/dc.py:192-218).
* Output layout: Y is allocated token-major ([B, T, H, D] memory, returned as the [B, H, T, D]
  view), so `FullRelation._out`'s transpose to [B, T, H*D] is free.
"""

from __future__ import annotations

import math
import os
from typing import Tuple

import torch
import torch.nn.functional as F

from . import _lib as L

DETERMINISTIC = os.environ.get("MOTE_DETERMINISTIC_RELATION", "0") == "1"  # atomic-free backward


def _hip_ready() -> bool:
    return L.available() and torch.cuda.is_available()


HAS_HIP = _hip_ready()
HAS_TRITON = HAS_HIP  # the name the reference's callers test (relation.py:29, 228); no Triton here


def _check_device(*ts):
    for t in ts:
        if not t.is_cuda:
            raise RuntimeError("flash_relation needs the HIP library and an MI355X: tensors are on the CPU")


def _token_major(B, H, T, D, like: torch.Tensor, dtype) -> torch.Tensor:
    """Empty [B, H, T, D] view over [B, T, H, D] memory."""
    return torch.empty(B, T, H, D, device=like.device, dtype=dtype).transpose(1, 2)


def _launch_fwd(p1, p2, info, lam, tau_s: float, q_start: int):
    B, H, TQ, D = p1.shape
    TK = p2.shape[2]
    if TK != q_start + TQ:
        raise ValueError("keys must cover exactly the cached prefix plus the new positions")
    if p2.dtype != p1.dtype or info.dtype != p1.dtype:
        raise TypeError("p1, p2 and info must share a dtype")
    _check_device(p1, p2, info, lam)
    return L.native().relation_fwd(p1, p2, info, lam, float(tau_s), q_start, None, 0, L.stream_of(p1))


def _launch_bwd(p1, p2, info, ibar, lse, g, dy, tau_s: float, q_start: int, deterministic: bool):
    _check_device(p1, p2, info, dy)
    return L.native().relation_bwd(p1, p2, info, ibar, lse, g, dy, float(tau_s), q_start, bool(deterministic),
                                   L.stream_of(p1))


@torch.library.custom_op("mote::relation_fwd", mutates_args=())
def _relation_fwd(p1: torch.Tensor, p2: torch.Tensor, info: torch.Tensor, lam: torch.Tensor, tau_s: float,
                  q_start: int) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    return _launch_fwd(p1, p2, info, lam, tau_s, q_start)


@_relation_fwd.register_fake
def _relation_fwd_fake(p1, p2, info, lam, tau_s, q_start):
    B, H, TQ, D = p1.shape
    return (
        p1.new_empty((B, TQ, H, D), dtype=info.dtype).transpose(1, 2),
        p1.new_empty((B, H, TQ), dtype=torch.float32),
        p1.new_empty((B, H, TQ, D), dtype=torch.float32),
        p1.new_empty((B, H, TQ), dtype=torch.float32),
    )


@torch.library.custom_op("mote::relation_bwd", mutates_args=())
def _relation_bwd(p1: torch.Tensor, p2: torch.Tensor, info: torch.Tensor, ibar: torch.Tensor, lse: torch.Tensor,
                  g: torch.Tensor, dy: torch.Tensor, tau_s: float,
                  q_start: int) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    return _launch_bwd(p1, p2, info, ibar, lse, g, dy, tau_s, q_start, DETERMINISTIC)


@_relation_bwd.register_fake
def _relation_bwd_fake(p1, p2, info, ibar, lse, g, dy, tau_s, q_start):
    B, H, TQ, D = p1.shape
    TK = p2.shape[2]
    return (
        p1.new_empty((B, TQ, H, D)).transpose(1, 2),
        p1.new_empty((B, TK, H, D), dtype=p2.dtype).transpose(1, 2),
        p1.new_empty((B, TK, H, D), dtype=info.dtype).transpose(1, 2),
        p1.new_empty((), dtype=torch.float32),
    )


def _setup_context(ctx, inputs, output):
    p1, p2, info, lam, tau_s, q_start = inputs
    y, g, ibar, lse = output
    ctx.save_for_backward(p1, p2, info, ibar, lse, g)
    ctx.tau_s, ctx.q_start = tau_s, q_start
    # no zero tensors for the outputs without a gradient (g, ibar, lse: the last as large as Y in fp32)
    ctx.set_materialize_grads(False)


def _backward(ctx, dy, _dg, _dibar, _dlse):
    p1, p2, info, ibar, lse, g = ctx.saved_tensors
    if dy is None:  # only g, ibar or lse was differentiated: no gradient flows through them
        dy = torch.zeros(p1.shape, device=p1.device, dtype=p1.dtype)
    dp1, dp2, dinfo, dlam = _relation_bwd(p1, p2, info, ibar, lse, g, dy, ctx.tau_s, ctx.q_start)
    return dp1, dp2, dinfo, dlam, None, None


_relation_fwd.register_autograd(_backward, setup_context=_setup_context)


def flash_relation(p1: torch.Tensor, p2: torch.Tensor, info: torch.Tensor, lam: torch.Tensor, tau_s: float = 2.0,
                   q_start: int = 0) -> Tuple[torch.Tensor, torch.Tensor]:
    """Fused Full Relation (mote/model/flash_relation.py:657-663).

    p1 [B,H,T,D] (RoPE applied); p2/info [B,H,q_start+T,D] (RoPE / Givens applied; any row/head
    strides, e.g. decode-arena views). Returns (Y [B,H,T,D] in info's dtype, g [B,H,T] fp32 exchange
    mass; no gradient flows through g)."""
    if not HAS_HIP or not p1.is_cuda:
        raise RuntimeError("flash_relation needs the HIP library (libmote_relation.so) and an MI355X")
    y, g, _ibar, _lse = _relation_fwd(p1, p2, info, lam, float(tau_s), int(q_start))
    return y, g.detach()


def relation_reference(p1: torch.Tensor, p2: torch.Tensor, info: torch.Tensor, lam: torch.Tensor, tau_s: float = 2.0,
                       q_start: int = 0) -> Tuple[torch.Tensor, torch.Tensor]:
    """The same function materialized in fp32, for callers' tests (flash_relation.py:666-682):
    scores U = p1 P2^T / sqrt(D) over every (query, key) pair, Self sigmoid(U_ii / tau_s) on the
    diagonal, SiLU(U_ij) - lam ln(i + 1) over the strict past, softmax, Y = F I~, g = the past's
    share of F. O(TQ * TK) memory; nothing in this package calls it."""
    TQ, D = p1.shape[-2], p1.shape[-1]
    TK = p2.shape[-2]
    q, k, v = p1.float(), p2.float(), info.float()
    u = torch.matmul(q, k.transpose(-1, -2)) / math.sqrt(D)
    pos = torch.arange(q_start, q_start + TQ, device=q.device).unsqueeze(-1)  # absolute query index
    key = torch.arange(TK, device=q.device).unsqueeze(0)
    count = torch.log((pos + 1).float())
    scores = torch.where(key == pos, torch.sigmoid(u / tau_s), F.silu(u) - lam.float() * count)
    scores = scores.masked_fill(key > pos, float("-inf"))
    flow = torch.softmax(scores, dim=-1)
    return torch.matmul(flow, v), (flow * (key < pos)).sum(-1)


# ---- varlen prefill (forward only) -------------------------------------------------------------
@torch.library.custom_op("mote::relation_fwd_varlen", mutates_args=())
def _relation_fwd_varlen(p1: torch.Tensor, p2: torch.Tensor, info: torch.Tensor, lam: torch.Tensor,
                         cu_seqlens: torch.Tensor, max_seqlen: int,
                         tau_s: float) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    _check_device(p1, p2, info, lam, cu_seqlens)
    cu = cu_seqlens.to(torch.int32).contiguous()
    y, g, ibar, lse = L.native().relation_fwd(p1.unsqueeze(0), p2.unsqueeze(0), info.unsqueeze(0), lam, float(tau_s), 0, cu,
                                              int(max_seqlen), L.stream_of(p1))
    return y[0], g[0], ibar[0], lse[0]


@_relation_fwd_varlen.register_fake
def _relation_fwd_varlen_fake(p1, p2, info, lam, cu_seqlens, max_seqlen, tau_s):
    H, total, D = p1.shape
    return (
        p1.new_empty((total, H, D), dtype=info.dtype).permute(1, 0, 2),
        p1.new_empty((H, total), dtype=torch.float32),
        p1.new_empty((H, total, D), dtype=torch.float32),
        p1.new_empty((H, total), dtype=torch.float32),
    )


def flash_relation_varlen(p1: torch.Tensor, p2: torch.Tensor, info: torch.Tensor, lam: torch.Tensor,
                          cu_seqlens: torch.Tensor, max_seqlen: int, tau_s: float = 2.0):
    """Relation prefill over packed sequences: p1/p2/info are [H, total, D] views (any row/head
    strides, e.g. a [total, H, D] projection output permuted); sequence b owns rows
    [cu_seqlens[b], cu_seqlens[b+1]) and starts at position 0. Returns (Y [H, total, D], g [H, total]).
    Equals `flash_relation` applied to each sequence alone."""
    if not HAS_HIP or not p1.is_cuda:
        raise RuntimeError("flash_relation_varlen needs the HIP library (libmote_relation.so) and an MI355X")
    y, g, _ibar, _lse = _relation_fwd_varlen(p1, p2, info, lam, cu_seqlens, int(max_seqlen), float(tau_s))
    return y, g
