"""The Relation backward's two workspace sizes: the full one (with the stored dU, where a path stores it) and the
least, with which padded bf16 head dims and fp32 run without it, as a step near the card's memory needs."""

from __future__ import annotations

import pytest
import torch

from conftest import rel_err
from mote_amd import _lib as L
from oracle import relation as O


def _args(dtype, B, H, TQ, D, S=0, row=None):
    a = L.BwdArgs()
    a.dtype, a.B, a.H, a.TQ, a.TK, a.D, a.q_start, a.tau_s = dtype, B, H, TQ, S + TQ, D, S, 2.0
    for n in ("p1", "p2", "info"):
        setattr(a, n, L.View(1 << 20, H * TQ * D, D, row or H * D))
    return a


def _sizes(a):
    return L.lib().mote_relation_bwd_workspace(a), L.lib().mote_relation_bwd_workspace_min(a)


def test_least_workspace_is_of_the_order_of_the_operands():
    # at most four copies of 64-wide rows, the fp32 dP1 and a few row vectors; dU is many times that
    for dtype, B, T, D, es in ((L.MOTE_BF16, 16, 8000, 48, 2), (L.MOTE_F32, 4, 3000, 64, 4)):
        full, least = _sizes(_args(dtype, B, 4, T, D))
        assert least < B * 4 * T * 64 * (4 * es + 4 + 1) < full, (dtype, full, least)


@pytest.mark.parametrize("a", [
    _args(L.MOTE_BF16, 2, 4, 1000, 64),                    # unpadded: the tile kernels are the only path
    _args(L.MOTE_BF16, 1, 4, 60000, 48),                   # beyond 8 GiB of dU
    _args(L.MOTE_F32, 1, 8, 20000, 64),                    # beyond 2 GiB
    _args(L.MOTE_BF16, 2, 2, 100, 48, row=1 << 24),        # rows off the tiles' offsets
], ids=["unpadded", "long padded", "long fp32", "far rows"])
def test_sizes_agree_where_nothing_is_chosen(a):
    full, least = _sizes(a)
    assert full == least > 0


@pytest.mark.parametrize("dtype,B,H,T,S,D,stored", [
    (L.MOTE_F32, 1, 8, 311, 4096, 64, False), (L.MOTE_F32, 1, 8, 311, 300, 64, True),     # fewer queries than prefix
    (L.MOTE_F32, 1, 8, 1000, 1500, 64, True),                                             # as many workgroups as CUs
    (L.MOTE_F32, 1, 16, 100, 1024, 128, True), (L.MOTE_F32, 1, 4, 311, 1024, 128, False),
    (L.MOTE_F32, 8, 8, 1300, 0, 32, True), (L.MOTE_F32, 8, 8, 2000, 0, 32, False), (L.MOTE_F32, 8, 8, 2000, 0, 64, True),
    (L.MOTE_BF16, 1, 4, 311, 4096, 48, False), (L.MOTE_BF16, 1, 4, 400, 4096, 48, True), (L.MOTE_BF16, 1, 2, 300, 1024, 48, True),
    (L.MOTE_BF16, 1, 1, 311, 4096, 120, False), (L.MOTE_BF16, 1, 8, 1, 8192, 64, True),
])
def test_few_queries_after_a_prefix_store_no_du(dtype, B, H, T, S, D, stored):
    """The rule's two sides: dU (8 or 16 KB a pair) is in the workspace or is not; a deterministic call stores it."""
    a = _args(dtype, B, H, T, D, S)
    a.deterministic = 1
    det = L.lib().mote_relation_bwd_workspace(a)
    a.deterministic = 0
    assert (L.lib().mote_relation_bwd_workspace(a) == det) == stored


@pytest.mark.parametrize("T", [1, 64, 65, 200])
def test_least_workspace_is_never_the_larger(T):
    for dtype, D in ((L.MOTE_BF16, 40), (L.MOTE_BF16, 120), (L.MOTE_F32, 8), (L.MOTE_F32, 128)):
        full, least = _sizes(_args(dtype, 2, 2, T, D))
        assert 0 < least <= full


def test_fewer_bytes_than_the_least_are_refused():
    a = _args(L.MOTE_F32, 1, 2, 100, 64)
    for n in ("dy", "dp1", "dp2", "dinfo"):
        setattr(a, n, a.p1)
    a.ibar = a.lse = a.g = a.dlam = 1 << 20
    a.workspace, a.workspace_bytes = 1 << 20, _sizes(a)[1] - 1
    assert L.lib().mote_relation_bwd(a, None) != 0 and b"workspace of" in L.lib().mote_last_error()


def _case(dtype, B, H, T, D, S, dev):
    g = torch.Generator().manual_seed(D + T)
    p1, dy = (torch.randn(B, H, T, D, generator=g).to(dtype).to(dev) for _ in range(2))
    p2, info = (torch.randn(B, H, S + T, D, generator=g).to(dtype).to(dev) for _ in range(2))
    return p1, p2, info, torch.tensor(0.4, device=dev), dy


@pytest.mark.gpu
@pytest.mark.parametrize("det", [0, 1])
@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 40), (torch.bfloat16, 48), (torch.bfloat16, 88), (torch.bfloat16, 120),
                                     (torch.float32, 24), (torch.float32, 64), (torch.float32, 128)])
@pytest.mark.parametrize("B,H,T,S", [(2, 1, 1400, 0), (1, 2, 1501, 37)])  # long enough for dU to outweigh the copies
def test_backward_on_the_least_workspace(cuda, dtype, D, B, H, T, S, det):
    """Against the float64 oracle at the suite's tolerances (2e-2 bf16, 1e-5 fp32 of the largest element)."""
    from mote_amd.flash_relation import _launch_fwd

    print(f"case least workspace {dtype} D={D} B={B} H={H} T={T} S={S} det={det}", flush=True)
    p1, p2, info, lam, dy = _case(dtype, B, H, T, D, S, cuda)
    _, gate, ibar, lse = _launch_fwd(p1, p2, info, lam, 2.0, S)
    a = _args(L.dtype_code(p1), B, H, T, D, S)
    out = [torch.full_like(t, float("nan")) for t in (p1, p2, info)]
    dlam = torch.full((), float("nan"), device=cuda)
    a.deterministic = det
    a.p1, a.p2, a.info, a.dy = (L.view(t) for t in (p1, p2, info, dy))
    a.ibar, a.lse, a.g, a.dlam = (t.data_ptr() for t in (ibar, lse, gate, dlam))
    a.dp1, a.dp2, a.dinfo = (L.view(t) for t in out)
    full, least = _sizes(a)
    assert least < full
    ws = torch.full((least,), 0xA5, device=cuda, dtype=torch.uint8)
    a.workspace, a.workspace_bytes = ws.data_ptr(), least
    L.check(L.lib().mote_relation_bwd(a, L.stream_of(p1)), "mote_relation_bwd")
    tol = 2e-2 if dtype == torch.bfloat16 else 1e-5
    ref = [t.cpu().double() for t in (p1, p2, info)]
    lr = torch.tensor(0.4, dtype=torch.float64)
    dr = O.relation_backward(*ref, lr, dy.cpu().double(), 2.0, S)
    for name, x, y in zip(("dp1", "dp2", "dinfo"), out, dr):
        assert rel_err(x, y) < tol, (name, rel_err(x, y))
    terms = O.relation_dlam_terms(*ref, lr, dy.cpu().double(), 2.0, S)
    assert abs(float(dlam) - float(dr[3])) < tol * max(float(terms.abs().sum()), 1e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,D,T,S", [(torch.float32, 24, 1, 70), (torch.float32, 48, 33, 300), (torch.float32, 96, 100, 101),
                                         (torch.bfloat16, 48, 1, 1536), (torch.bfloat16, 88, 65, 2000), (torch.bfloat16, 120, 7, 1600)])
def test_few_queries_after_a_prefix_match_oracle(cuda, dtype, D, T, S):
    """The route of few queries through the op, tolerances as above."""
    from mote_amd.flash_relation import flash_relation

    print(f"case few queries {dtype} D={D} T={T} S={S}", flush=True)
    p1, p2, info, lam, dy = _case(dtype, 1, 2, T, D, S, cuda)
    xs = [t.requires_grad_(True) for t in (p1, p2, info, lam)]
    got = torch.autograd.grad(flash_relation(*xs, 2.0, S)[0], xs, dy)
    tol = 2e-2 if dtype == torch.bfloat16 else 1e-5
    ref = [t.detach().cpu().double() for t in (p1, p2, info)]
    lr = torch.tensor(0.4, dtype=torch.float64)
    dr = O.relation_backward(*ref, lr, dy.cpu().double(), 2.0, S)
    for name, x, y in zip(("dp1", "dp2", "dinfo"), got, dr):
        assert rel_err(x, y) < tol, (name, rel_err(x, y))
    terms = O.relation_dlam_terms(*ref, lr, dy.cpu().double(), 2.0, S)
    assert abs(float(got[3]) - float(dr[3])) < tol * max(float(terms.abs().sum()), 1e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,D,T,spare", [(torch.bfloat16, 48, 4096, 80), (torch.float32, 64, 2048, 60)])
def test_backward_without_memory_for_the_stored_du(cuda, dtype, D, T, spare):
    """With the allocator held to `spare` MB more (the stored dU takes 136 and 69 MB, everything else under 45), the
    backward runs on the least workspace: the same gradients within the order of their sums (fp32) or a
    rounding of dU and of the result (bf16)."""
    from mote_amd import flash_relation as FR

    print(f"case bwd short of memory {dtype}", flush=True)
    p1, p2, info, lam, dy = _case(dtype, 1, 8, T, D, 0, cuda)
    _, gate, ibar, lse = FR._launch_fwd(p1, p2, info, lam, 2.0, 0)
    run = lambda: FR._launch_bwd(p1, p2, info, ibar, lse, gate, dy, 2.0, 0, False)
    want = [t.cpu() for t in run()]
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total, ooms = torch.cuda.mem_get_info()[1], torch.cuda.memory_stats()["num_ooms"]
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + spare * 2 ** 20) / total)
    try:
        got = run()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.cuda.memory_stats()["num_ooms"] > ooms, "the full workspace did not fit"
    for a, b in zip(got, want):
        assert rel_err(a, b) < (1e-2 if dtype == torch.bfloat16 else 1e-5), rel_err(a, b)
