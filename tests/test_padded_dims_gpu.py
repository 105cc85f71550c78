"""bf16 head dims off 32 / 64 / 96 / 128 on the tile kernels, padded to the next of them: forward and
backward against the float64 oracle of the same bf16 inputs at the suite's bf16 tolerance (2e-2 of the
largest element). Every operand is a column window of wider rows whose other columns hold NaN, so a
kernel that read past a head's own columns (instead of repeating its last chunk) would show it; lengths
cover one row, one block, block edges and several blocks with a cached prefix off the block grid."""

from __future__ import annotations

import pytest
import torch

from conftest import rel_err
from oracle import relation as O

pytestmark = pytest.mark.gpu


def _window(g, B, T, H, D, dev):
    """bf16 [B, H, T, D] values inside [B, T, H, D + 8] rows whose last 8 columns are NaN."""
    buf = torch.full((B, T, H, D + 8), float("nan"))
    buf[..., :D] = torch.randn(B, T, H, D, generator=g)
    return buf.bfloat16().to(dev)[..., :D].transpose(1, 2)


@pytest.mark.parametrize("D", [8, 24, 40, 48, 56, 72, 88, 104, 120])
@pytest.mark.parametrize("B,H,T,S", [(1, 2, 1, 0), (2, 1, 64, 0), (1, 4, 130, 37), (1, 2, 300, 0)])
def test_padded_head_dims_match_oracle(cuda, D, B, H, T, S):
    from mote_amd.flash_relation import flash_relation

    print(f"case padded D={D} B={B} H={H} T={T} S={S}", flush=True)
    g = torch.Generator().manual_seed(D + T)
    p1, p2, info = _window(g, B, T, H, D, cuda), _window(g, B, S + T, H, D, cuda), _window(g, B, S + T, H, D, cuda)
    dy = _window(g, B, T, H, D, cuda)
    lam = torch.tensor(0.4, device=cuda, requires_grad=True)
    xs = [t.detach().requires_grad_(True) for t in (p1, p2, info)]
    y, gate = flash_relation(*xs, lam, 2.0, S)
    grads = torch.autograd.grad(y, [*xs, lam], dy)
    ref = [t.cpu().double() for t in (p1, p2, info)]
    lr = torch.tensor(0.4, dtype=torch.float64)
    yr, gr = O.relation_reference(*ref, lr, 2.0, S, dtype=torch.float64)
    dr = O.relation_backward(*ref, lr, dy.cpu().double(), 2.0, S)
    assert rel_err(y, yr) < 2e-2 and rel_err(gate, gr) < 2e-2
    for name, a, b in zip(("dp1", "dp2", "dinfo"), grads[:3], dr[:3]):
        assert rel_err(a, b) < 2e-2, (name, rel_err(a, b))
    terms = O.relation_dlam_terms(*ref, lr, dy.cpu().double(), 2.0, S)
    assert abs(float(grads[3]) - float(dr[3])) < 2e-2 * max(float(terms.abs().sum()), 1e-3)
    again = torch.autograd.grad(flash_relation(*xs, lam, 2.0, S)[0], xs, dy)
    assert all(torch.equal(a, b) for a, b in zip(again, grads)), "no atomics: the gradients repeat bit for bit"


@pytest.mark.parametrize("D", [40, 48, 104])
def test_padded_varlen_equals_dense(cuda, D):
    """The packed launch (persistent workgroups from eight query blocks per CU, forced here) and the
    two-launch backward of padded head dims against the dense one-launch forms."""
    import os

    from mote_amd.flash_relation import flash_relation, flash_relation_varlen

    print(f"case padded varlen D={D}", flush=True)
    g = torch.Generator().manual_seed(D)
    lens = [1, 63, 200]
    cu = torch.tensor([0, 1, 64, 264], dtype=torch.int32, device=cuda)
    p = [_window(g, 1, 264, 2, D, cuda)[0] for _ in range(3)]
    lam = torch.tensor(0.3, device=cuda)
    old = os.environ.get("MOTE_FWD_PERSIST"), os.environ.get("MOTE_BWD_FUSED")
    try:
        os.environ["MOTE_FWD_PERSIST"] = "1"
        yv, gv = flash_relation_varlen(*p, lam, cu, 200)
        os.environ["MOTE_FWD_PERSIST"] = "0"
        r = 0
        for n in lens:
            one = [t[None, :, r: r + n].detach().requires_grad_(True) for t in p]
            y, gate = flash_relation(*one, lam)
            assert torch.equal(yv[:, r: r + n], y[0]) and torch.equal(gv[:, r: r + n], gate[0])
            grads = []
            for fused in ("0", "1"):
                os.environ["MOTE_BWD_FUSED"] = fused
                grads.append(torch.autograd.grad(flash_relation(*one, lam)[0].float().square().sum(), one))
            assert torch.equal(grads[0][0], grads[1][0])
            assert all(rel_err(a, b) < 1e-2 for a, b in zip(grads[0][1:], grads[1][1:]))
            r += n
    finally:
        for k, v in zip(("MOTE_FWD_PERSIST", "MOTE_BWD_FUSED"), old):
            os.environ.pop(k, None) if v is None else os.environ.__setitem__(k, v)


@pytest.mark.parametrize("D", [8, 24, 48, 88, 120])
@pytest.mark.parametrize("T,S", [(1, 40), (64, 0), (300, 37)])
def test_padded_row_sums_are_fp32(cuda, D, T, S):
    """lse and g come from weights added in fp32 before their rounding to bf16, so they are off the float64
    values of the same inputs by fp32 arithmetic alone: the scores' sums and the exponentials, a few 2^-24 of
    exponents up to about 10, under 1e-5 (weights summed after the rounding: 1e-3). I-bar keeps one bf16 rounding
    a weight, 2^-9 at most."""
    from mote_amd.flash_relation import _launch_fwd

    print(f"case padded sums D={D} T={T} S={S}", flush=True)
    g = torch.Generator().manual_seed(D + T)
    p1, p2, info = _window(g, 1, T, 2, D, cuda), _window(g, 1, S + T, 2, D, cuda), _window(g, 1, S + T, 2, D, cuda)
    _, gate, ibar, lse = _launch_fwd(p1, p2, info, torch.tensor(0.4, device=cuda), 2.0, S)
    u = torch.matmul(p1.double(), p2.double().transpose(2, 3).contiguous()) / D ** 0.5
    at = torch.arange(S, S + T, device=cuda)
    past = torch.arange(S + T, device=cuda)[None] < at[:, None]
    e = torch.nn.functional.silu(u).masked_fill(~past, float("-inf"))
    ref = torch.logsumexp(e, -1)
    self_ = torch.sigmoid(torch.diagonal(u, S, 2, 3) / 2.0)
    has = past.any(-1)
    gref = torch.sigmoid(ref - 0.4 * torch.log(at.double() + 1) - self_)
    assert float((lse.double() - ref)[..., has].abs().max()) < 1e-5
    assert bool((lse[..., ~has] == float("-inf")).all()) and bool((gate[..., ~has] == 0).all())
    assert float((gate.double() - gref)[..., has].abs().max()) < 1e-5
    bref = torch.matmul(torch.softmax(e, -1).nan_to_num(), info.double().contiguous())
    assert float((ibar.double() - bref).norm() / bref.norm()) < 2.0 ** -9
