"""bf16 rows 2^24 or more elements apart: past the tile kernels' 32-bit row offsets, so the forward and the
backward run register-staged at every head dim, here against the float64 oracle of the same bf16 inputs at the
suite's bf16 tolerance (2e-2 of the largest element). The columns beside each head's own hold NaN."""

from __future__ import annotations

import pytest
import torch

from conftest import rel_err
from oracle import relation as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("det", [False, True])
@pytest.mark.parametrize("H,T,S,D", [(2, 1, 0, 64), (2, 130, 0, 32), (1, 65, 40, 64), (2, 64, 0, 96), (2, 97, 33, 128),
                                     (2, 100, 0, 48)])
def test_rows_past_the_tiles_offsets(cuda, H, T, S, D, det):
    from mote_amd.flash_relation import _launch_bwd, _launch_fwd

    print(f"case far rows H={H} T={T} S={S} D={D} det={det}", flush=True)
    g = torch.Generator().manual_seed(D + T)
    W = 8 * (3 * H * (D // 8 + 1))  # P1, P2 and I~ heads beside each other, eight NaN columns after each
    mem = torch.empty((S + T - 1) * (1 << 24) + W, device=cuda, dtype=torch.bfloat16)
    rows = mem.as_strided((S + T, W), (1 << 24, 1))
    rows.copy_(torch.randn(S + T, W, generator=g).bfloat16())
    heads = rows.unflatten(1, (3, H, D + 8))
    heads[..., D:] = float("nan")
    p1, p2, info = (heads[:, i, :, :D].transpose(0, 1)[None] for i in range(3))
    p1 = p1[:, :, S:]
    dy = torch.randn(1, H, T, D, generator=g).bfloat16().to(cuda)
    lam = torch.tensor(0.4, device=cuda)
    y, gate, ibar, lse = _launch_fwd(p1, p2, info, lam, 2.0, S)
    grads = _launch_bwd(p1, p2, info, ibar, lse, gate, dy, 2.0, S, det)
    ref = [t.cpu().double() for t in (p1, p2, info)]
    lr = torch.tensor(0.4, dtype=torch.float64)
    yr, gr = O.relation_reference(*ref, lr, 2.0, S, dtype=torch.float64)
    dr = O.relation_backward(*ref, lr, dy.cpu().double(), 2.0, S)
    assert rel_err(y, yr) < 2e-2 and rel_err(gate, gr) < 2e-2
    for name, a, b in zip(("dp1", "dp2", "dinfo"), grads[:3], dr[:3]):
        assert rel_err(a, b) < 2e-2, (name, rel_err(a, b))
    terms = O.relation_dlam_terms(*ref, lr, dy.cpu().double(), 2.0, S)
    assert abs(float(grads[3]) - float(dr[3])) < 2e-2 * max(float(terms.abs().sum()), 1e-3)
