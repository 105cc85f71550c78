"""The checks of test_call_checks.py on the GPU: what a refused call must leave alone, and what is not refused."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,H,wrong", [(768, 8, 1024), (192, 4, 256)])
def test_refused_width_leaves_the_cache_alone(cuda, d, H, wrong):
    from mote_amd.arena import ArenaState, RelationArena
    from mote_amd.relation import FullRelation

    print(f"case refused width {wrong} at {d} x {H}", flush=True)
    m = FullRelation(d, H, 0, device=cuda, dtype=torch.bfloat16)
    arena = RelationArena(1, H, 256, d // H, "cuda", torch.bfloat16)
    arena.store.normal_()
    before = arena.store.clone()
    with pytest.raises(RuntimeError, match=f"takes x .*{d}"), torch.no_grad():
        m(torch.zeros(1, 256, wrong, device=cuda, dtype=torch.bfloat16), cache=ArenaState(arena, n=0)[0])
    assert torch.equal(arena.store, before)


@pytest.mark.parametrize("longer", ["w", "inv_freq", "theta"])
def test_prologue_reads_longer_operands_at_their_start(cuda, longer):
    from mote_amd.relation import qkv_rope

    print(f"case longer {longer}", flush=True)
    g = torch.Generator().manual_seed(3)
    ops = {"w": torch.randn(768, 256, generator=g).bfloat16(), "inv_freq": torch.rand(32, generator=g), "theta": torch.rand(2, generator=g)}
    ops = {k: v.to(cuda) for k, v in ops.items()}
    x = torch.randn(1, 70, 256, generator=g).bfloat16().to(cuda)
    call = lambda o: qkv_rope(x, o["w"], 4, o["inv_freq"], o["theta"], 0, 0)
    with torch.no_grad():
        want, got = call(ops), call({**ops, longer: torch.cat([ops[longer], torch.full_like(ops[longer], float("nan"))])})
    assert all(torch.equal(a, b) for a, b in zip(want, got))
