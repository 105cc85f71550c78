"""The refusals of test_call_checks.py through the module on the GPU: what a refused call must leave alone."""

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
