"""The memo of the prologue's cos / sin tables: a table enters it once a launch has filled it, never from a
call that was refused or had no rows to launch for."""

from __future__ import annotations

import pytest
import torch

from conftest import rel_err


@pytest.mark.parametrize("rows", [0, 5])
def test_only_filled_tables_are_kept(monkeypatch, rows):
    """Host logic, with the launcher replaced: a refusal and an empty batch leave nothing behind, an accepted
    call its table."""
    from mote_amd import relation as R

    refuse = True

    class Native:
        @staticmethod
        def qkv_rope(x, *args):
            if refuse and rows:
                raise RuntimeError("refused")
            return x, x, x, x, x

    class Rows(torch.Tensor):
        is_cuda = True  # the launcher's device check; nothing here touches a GPU

    monkeypatch.setattr(R, "_ROPE_TABLES", {})
    monkeypatch.setattr(R.L, "native", lambda: Native)
    monkeypatch.setattr(R.L, "stream_of", lambda t: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    x = torch.zeros(rows, 3, 128, dtype=torch.bfloat16).as_subclass(Rows)
    w, inv = torch.zeros(384, 128, dtype=torch.bfloat16), R.rope_inv_freq(64, 10000.0)
    call = lambda: R._qkv_rope_launch(x, w, inv, None, 2, 0, 0, False, None, None, 1e-5)
    if rows:
        with pytest.raises(RuntimeError, match="refused"):
            call()
    else:
        call()
    assert not R._ROPE_TABLES
    refuse = False
    call()
    assert len(R._ROPE_TABLES) == (1 if rows else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["refused", "no rows"])
def test_call_after_an_unlaunched_one_matches_the_unfused_path(cuda, monkeypatch, how):
    """Head dim 48: QK-Norm is refused there, an empty batch launches nothing; the same call in earnest then
    equals the product and the RoPE kernel apart: the products differ in their fp32 order, so by one bf16 ulp
    (at most 2^-7 of the largest element) of either rotated operand and one of the result, under 2e-2."""
    from mote_amd import relation as R

    print(f"case rope table after {how}", flush=True)
    monkeypatch.setattr(R, "_ROPE_TABLES", {})
    g = torch.Generator().manual_seed(1)
    ws = tuple((torch.randn(192, 192, generator=g) / 14).bfloat16().to(cuda) for _ in range(3))
    x = torch.randn(2, 37, 192, generator=g).bfloat16().to(cuda)
    inv, one = R.rope_inv_freq(48, 10000.0, cuda), torch.ones(48, device=cuda)
    with torch.no_grad():
        if how == "refused":
            with pytest.raises(RuntimeError):
                R.qkv_rope(x, ws, 4, inv, None, 0, 3, (one, one, 1e-5))
        else:
            R.qkv_rope(x[:0], ws, 4, inv, None, 0, 3)
        got = R.qkv_rope(x, ws, 4, inv, None, 0, 3)
        want = R.rope_givens(torch.nn.functional.linear(x, torch.cat(ws)), 4, inv, None, 0, 3)
    for a, b in zip(got, want):
        assert rel_err(a, b) < 2e-2, rel_err(a, b)
