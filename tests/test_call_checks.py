"""Calls that must be refused on the host, before anything is launched: shapes, dtypes and devices that the
kernels would read or write out of range with. The launchers check them ahead of the device, so CPU
tensors show every refusal."""

from __future__ import annotations

import ctypes as C

import pytest
import torch

from mote_amd import _lib as L
from mote_amd import relation as R

BF16 = torch.bfloat16


def _prologue(x, ws, p2=None, info=None, inv=None, theta=None, H=4):
    table = torch.empty(max(16, x.shape[1] * 2 * (x.shape[2] // H)), dtype=torch.uint8)
    return L.native().qkv_rope(x, ws, inv, theta, H, 0, 0, False, None, None, 1e-5, table, False, p2, info, 0)


@pytest.mark.parametrize("shape", [(2, 5, 1024), (2, 5, 512), (5, 768)])
def test_module_refuses_rows_of_another_width(shape):
    """768 x 8 (head dim 96): 1024-wide rows would run the prologue at head dim 128 over weights and cache
    rows of 96."""
    m = R.FullRelation(768, 8, 0, dtype=BF16)
    x = torch.zeros(shape, dtype=BF16)
    for call in (m, lambda t: m.heads(t, 0), lambda t: m._heads_into(t, 0, None)):
        with pytest.raises(RuntimeError, match=r"takes x \[B, T, 768\]"), torch.no_grad():
            call(x)


@pytest.mark.parametrize("bad", [
    lambda: torch.zeros(2, 4, 5, 48, dtype=BF16),     # another head dim
    lambda: torch.zeros(2, 4, 4, 64, dtype=BF16),     # fewer rows
    lambda: torch.zeros(1, 4, 5, 64, dtype=BF16),     # a smaller batch
    lambda: torch.zeros(2, 4, 5, 64),                 # another dtype
    lambda: torch.zeros(2, 4, 5, 64, dtype=BF16, device="meta"),
], ids=["head dim", "rows", "batch", "dtype", "device"])
def test_prologue_refuses_cache_rows_of_another_form(bad):
    x, w = torch.zeros(2, 5, 256, dtype=BF16), [torch.zeros(256, 256, dtype=BF16)] * 3
    good = torch.zeros(2, 4, 5, 64, dtype=BF16)
    for p2, info in ((bad(), good), (good, bad())):
        with pytest.raises(RuntimeError, match="P2 and I~ must be"):
            _prologue(x, w, p2, info)


@pytest.mark.parametrize("view", ["p1", "p2", "info"])
@pytest.mark.parametrize("stride", ["stride_b", "stride_h", "stride_r"])
def test_prologue_entry_refuses_overlapping_rows(view, stride):
    """The C entry knows no extents, but rows of D elements closer than D apart are refused."""
    a = L.QkvRopeArgs()
    a.B, a.T, a.H, a.D = 2, 5, 4, 128
    a.x, a.x_sb, a.x_sr, a.w, a.w_sr = 1 << 20, 5 * 512, 512, 1 << 21, 512
    for n in ("p1", "p2", "info"):
        setattr(a, n, L.View(1 << 22, 4 * 5 * 128, 5 * 128, 128))
    setattr(getattr(a, view), stride, 96)
    rc = L.lib().mote_qkv_rope_parts_fwd(a, C.c_void_p(1 << 21), C.c_void_p(1 << 21), None)
    assert rc != 0 and b"strides of at least 128" in L.lib().mote_last_error()


@pytest.mark.parametrize("what,match", [
    ("x dtype", "x must be bf16"), ("heads", "x must be bf16"), ("one weight", "weights must be"), ("stack", "weights must be"),
    ("weight dtype", "weights must be"), ("weight device", "weights must be"), ("inv_freq", "inv_freq needs"), ("theta", "theta needs"),
])
def test_prologue_refuses_operands_of_other_sizes(what, match):
    """256-wide rows over the weights and frequencies of another layer would be read past their ends."""
    x, w = torch.zeros(2, 5, 256, dtype=BF16), torch.zeros(256, 256, dtype=BF16)
    args = {"x dtype": (x.float(), [w] * 3), "heads": (x, [w] * 3, None, None, None, None, 3), "one weight": (x, [w, w[:192], w]),
            "stack": (x, [torch.zeros(768, 192, dtype=BF16)]), "weight dtype": (x, [w, w.float(), w]),
            "weight device": (x, [w, w, w.to("meta")]), "inv_freq": (x, [w] * 3, None, None, torch.zeros(24)),
            "theta": (x, [w] * 3, None, None, torch.zeros(32), torch.zeros(1))}[what]
    with pytest.raises(RuntimeError, match=match):
        _prologue(*args)


@pytest.mark.parametrize("shapes", [((64, 64), (64, 32), (64, 64)), ((64, 64), (64, 64), (32, 64))])
def test_weight_stack_refuses_unequal_weights(shapes):
    x, ws = torch.zeros(1, 1, 64, dtype=BF16), [torch.zeros(s) for s in shapes]
    with pytest.raises(RuntimeError, match="of one shape"):
        R._packed(x, *ws)
    ws = [torch.zeros(64, 64), torch.zeros(64, 64, device="meta"), torch.zeros(64, 64)]
    with pytest.raises(RuntimeError, match="on x's device"):
        R._packed(x, *ws)


@pytest.mark.parametrize("x", [torch.zeros(6, 64, dtype=BF16), torch.zeros(7, 64), torch.zeros(7, 64, dtype=BF16, device="meta"),
                               torch.zeros(1, 7, 64, dtype=BF16)], ids=["rows", "dtype", "device", "dims"])
def test_weight_gradient_refuses_unlike_operands(x):
    """A shorter x would be read past its end, an fp32 one as bf16."""
    with pytest.raises(RuntimeError, match=r"linear_wgrad: a \[M, N\] and x"):
        L.native().linear_wgrad(torch.zeros(7, 128, dtype=BF16), x, torch.float32, 0)


@pytest.mark.parametrize("bad", [torch.zeros(1, 4, 64, dtype=BF16), torch.zeros(1, 5, 64), torch.zeros(1, 5, 64, dtype=BF16, device="meta")],
                         ids=["shape", "dtype", "device"])
def test_gate_backward_refuses_unlike_operands(bad):
    """The launch is sized by dz: a smaller y or s would be read, a smaller dy written, past the end."""
    good = torch.zeros(1, 5, 64, dtype=BF16)
    for args in ((good, bad, good), (good, good, bad)):
        with pytest.raises(RuntimeError, match="of one shape on one device"):
            R._gate_bwd._init_fn(*args)
