"""mote_wgrad: the projections' weight gradient dW = A^T X (bf16, fp32 sums over the token rows),
through the C ABI and through mote::wgrad, against the float64 product of the same bf16 inputs.

The inputs are bf16, so the float64 product is the exact sum; the kernel's only roundings are its
fp32 accumulation and the one bf16 rounding of each output (2^-9 of the element), so 4e-3 of the
largest element bounds it. A transposed operand, a dropped or doubled stage, or the rows past M of
a ragged last stage counted would each miss by far more.
"""

from __future__ import annotations

import pytest
import torch

from conftest import rel_err

pytestmark = pytest.mark.gpu


def _abi_wgrad(a: torch.Tensor, x: torch.Tensor, dw: torch.Tensor) -> None:
    from mote_amd import _lib as Lb

    args = Lb.WgradArgs()
    args.dtype, args.M, args.N, args.K = Lb.MOTE_BF16, a.shape[0], a.shape[1], x.shape[1]
    args.a, args.a_sr = a.data_ptr(), a.stride(0)
    args.x, args.x_sr = x.data_ptr(), x.stride(0)
    args.dw, args.dw_sr = dw.data_ptr(), dw.stride(0)
    n = int(Lb.lib().mote_wgrad_workspace(args))
    ws = torch.full((max(n, 16),), 0x7F, device=a.device, dtype=torch.uint8)  # NaN-patterned partials
    args.workspace, args.workspace_bytes = ws.data_ptr(), ws.numel()
    Lb.check(Lb.lib().mote_wgrad(args, Lb.stream_of(a)), "mote_wgrad")
    torch.cuda.synchronize()


# (M, N, K): one stage, ragged last stages (1, 63, 65 rows past a stage), one tile and many splits,
# the Mote-96M prologue (2304 x 768, four splits) and gate (768 x 768) shapes
CASES = [(1, 128, 128), (63, 256, 128), (64, 128, 256), (65, 384, 128), (300, 1536, 512), (2000, 128, 128),
         (4964, 2304, 768), (4964, 768, 768), (9001, 256, 384)]


@pytest.mark.parametrize("M,N,K", CASES)
def test_wgrad_matches_float64(cuda, M, N, K):
    print(f"case wgrad M={M} N={N} K={K}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(M, N, generator=g).bfloat16()
    x = torch.randn(M, K, generator=g).bfloat16()
    ref = a.double().t() @ x.double()
    ac, xc = a.to(cuda), x.to(cuda)
    dw = torch.full((N, K), float("nan"), device=cuda, dtype=torch.bfloat16)
    _abi_wgrad(ac, xc, dw)
    assert rel_err(dw, ref) < 4e-3, rel_err(dw, ref)
    again = torch.full_like(dw, float("nan"))
    _abi_wgrad(ac, xc, again)
    assert torch.equal(dw, again), "bitwise reproducible"


# widths off 128 (64-wide tiles on either side or both), both output types, one split and many, ragged
# last stages, an empty reduction. fp32 dW: sums of products of bf16 values in fp32 over M rows, so M
# roundings of 2^-24 against a sum whose terms reach about M^(1/2) times less than their absolute sum:
# 1e-5 of the largest element holds with room for every M here.
@pytest.mark.parametrize("M,N,K", [(0, 64, 64), (1, 64, 192), (65, 192, 64), (300, 576, 192), (1241, 192, 128), (9929, 320, 192),
                                   (4964, 256, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_linear_wgrad_widths_and_types(cuda, M, N, K, dtype):
    from mote_amd.relation import _linear_wgrad

    print(f"case linear_wgrad M={M} N={N} K={K} {dtype}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(M, N + 8, generator=g).bfloat16().to(cuda)[:, :N]  # row stride above the width
    x = torch.randn(M, K, generator=g).bfloat16().to(cuda)
    dw = _linear_wgrad(a, x, dtype)
    ref = a.double().t().contiguous() @ x.double()
    assert dw.shape == (N, K) and dw.dtype == dtype
    assert rel_err(dw, ref) < (1e-5 if dtype == torch.float32 else 4e-3), rel_err(dw, ref)
    assert torch.equal(dw, _linear_wgrad(a, x, dtype)), "bitwise reproducible"


def test_wgrad_strided_rows(cuda):
    """Operands and output as column windows of wider row-major tensors (row strides above the
    widths): only the window is read and written."""
    print("case wgrad strided", flush=True)
    g = torch.Generator().manual_seed(3)
    A = torch.randn(777, 640, generator=g).bfloat16().to(cuda)
    X = torch.randn(777, 512, generator=g).bfloat16().to(cuda)
    a, x = A[:, 128:384], X[:, 256:384]
    out = torch.full((256, 384), 7.0, device=cuda, dtype=torch.bfloat16)
    dw = out[:, 128:256]
    _abi_wgrad(a, x, dw)
    ref = a.cpu().double().t() @ x.cpu().double()
    assert rel_err(dw, ref) < 4e-3
    assert bool((out[:, :128] == 7).all()) and bool((out[:, 256:] == 7).all())


def test_wgrad_empty_reduction_writes_zeros(cuda):
    print("case wgrad M=0", flush=True)
    a = torch.empty(0, 128, device=cuda, dtype=torch.bfloat16)
    x = torch.empty(0, 256, device=cuda, dtype=torch.bfloat16)
    dw = torch.full((128, 256), float("nan"), device=cuda, dtype=torch.bfloat16)
    _abi_wgrad(a, x, dw)
    assert bool((dw == 0).all())


def test_weight_grad_op_and_dispatch(cuda):
    """mote::wgrad through weight_grad (batched rows, a non-contiguous x) against torch's product,
    the op's registration checked by opcheck, and the library product for widths off 128."""
    from mote_amd.relation import _wgrad, weight_grad

    print("case wgrad op", flush=True)
    g = torch.Generator().manual_seed(5)
    a = torch.randn(2, 301, 384, generator=g).bfloat16().to(cuda)
    xw = torch.randn(2, 301, 512, generator=g).bfloat16().to(cuda)
    x = xw[..., :256]
    got = weight_grad(a, x)
    ref = a.reshape(-1, 384).double().t() @ x.reshape(-1, 256).double()
    assert got.shape == (384, 256) and got.dtype == torch.bfloat16
    assert rel_err(got, ref) < 4e-3
    torch.library.opcheck(_wgrad, (a.reshape(-1, 384), x.reshape(-1, 256).contiguous()))
    odd = weight_grad(a[..., :200], x)  # N = 200: the library product
    assert rel_err(odd, a[..., :200].reshape(-1, 200).double().t() @ x.reshape(-1, 256).double()) < 1e-2


@pytest.mark.parametrize("autocast", [False, True])
def test_module_weight_gradients_on_wgrad(cuda, monkeypatch, autocast):
    """FullRelation's backward with the weight gradients of the prologue, the gate and wo on
    mote_wgrad against the same step with them on the GEMM library: bf16 weights, or fp32 weights
    under bf16 autocast (the weights' bf16 casts carry the gradients back to fp32)."""
    from mote_amd import relation as R

    print(f"case wgrad module autocast={autocast}", flush=True)
    torch.manual_seed(12)
    dtype = torch.float32 if autocast else torch.bfloat16
    m = R.FullRelation(256, 4, 1, out_gate=True, dtype=dtype).to(cuda)
    x = (torch.randn(2, 300, 256, device=cuda) * 0.5).to(dtype)
    dy = torch.randn(2, 300, 256, device=cuda).to(dtype)

    def grads(use):
        monkeypatch.setattr(R, "USE_WGRAD", use)
        m.zero_grad(set_to_none=True)
        xi = x.clone().requires_grad_(True)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
            out = m(xi)
        (out.float() * dy.float()).sum().backward()
        return {n: p.grad.clone() for n, p in m.named_parameters() if p.grad is not None}, xi.grad.clone()

    got, gx = grads(True)
    ref, rx = grads(False)
    assert set(got) == set(ref) and {"w1.weight", "wo.weight", "wg.weight"} <= set(got)
    for n in ref:
        assert got[n].dtype == ref[n].dtype, n
        assert rel_err(got[n], ref[n]) < 1e-2, (n, rel_err(got[n], ref[n]))
    assert rel_err(gx, rx) < 1e-2


def test_linear_wgrad_function_under_create_graph(cuda):
    """linear_wgrad with fp32 weights under autocast: its first gradients carry W's own dtype, and a
    second differentiation goes through both products and the cast, as through F.linear."""
    from mote_amd.relation import linear_wgrad

    print("case linear_wgrad create_graph", flush=True)
    torch.manual_seed(3)
    x = torch.randn(40, 192, device=cuda, dtype=torch.bfloat16, requires_grad=True)
    w = (torch.randn(64, 192, device=cuda) / 14).requires_grad_(True)

    def second(fn):
        with torch.autocast("cuda", torch.bfloat16):
            y = fn(x, w)
        gx, gw = torch.autograd.grad(y.float().square().sum(), (x, w), create_graph=True)
        assert gx.dtype == torch.bfloat16 and gw.dtype == torch.float32
        return torch.autograd.grad(gx.float().square().sum() + gw.square().sum(), (x, w))

    for a, b in zip(second(linear_wgrad), second(torch.nn.functional.linear)):
        assert a.dtype == b.dtype and rel_err(a, b) < 2e-2, rel_err(a, b)


def _rows(form, M, N, dev):
    """bf16 [M, N] operands whose rows the kernel cannot walk where they are."""
    t = torch.randn(M, N, device=dev).bfloat16()
    if form == "expanded":
        return t[:1].expand(M, N)
    if form == "far apart":  # a row stride past the kernel's 32-bit offsets
        return torch.empty((M - 1) * (1 << 24) + N, device=dev, dtype=torch.bfloat16).as_strided((M, N), (1 << 24, 1)).copy_(t)
    if form == "overlapping":
        return torch.randn((M - 1) * 8 + N, device=dev).bfloat16().as_strided((M, N), (8, 1))
    if form == "off a boundary":  # contiguous, so contiguous() would keep it
        return torch.empty(M * N + 1, device=dev, dtype=torch.bfloat16)[1:].view(M, N).copy_(t)
    if form == "one row":  # contiguous whatever its row stride says
        return t[0].clone().as_strided((1, N), (1, 1))
    return t


@pytest.mark.parametrize("N,K", [(192, 64), (128, 256)])
@pytest.mark.parametrize("form", ["expanded", "far apart", "overlapping", "off a boundary", "one row"])
def test_rows_the_kernel_cannot_walk_are_copied(cuda, N, K, form):
    """Either operand, through mote::linear_wgrad and (multiples of 128) mote::wgrad; bounds as above."""
    from mote_amd.relation import _linear_wgrad, _wgrad

    print(f"case wgrad rows {form} N={N} K={K}", flush=True)
    torch.manual_seed(N)
    for fa, fx in ((form, "plain"), ("plain", form)):
        M = 1 if form == "one row" else 5
        a, x = _rows(fa, M, N, cuda), _rows(fx, M, K, cuda)
        ref = a.double().t().contiguous() @ x.double().contiguous()
        assert rel_err(_linear_wgrad(a, x, torch.float32), ref) < 1e-5
        if N % 128 == 0:
            assert rel_err(_wgrad(a, x), ref) < 4e-3


@pytest.mark.parametrize("reduce", [lambda y: y.sum((0, 1)), lambda y: y.sum(1)], ids=["sum over rows", "sum over time"])
@pytest.mark.parametrize("d,H", [(192, 4), (256, 4)])
def test_output_reduced_over_its_rows(cuda, monkeypatch, d, H, reduce):
    """A layer's output summed over its rows hands wo's backward a gradient of row stride 0: weight
    gradients as with the products on the GEMM library (bf16 there: 2^-9 an element, and a change of order)."""
    from mote_amd import relation as R

    print(f"case reduced output d={d}", flush=True)
    torch.manual_seed(2)
    m = R.FullRelation(d, H, 0, device=cuda)
    x = torch.randn(1, 77, d, device=cuda)
    dy = torch.randn(d, device=cuda)

    def grads(use):
        monkeypatch.setattr(R, "USE_WGRAD", use)
        with torch.autocast("cuda", torch.bfloat16):
            out = reduce(m(x))
        return torch.autograd.grad(out, list(m.parameters()), dy.to(out.dtype).expand_as(out))

    for a, b in zip(grads(True), grads(False)):
        assert rel_err(a, b) < 1e-2, rel_err(a, b)


@pytest.mark.parametrize("d,H", [(192, 4), (256, 4)])
def test_backward_after_an_in_place_weight_update(cuda, d, H):
    """Under autocast a graph keeps the weights' bf16 copies, so a backward after an optimizer's in-place step
    on the fp32 masters gives the gradients it would have given before (Givens off: theta itself is saved)."""
    from mote_amd.relation import FullRelation

    print(f"case backward after update d={d}", flush=True)
    torch.manual_seed(4)
    m = FullRelation(d, H, 0, givens=False, device=cuda)
    x = torch.randn(2, 50, d, device=cuda, requires_grad=True)
    leaves = [x, *m.parameters()]
    with torch.autocast("cuda", torch.bfloat16):
        out = m(x)
    dy = torch.randn_like(out)
    before = torch.autograd.grad(out, leaves, dy, retain_graph=True)
    with torch.no_grad():
        for p in m.parameters():
            p.mul_(0.5)
    for a, b in zip(torch.autograd.grad(out, leaves, dy), before):
        assert a.dtype == torch.float32 and torch.equal(a, b)


@pytest.mark.parametrize("N,K", [(64, 192), (128, 128)])
def test_linear_wgrad_under_transforms(cuda, N, K):
    """grad, vmap, jvp, forward-mode levels and batched gradients over linear_wgrad, as over F.linear: every
    product the library's, so they differ by the order of a batched one alone: one bf16 rounding, 2^-7 of the
    largest element."""
    from mote_amd.relation import linear_wgrad

    print(f"case linear_wgrad transforms N={N}", flush=True)
    torch.manual_seed(6)
    x, t = (torch.randn(3, 20, K, device=cuda).bfloat16() for _ in range(2))
    w = (torch.randn(N, K, device=cuda) / K ** 0.5).bfloat16()
    F = torch.nn.functional

    def forward_mode(fn):
        with torch.autograd.forward_ad.dual_level():
            return torch.autograd.forward_ad.unpack_dual(fn(torch.autograd.forward_ad.make_dual(x, t), w)).tangent

    def batched(fn):
        wr = w.clone().requires_grad_(True)
        y = fn(x, wr)
        return torch.autograd.grad(y, wr, torch.stack([y.detach(), 2 * y.detach()]), is_grads_batched=True)[0]

    for run in (lambda fn: torch.func.grad(lambda v: fn(x, v).float().square().sum())(w),
                lambda fn: torch.func.vmap(fn, (0, None))(x, w),
                lambda fn: torch.func.jvp(lambda v: fn(v, w), (x,), (t,))[1], forward_mode, batched):
        got, want = run(linear_wgrad), run(F.linear)
        assert got.shape == want.shape and rel_err(got, want) < 2.0 ** -7, rel_err(got, want)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float16])
@pytest.mark.parametrize("N", [64, 72])
def test_linear_wgrad_casts_other_weights_under_autocast(cuda, N, dtype):
    """Weights that autocast's own F.linear refuses (fp64) or casts (fp16), at a served width and beside it:
    the product of the bf16 casts, gradients in the weights' dtype (bf16 roundings, 2^-9 each)."""
    from mote_amd.relation import linear_wgrad

    print(f"case linear_wgrad weights {dtype} N={N}", flush=True)
    torch.manual_seed(7)
    x = torch.randn(30, 128, device=cuda, requires_grad=True)
    w = (torch.randn(N, 128, device=cuda) / 12).to(dtype).requires_grad_(True)
    with torch.autocast("cuda", torch.bfloat16):
        y = linear_wgrad(x, w)
    xb, wb = x.detach().bfloat16().double(), w.detach().bfloat16().double()
    assert y.dtype == torch.bfloat16 and rel_err(y, xb @ wb.t()) < 1e-2
    dx, dw = torch.autograd.grad(y, (x, w), torch.ones_like(y))
    assert dx.dtype == torch.float32 and dw.dtype == dtype
    assert rel_err(dx, wb.sum(0).expand_as(dx)) < 1e-2 and rel_err(dw, xb.sum(0).expand_as(dw)) < 1e-2
