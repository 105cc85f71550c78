"""The calls a program makes of this package, as cases that can be timed and compared.

Kinds of case:

* block    One residual block of the chunk-level network in training: RMSNorm with the fused residual
           add, FullRelation (projections, RoPE / Givens, the Relation core, optional QK-Norm and
           output gate, wo), forward and backward, under bf16 autocast with fp32 master weights or in
           fp32. With `graph` the step is captured once as a HIP graph and replayed, as a program with
           bucketed windows does where a layer is shorter than its own launches.
* prefill  flash_relation_varlen over a ragged batch of packed sequences.
* extend   New rows appended to a cached prefix: FullRelation.forward with an arena, no gradients (a
           prompt or a turn of a conversation after the rows that the cache already holds).
* decode   The decode engine's token: RMSNorm and the Relation step of every layer, chained through
           the residual stream, captured as one HIP graph.
* chunk    Bytes to chunks and back, forward and backward: boundary routing, gather, EMA dechunk.

Widths and heads are those of the presets this repository is measured on (192 x 4 heads, 512 x 8,
768 x 8) and the generic head dim 128 (1024 x 8).
"""

from __future__ import annotations

import math

import torch

WIDTHS = {192: 4, 512: 8, 768: 8, 1024: 8}  # d_model -> heads: head dims 48, 64, 96, 128


# ---- the cases -----------------------------------------------------------------------------------
def _block(name, d, batch, T, dtype="bf16", gate=False, norm=False, graph=False, odd=False):
    c = dict(kind="block", d=d, batch=batch, T=T, dtype=dtype, gate=gate, norm=norm, graph=graph, odd=odd)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest preset in fp32 at two short windows, eager: launch-bound
        _block("block_192_fp32_small", 192, 2, 256, "fp32"),
        # the smallest preset trained as it is meant to be: bf16, sixteen 4 KB windows, head dim 48
        _block("block_192_bf16", 192, 16, 1241, graph=True, odd=True),
        # four 2 KB windows padded to the longest
        _block("block_512", 512, 4, 658, graph=True),
        # the same preset in full precision (a debugging or ablation run)
        _block("block_512_fp32", 512, 4, 620, "fp32", graph=True, odd=True),
        # one 16 KB window of the 768-wide preset
        _block("block_768", 768, 1, 4964, graph=True),
        # two 8 KB windows with every module option on
        _block("block_768_options", 768, 2, 2483, gate=True, norm=True, graph=True, odd=True),
        # head dim 128, four long windows, eager: the largest
        _block("block_1024", 1024, 4, 4096),
        # a serving prefill: eight ragged sequences of 1000 to 5000 chunks
        dict(name="prefill_768_ragged", kind="prefill", d=768, batch=8, low=1000, high=5000),
        # a 1 KB turn after 4096 cached chunks
        dict(name="extend_768", kind="extend", d=768, batch=1, S=4096, T=311),
        # the decode engine, one sequence and sixteen
        dict(name="decode_768_b1", kind="decode", d=768, layers=12, batch=1, S=4096),
        dict(name="decode_768_b16", kind="decode", d=768, layers=12, batch=16, S=4096),
        # eight 16 KB windows of bytes at the encoder's width
        dict(name="chunk_512_b8", kind="chunk", d=512, batch=8, L=16384),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["block"] * 6 + ["prefill", "extend", "decode", "chunk"])
    if kind == "block":
        d = rng.choice([192, 512, 768, 1024])
        dtype = "fp32" if d <= 512 and rng.random() < 0.3 else "bf16"
        T = _log(rng, 64, 1300 if dtype == "fp32" else 5000)
        most = 8192 if dtype == "fp32" else 16384      # token rows of a step
        most = max(1, min(most // T, int(5.0e7 / (T * T)) if dtype == "bf16" else int(4.0e6 / (T * T)), 32))
        batch = min(most, _log(rng, 1, 32))
        return _block(None, d, batch, T, dtype, gate=rng.random() < 0.25, norm=rng.random() < 0.25,
                      graph=rng.random() < 0.7, odd=rng.random() < 0.5)
    if kind == "prefill":
        high = _log(rng, 200, 5000)
        return dict(kind="prefill", d=rng.choice([512, 768, 1024]), batch=rng.randint(2, 8), low=max(1, high // 5), high=high)
    if kind == "extend":
        return dict(kind="extend", d=rng.choice([512, 768]), batch=1, S=_log(rng, 256, 8192), T=_log(rng, 16, 1300))
    if kind == "decode":
        return dict(kind="decode", d=rng.choice([512, 768]), layers=rng.choice([8, 12]), batch=rng.choice([1, 2, 4, 8, 16]),
                    S=_log(rng, 256, 8192))
    return dict(kind="chunk", d=rng.choice([256, 512, 768]), batch=_log(rng, 1, 8), L=_log(rng, 1024, 16384))


# ---- inputs ----------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)


def _weights(g, m):
    """The module's parameters from the seed: projections as nn.Linear starts them, angles and
    gains as they are some way into training."""
    d = m.d_model
    with torch.no_grad():
        for n, p in m.named_parameters():
            if n == "lam":
                p.fill_(0.5)
            elif n == "theta":
                p.copy_(torch.rand(p.shape, generator=g, device="cuda") * 0.6 - 0.3)
            elif "norm" in n:
                p.copy_(1.0 + 0.1 * torch.randn(p.shape, generator=g, device="cuda"))
            else:
                p.copy_((torch.rand(p.shape, generator=g, device="cuda") * 2 - 1) / math.sqrt(d))


def _relation(c, g, layer):
    from mote_amd.relation import FullRelation

    m = FullRelation(c["d"], WIDTHS[c["d"]], layer, qk_norm=c.get("norm", False), out_gate=c.get("gate", False),
                     device="cuda")
    _weights(g, m)
    return m


def _norm(c, g):
    from mote_amd.norm import RMSNorm

    n = RMSNorm(c["d"], device="cuda")
    with torch.no_grad():
        n.weight.copy_(1.0 + 0.1 * torch.randn(c["d"], generator=g, device="cuda"))
    return n


def _capture(fn):
    """fn() as a HIP graph: (the graph, its static outputs)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = fn()
    return graph, out


def _prepare_block(c, g):
    dt = torch.float32 if c["dtype"] == "fp32" else torch.bfloat16
    B, T, d = c["batch"], c["T"], c["d"]
    st = {"case": c, "norm": _norm(c, g), "mixer": _relation(c, g, int(c["odd"]))}
    st["x"] = _randn(g, B, T, d, dtype=dt).requires_grad_(True)
    st["res"] = _randn(g, B, T, d).requires_grad_(True)
    # the gradient of a loss: noise, and a part along the layer's own values (wo wi y). Without that
    # part lam's gradient is a sum of random signs, near zero by chance.
    with torch.no_grad():
        m = st["mixer"]
        y = torch.nn.functional.rms_norm(st["x"].float() + st["res"], (d,), st["norm"].weight)
        own = torch.nn.functional.linear(torch.nn.functional.linear(y, m.wi.weight), m.wo.weight)
        st["dout"] = (_randn(g, B, T, d) + 0.5 * own).to(dt)
    st["ds"] = _randn(g, B, T, d)
    st["leaves"] = [st["x"], st["res"], st["norm"].weight, *st["mixer"].parameters()]
    if c["graph"]:
        st["graph"], st["out"] = _capture(lambda: _step_block(st))
    return st


def _step_block(st):
    c = st["case"]
    # cache_enabled off: a captured step casts the weights on every replay, as an eager step does once
    with torch.autocast("cuda", torch.bfloat16, enabled=c["dtype"] == "bf16", cache_enabled=not c["graph"]):
        y, s = st["norm"](st["x"], st["res"], prenorm=True)
        out = st["mixer"](y)
    grads = torch.autograd.grad((out, s), st["leaves"], (st["dout"], st["ds"]))
    return [out, s, *grads]


def _lengths(c):
    """Sequence lengths, spread evenly over the range in a fixed order (the same for every seed, so
    that a case is one amount of work)."""
    n = c["batch"]
    step = (c["high"] - c["low"]) / max(1, n - 1)
    order = sorted(range(n), key=lambda i: (i * 5) % (n + 1))
    return [c["low"] + int(round(step * i)) for i in order]


def _prepare_prefill(c, g):
    H = WIDTHS[c["d"]]
    lens = _lengths(c)
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32).cuda()
    rows = sum(lens)
    # projections of a normalised stream, token-major as the prologue leaves them
    p = [_randn(g, rows, H, c["d"] // H, dtype=torch.bfloat16, scale=0.577).permute(1, 0, 2) for _ in range(3)]
    return {"p": p, "lam": torch.tensor(0.5, device="cuda"), "cu": cu, "lens": lens}


def _prepare_extend(c, g):
    from mote_amd.arena import ArenaState, RelationArena

    H, B = WIDTHS[c["d"]], c["batch"]
    m = _relation(c, g, 0).bfloat16().requires_grad_(False)
    cap = -(-(c["S"] + c["T"] + 1) // 256) * 256
    arena = RelationArena(1, H, cap, c["d"] // H, "cuda", torch.bfloat16, batch=B)
    arena.store[..., : c["S"], :] = _randn(g, 1, 2, B, H, c["S"], c["d"] // H, dtype=torch.bfloat16, scale=0.577)
    return {"case": c, "mixer": m, "arena": arena, "layer": ArenaState(arena, n=c["S"])[0],
            "x": _randn(g, B, c["T"], c["d"], dtype=torch.bfloat16)}


def _prepare_decode(c, g):
    from mote_amd.arena import RelationArena
    from mote_amd.graph import RelationMainStep

    H, B, n = WIDTHS[c["d"]], c["batch"], c["layers"]
    cap = -(-(c["S"] + 257) // 256) * 256
    arena = RelationArena(n, H, cap, c["d"] // H, "cuda", torch.bfloat16, batch=B)
    for li in range(n):
        arena.store[li, ..., : c["S"], :] = _randn(g, 2, B, H, c["S"], c["d"] // H, dtype=torch.bfloat16, scale=0.577)
    mixers = [_relation(c, g, li).requires_grad_(False) for li in range(n)]
    norms = [_norm(c, g).requires_grad_(False) for _ in range(n)]
    for m in mixers:
        for lin in (m.w1, m.w2, m.wi, m.wo):
            lin.to(torch.bfloat16)
    S = torch.full((B,), c["S"], device="cuda", dtype=torch.int64)
    xm = torch.zeros(n, B, device="cuda")
    # the position stays where it is (an engine that moves S between replays), so that every pass is
    # the same token: it writes the same cache row again
    step = RelationMainStep(arena, S, xm_dev=xm, advance=False)
    x = _randn(g, B, 1, c["d"], dtype=torch.bfloat16)
    res0 = _randn(g, B, 1, c["d"])
    st = {"case": c, "arena": arena, "mixers": mixers, "norms": norms, "x": x, "res0": res0, "xm": xm, "step": step}

    def token():
        h, res = x, res0
        for li in range(n):
            y, res = norms[li](h, res, prenorm=True)
            h = step(mixers[li], y, li=li)
        return h, res

    with torch.no_grad():
        st["graph"], (h, res) = _capture(token)
    st["out"] = [h, res, xm, arena.store[..., c["S"], :]]  # the arena's own rows at S, appended by the step
    return st


def _prepare_chunk(c, g):
    from mote_amd.dc import ChunkLayer, DeChunkLayer

    B, Ln, d = c["batch"], c["L"], c["d"]
    mask = torch.rand(B, Ln, generator=g, device="cuda") < 1.0 / 3.3
    mask[:, 0] = True
    p = torch.rand(B, Ln, generator=g, device="cuda") * 0.5
    p = torch.where(mask, 0.5 + p, p)  # a router puts a boundary where p is over a half
    return {"chunk": ChunkLayer(bucket=64), "dechunk": DeChunkLayer(d), "mask": mask,
            "prob": torch.stack([1 - p, p], -1).requires_grad_(True),
            "x": _randn(g, B, Ln, d, dtype=torch.bfloat16).requires_grad_(True),
            "dout": _randn(g, B, Ln, d, dtype=torch.bfloat16)}


def prepare(case, seed):
    make = {"block": _prepare_block, "prefill": _prepare_prefill, "extend": _prepare_extend,
            "decode": _prepare_decode, "chunk": _prepare_chunk}[case["kind"]]
    return dict(make(case, _gen(seed)), kind=case["kind"])


# ---- one pass --------------------------------------------------------------------------------------
def run(st):
    kind = st["kind"]
    if kind == "prefill":
        from mote_amd.flash_relation import flash_relation_varlen

        return flash_relation_varlen(*st["p"], st["lam"], st["cu"], max(st["lens"]))
    if kind == "extend":
        c = st["case"]
        with torch.no_grad():
            out = st["mixer"](st["x"], cache=st["layer"])
        return [out, st["arena"].store[..., c["S"]: c["S"] + c["T"], :]]  # the arena's own new rows
    if kind == "chunk":
        rows, _ = st["chunk"](st["x"], st["mask"])
        out = st["dechunk"](rows, st["mask"], st["prob"])
        return [out, *torch.autograd.grad(out, (st["x"], st["prob"]), st["dout"])]
    if "graph" in st:
        st["graph"].replay()
        return st["out"]
    return _step_block(st)


# ---- what a pass cannot do without -----------------------------------------------------------------
def work(case):
    c, d = case, case["d"]
    if c["kind"] == "block":
        rows, es = c["batch"] * c["T"], 4 if c["dtype"] == "fp32" else 2
        mats = 5 if c["gate"] else 4
        flops = 6.0 * rows * d * d * mats + 7.0 * c["batch"] * d * c["T"] ** 2
        # x, dout, out, dx; residual, its gradient, the stream and its gradient; weights and theirs
        return {"flops": flops, "bytes": rows * d * (4 * es + 4 * 4) + mats * d * d * 8.0}
    if c["kind"] == "prefill":
        lens = _lengths(c)
        return {"flops": 2.0 * d * sum(n * n for n in lens), "bytes": sum(lens) * (4.0 * d * 2 + 4 * WIDTHS[d])}
    if c["kind"] == "extend":
        pairs = c["T"] * (c["S"] + c["T"] / 2)
        return {"flops": c["batch"] * (8.0 * c["T"] * d * d + 4.0 * d * pairs),
                "bytes": c["batch"] * (2.0 * (c["S"] + c["T"]) * d * 2 + 2.0 * c["T"] * d * 2) + 8.0 * d * d}
    if c["kind"] == "decode":
        cache = 2.0 * c["batch"] * (c["S"] + 1) * d * 2
        return {"flops": c["layers"] * c["batch"] * (8.0 * d * d + 4.0 * d * c["S"]), "bytes": c["layers"] * (cache + 8.0 * d * d)}
    # bytes' states and gradients in and out, the mask and the probabilities with their gradient
    return {"flops": 8.0 * c["batch"] * c["L"] * d, "bytes": c["batch"] * c["L"] * (4.0 * d * 2 + 1 + 16)}


def tolerance(case):
    if case["kind"] == "block":
        return {"rel": 1e-5} if case["dtype"] == "fp32" else {"rel": 2.5e-2, "max": 0.5}
    if case["kind"] == "decode":
        return {"rel": 2.5e-2, "max": 0.5}
    return {"rel": 1.2e-2, "max": 0.2}


# ---- the same in 64 bits ---------------------------------------------------------------------------
def _core64(p1, p2, info, lam, S=0, tau=2.0):
    """[T, dh] queries at positions S.. against [S + T, dh] rows: (Y, exchange mass)."""
    T, n = p1.shape[0], p2.shape[0]
    u = p1 @ p2.t() / math.sqrt(p1.shape[1])
    i = torch.arange(S, S + T, device=u.device)[:, None]
    j = torch.arange(n, device=u.device)[None]
    score = torch.nn.functional.silu(u) - lam * torch.log((i + 1).double())
    score = torch.where(j == i, torch.sigmoid(u / tau), score).masked_fill(j > i, float("-inf"))
    f = torch.softmax(score, -1)
    return f @ info, 1 - f[torch.arange(T, device=u.device), torch.arange(S, S + T, device=u.device)]


def _rms64(x, w, eps=1e-5):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _rope64(x, pos0):
    """[B, T, H, dh] rotated at positions pos0..; the angles are the fp32 products of the tables."""
    T, dh = x.shape[1], x.shape[3]
    inv = 1.0 / (10000.0 ** (torch.arange(0, dh, 2, dtype=torch.float32) / dh))
    a = (torch.arange(pos0, pos0 + T, dtype=torch.float32)[:, None] * inv[None]).cuda().double()[:, None]
    lo, hi = x[..., : dh // 2], x[..., dh // 2:]
    return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin()], -1)


def _givens64(x, theta, layer):
    H = x.shape[2]
    a = torch.arange(layer % 2, H, 2, device=x.device)
    b = (a + 1) % H
    c, s = theta.cos()[:, None], theta.sin()[:, None]
    out = torch.empty_like(x)
    out = out.index_copy(2, a, c * x[:, :, a] - s * x[:, :, b])
    return out.index_copy(2, b, s * x[:, :, a] + c * x[:, :, b])


def _heads64(P, x, H, layer, pos0, norm):
    B, T, d = x.shape
    q, k, v = (torch.matmul(x, P[n + ".weight"].t().contiguous()).view(B, T, H, d // H) for n in ("w1", "w2", "wi"))
    if norm:
        q, k = _rms64(q, P["p1_norm.weight"]), _rms64(k, P["p2_norm.weight"])
    return _rope64(q, pos0), _rope64(k, pos0), _givens64(v, P["theta"], layer)


def _exact_block(c, seed):
    st = prepare(dict(c, graph=False), seed)
    H = WIDTHS[c["d"]]
    names = ["x", "res", "norm", *[n for n, _ in st["mixer"].named_parameters()]]
    P = {n: t.detach().double().requires_grad_(True) for n, t in zip(names, st["leaves"])}
    s = P["x"] + P["res"]
    y = _rms64(s, P["norm"])
    q, k, v = _heads64(P, y, H, int(c["odd"]), 0, c["norm"])
    B, T = c["batch"], c["T"]
    rows = []
    for b in range(B):
        rows.append(torch.stack([_core64(q[b, :, h], k[b, :, h], v[b, :, h], P["lam"])[0] for h in range(H)], 1))
    z = torch.stack(rows).reshape(B, T, c["d"])
    if c["gate"]:
        z = z * torch.sigmoid(torch.matmul(y, P["wg.weight"].t().contiguous()))
    out = torch.matmul(z, P["wo.weight"].t().contiguous())
    grads = torch.autograd.grad((out, s), [P[n] for n in names], (st["dout"].double(), st["ds"].double()))
    return [out, s, *grads]


def _exact_chunk(c, seed):
    st = prepare(c, seed)
    x, prob = (st[n].detach().double().requires_grad_(True) for n in ("x", "prob"))
    mask = st["mask"]
    B, Ln = mask.shape
    p = prob[..., 1].clamp(1e-4, 1 - 1e-4)
    order = torch.argsort(torch.arange(Ln, device="cuda")[None] + (~mask).long() * Ln, dim=1)
    order = order[:, : int(mask.sum(1).max())]
    rows = torch.gather(x, 1, order[:, :, None].expand(-1, -1, c["d"]))
    pm = torch.gather(p, 1, order)[..., None]
    z, zs = torch.zeros(B, c["d"], device="cuda", dtype=torch.float64), []
    for xm, qm in zip(rows.unbind(1), pm.unbind(1)):
        z = z + qm * (xm - z)
        zs.append(z)
    at = mask.long().cumsum(1) - 1
    out = torch.gather(torch.stack(zs, 1), 1, at[:, :, None].expand(-1, -1, c["d"]))
    return [out, *torch.autograd.grad(out, (x, prob), st["dout"].double())]


def _exact_prefill(c, seed):
    st = prepare(c, seed)
    ys, gs, r = [], [], 0
    for n in st["lens"]:
        one = [_core64(*(t[h, r: r + n].double() for t in st["p"]), st["lam"].double()) for h in range(WIDTHS[c["d"]])]
        ys.append(torch.stack([a for a, _ in one]))
        gs.append(torch.stack([b for _, b in one]))
        r += n
    return [torch.cat(ys, 1), torch.cat(gs, 1)]


def _layer64(c, m, layer, x, cache, S):
    """One layer's new rows after a cached prefix [2, B, H, S, dh]: (out, exchange mass [B, H, T], the
    rows it appends [2, B, H, T, dh])."""
    P = {n: t.detach().double() for n, t in m.named_parameters()}
    H, (B, T, d) = WIDTHS[c["d"]], x.shape
    q, k, v = (t.transpose(1, 2) for t in _heads64(P, x, H, layer, S, False))
    ys, gs = [], []
    for b in range(B):
        one = [_core64(q[b, h], torch.cat([cache[0, b, h].double(), k[b, h]]), torch.cat([cache[1, b, h].double(), v[b, h]]),
                       P["lam"], S) for h in range(H)]
        ys.append(torch.stack([a for a, _ in one], 1))
        gs.append(torch.stack([e for _, e in one]))
    out = torch.matmul(torch.stack(ys).reshape(B, T, d), P["wo.weight"].t().contiguous())
    return out, torch.stack(gs), torch.stack([k, v])


def _exact_extend(c, seed):
    st = prepare(c, seed)
    out, _, rows = _layer64(c, st["mixer"], 0, st["x"].double(), st["arena"].store[0, ..., : c["S"], :], c["S"])
    return [out, rows[None]]


def _exact_decode(c, seed):
    st = prepare(c, seed)
    h, res, xm, rows = st["x"].double(), st["res0"].double(), [], []
    for li, (m, n) in enumerate(zip(st["mixers"], st["norms"])):
        res = res + h
        y = _rms64(res, n.weight.double())
        h, g, new = _layer64(c, m, li, y, st["arena"].store[li, ..., : c["S"], :], c["S"])
        xm.append(g[..., 0].mean(1))
        rows.append(new[..., 0, :])
    return [h, res, torch.stack(xm), torch.stack(rows)]


def exact(case, seed):
    return {"block": _exact_block, "prefill": _exact_prefill, "extend": _exact_extend, "decode": _exact_decode,
            "chunk": _exact_chunk}[case["kind"]](case, seed)
