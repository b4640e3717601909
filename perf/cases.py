"""The work this package is used for, as measurable cases: one pass of each goes through the public entry points as a
caller's program does, on inputs made from a seed.

Four kinds of program:
  step      serving: one pass of the whole hot path on rank 0 (pipeline.DispatchPipeline), every buffer allocated up front --
            route, count and pack as a source, row map, grouped expert MLP and return as a destination, combine as a source --
            either enqueued stage by stage ("eager") or replayed as one HIP graph ("graph")
  train     one training pass of the expert MLP on expert-major rows (layers.expert_mlp): forward, backward to the rows and
            all weights, and, where the case says so, an in-place update of the weights (so that the kernels' own copies of
            them are made anew on every pass)
  dispatch  one training pass of the data movement around the experts: routing, counting, the fixed-capacity pack and the
            weighted combine (layers.pack_fixed_m, layers.combine), forward and backward
  flow      the original operator chain under its own names (route_and_pack_padding_free, custom_a2a, shuffle, expert) with
            padding-free payloads
The named sizes are those of configs.CONFIGS and of the sweep driver (benchmark.py); the ranges of draw() surround them.
"""
from __future__ import annotations

import math

import torch

from iris_testing_amd import harness, ops
from iris_testing_amd.configs import MoEConfig
from iris_testing_amd.layers import ExpertWeights, combine, custom_a2a, expert, expert_mlp, pack_fixed_m, shuffle
from iris_testing_amd.layers.all_to_all import SimulatedWorld, simulated_world
from iris_testing_amd.pipeline import DispatchPipeline
from iris_testing_amd.utils import alloc_counts_buffers, alloc_token_buffers, compute_capacity_from_pca, route_and_pack_padding_free

DEV = "cuda"


# ---- the cases ------------------------------------------------------------------------------------------------------------
def _step(tokens, hidden, dtype, experts, topk, world, ffn, act, bias="none", mode="fixed", launch="eager", name=None):
    """dtype: f32 | bf16 | fp8 (fp8 experts on bf16 tokens); bias: what skews the routing (none | normal | zipf); mode: the
    layout the rows travel in (fixed [W,M,H] slots | gated: their gates with them | flat: padding-free)."""
    c = dict(kind="step", tokens=tokens, hidden=hidden, dtype=dtype, experts=experts, topk=topk, world=world, ffn=ffn, act=act,
             bias=bias, mode=mode, launch=launch)
    return c if name is None else dict(c, name=name)


def _train(rows, hidden, experts, ffn, act, skew, update, name=None):
    """skew: exponent of the power law the rows are spread over the local experts with (0: evenly)."""
    c = dict(kind="train", rows=rows, hidden=hidden, experts=experts, ffn=ffn, act=act, skew=skew, update=update)
    return c if name is None else dict(c, name=name)


def _dispatch(tokens, hidden, experts, topk, world, bias, name=None):
    c = dict(kind="dispatch", tokens=tokens, hidden=hidden, experts=experts, topk=topk, world=world, bias=bias)
    return c if name is None else dict(c, name=name)


def _flow(tokens, hidden, experts, topk, world, ffn, name=None):
    c = dict(kind="flow", tokens=tokens, hidden=hidden, experts=experts, topk=topk, world=world, ffn=ffn)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # the fp32 plumbing workload: the smallest step, all launches and host work
        _step(256, 256, "f32", 8, 2, 4, 512, "gelu", name="step plumbing"),
        # small messages, top-1: a latency-bound serving step, replayed as a graph
        _step(512, 2048, "bf16", 16, 1, 8, 4096, "silu", launch="graph", name="step small"),
        # few large experts, long prompts: the headline serving step (prefill)
        _step(16384, 4096, "bf16", 8, 2, 8, 14336, "swiglu", name="step mixtral"),
        # many small experts with uneven popularity (prefill)
        _step(4096, 7168, "bf16", 256, 8, 8, 2048, "swiglu", bias="normal", name="step finegrained"),
        # the same experts while generating: two dozen sequences per rank, one token each (decode)
        _step(24, 7168, "bf16", 256, 8, 8, 2048, "swiglu", bias="normal", launch="graph", name="step finegrained decode"),
        # fp8 experts under skewed routing, eight experts a token
        _step(8192, 2048, "fp8", 60, 8, 4, 1408, "swiglu", bias="zipf", name="step zipf_k8"),
        # the same model on a short odd batch, two experts a token, rows sent without padding
        _step(777, 2048, "fp8", 60, 2, 4, 1408, "swiglu", bias="zipf", mode="flat", launch="graph", name="step zipf_k2 short"),
        # training pass of one large expert on what its rank receives (a micro-batch: the weights stay)
        _train(32768, 4096, 1, 14336, "swiglu", 0.0, False, name="train mixtral"),
        # training step of 32 small experts with uneven row counts, weights updated
        _train(33618, 7168, 32, 2048, "swiglu", 0.8, True, name="train finegrained"),
        # a small odd training batch of two-layer experts
        _train(1003, 2048, 2, 4096, "silu", 0.5, False, name="train small"),
        # forward and backward of the row movement at the fine-grained model's sizes
        _dispatch(4096, 7168, 256, 8, 8, "normal", name="dispatch finegrained"),
        # the operator chain at the sizes of the original's own figures (batch 4, sequence 2048, 32 experts a rank)
        _flow(8192, 768, 256, 2, 8, 768, name="flow figures"),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, round(v / step) * step)))


def draw(rng):
    top = work(listed()[7])  # (no drawn case costs more than the largest listed one)
    while True:
        kind = rng.choice(["step"] * 5 + ["train"] * 3 + ["dispatch", "flow"])
        world = rng.choice([4, 8])
        e_local = rng.choice([1, 2, 4, 8, 15, 32])
        experts = world * e_local
        topk = rng.choice([k for k in (1, 2, 4, 8) if k <= experts // 2])
        if kind == "step":
            dtype = rng.choice(["bf16"] * 5 + ["fp8"] * 4 + ["f32"])
            bias = rng.choice(["none", "normal", "zipf"])
            launch = rng.choice(["eager", "graph"])
            if dtype == "f32":
                c = _step(_log(rng, 32, 1024), _log(rng, 128, 512, 4), dtype, experts, topk, world, _log(rng, 128, 1024, 4),
                          rng.choice(["gelu", "silu"]), bias, "fixed", launch)
            else:
                q = 128 if dtype == "fp8" else 64
                c = _step(_log(rng, 16, 16384), _log(rng, 512, 7168, q), dtype, experts, topk, world, _log(rng, 512, 14336, q),
                          "swiglu" if dtype == "fp8" else rng.choice(["swiglu", "swiglu", "silu", "gelu"]), bias,
                          rng.choice(["fixed"] * 4 + ["gated", "flat"]), launch)
        elif kind == "train":
            c = _train(_log(rng, 256, 32768), _log(rng, 512, 7168, 64), e_local, _log(rng, 512, 14336, 64),
                       rng.choice(["swiglu", "swiglu", "silu", "gelu"]), rng.choice([0.0, 0.5, 1.0]), rng.random() < 0.5)
        elif kind == "dispatch":
            c = _dispatch(_log(rng, 64, 16384), _log(rng, 512, 7168, 8), experts, topk, world, rng.choice(["none", "normal"]))
        else:
            c = _flow(_log(rng, 128, 16384), _log(rng, 512, 4096, 64), experts, topk, world, _log(rng, 512, 4096, 64))
        w = work(c)
        if w["flops"] <= 0.5 * top["flops"] and w["bytes"] <= 8e9 and (kind != "step" or _share(c)[1] * c["hidden"] < 1 << 30):
            return c


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------
def _share(c):
    """(rows rank 0 receives, rows of the [W,M] layout, local experts that receive any) to be expected: what the routing of
    N(0,1) logits under the case's bias makes of them, by a fixed sample."""
    E, W, k, T = c["experts"], c["world"], c["topk"], c["tokens"]
    g = torch.Generator().manual_seed(1)
    z = torch.randn(2048, E, generator=g)
    b = _bias(c.get("bias", "none"), E, 2)
    sel = torch.topk(z if b is None else z + b, k).indices
    per_rank = torch.bincount((sel // (E // W)).reshape(-1), minlength=W).double() / sel.shape[0]
    p = torch.bincount(sel.reshape(-1), minlength=E)[: E // W].double() / sel.shape[0]
    hit = float((1 - (1 - p) ** (T * W)).sum())
    return max(1.0, float(per_rank[0]) * T * W), max(1.0, float(per_rank.max()) * T) * W, max(1.0, hit)


def work(case):
    c = case
    H = c["hidden"]
    if c["kind"] == "train":
        S, E_l, F = c["rows"], c["experts"], c["ffn"]
        n = 3 if c["act"] == "swiglu" else 2
        params = E_l * n * H * F
        # rows, their gradient and the result's, in and out; weights read, their gradients written; with the update the
        # weights read again and written
        return {"bytes": 2 * (4 * S * H + 2 * params + (2 * params if c["update"] else 0)), "flops": 6.0 * S * H * F * n}
    T, E, k = c["tokens"], c["experts"], c["topk"]
    S, slots, hit = _share(c)  # (the weights of an expert without rows are not needed)
    if c["kind"] == "dispatch":
        # tokens, router -> logits, choice; send buffer; returned rows and result; then the gradients of all of them
        return {"bytes": 2 * (T * H + H * E + slots * H + T * k * H + T * H) + 4 * T * E + 8 * T * k
                + 2 * (T * k * H + T * H) + 2 * (T * H + T * k * H + slots * H) + 4 * T * k, "flops": 2.0 * T * H * E}
    if c["kind"] == "flow":
        F = c["ffn"]
        # tokens, router -> payload; payloads -> receive layout (padded to its largest block) -> rows -> expert
        return {"bytes": 2 * (T * H + H * E + T * k * H + S * H + slots * H + 2 * S * H + hit * H * F + S * F),
                "flops": 2.0 * T * H * E + 2.0 * S * H * F}
    B, F = (4 if c["dtype"] == "f32" else 2), c["ffn"]
    n = 3 if c["act"] == "swiglu" else 2
    row = 1 if c["dtype"] == "fp8" and c["mode"] != "flat" else B  # (bytes of a row element on its way to the expert)
    out_rows = T * k if c["mode"] == "flat" else slots
    ret_rows = S if c["mode"] == "flat" else slots
    return {"bytes": T * H * B + H * E * B + 4 * T * E + 8 * T * k + out_rows * H * row + S * H * row
            + hit * n * H * F * (1 if c["dtype"] == "fp8" else B) + ret_rows * H * B + T * k * H * B + T * H * B,
            "flops": 2.0 * S * H * F * n + 2.0 * T * H * E}


def tolerance(case):
    if case["kind"] == "step" and case["dtype"] == "f32":
        return {"rel": 1e-5}  # fp32 sums in another order
    if case["kind"] == "step" and case["dtype"] == "fp8":
        # one bf16 rounding of the result, and now and then a neighbouring fp8 code of a hidden value
        return {"rel": 1e-2, "max": 0.3}
    # bf16 results of fp32 sums; every choice, count and position is a whole number and stays what it is
    return {"rel": 1e-2, "max": 0.1}


# ---- inputs ---------------------------------------------------------------------------------------------------------------
def _gen(seed, k):
    return torch.Generator(device=DEV).manual_seed(seed * 1000003 + k)


def _bias(kind, E, seed):
    if kind == "none":
        return None
    if kind == "normal":
        return torch.randn(E, generator=torch.Generator().manual_seed(seed * 7919 + 5))
    p = torch.arange(1, E + 1, dtype=torch.float64) ** -1.2
    return torch.log(p / p.sum()).float()


def _normal(g, shape, dtype, scale=1.0):
    t = torch.randn(shape, generator=g, device=DEV, dtype=dtype)
    return t if scale == 1.0 else t.mul_(scale)


def _weight(g, E_l, i, o, dtype):
    return _normal(g, (E_l, i, o), dtype, i ** -0.5)


def _routing(c, seed, dtype):
    """Token shards of all ranks, the router and what every rank makes of its shard.  The seed deals a fixed set of N(0,1)
    tokens out in another order, and flips the sign of other columns (of tokens and router alike): other inputs everywhere,
    with the same number of rows for every expert, so that all shapes are those of the case."""
    T, H, E, W = c["tokens"], c["hidden"], c["experts"], c["world"]
    cfg = MoEConfig("case", seed, T, H, "f32" if dtype == torch.float32 else "bf16", E, c["topk"], W, c.get("ffn", H),
                    c.get("act", "silu"), quant="fp8" if c.get("dtype") == "fp8" else "none")
    sign = torch.randint(0, 2, (H,), generator=_gen(seed, 1), device=DEV).mul_(2).sub_(1).to(dtype)
    router = _normal(_gen(0, 1), (H, E), dtype, H ** -0.5).mul_(sign[:, None])
    bias = _bias(c.get("bias", "none"), E, 2)  # (the popularity of the experts belongs to the model, not to the batch)
    bias = None if bias is None else bias.to(DEV)
    shards = [_normal(_gen(0, 10 + s), (T, H), dtype)[torch.randperm(T, generator=_gen(seed, 10 + s), device=DEV)].mul_(sign)
              for s in range(W)]
    routes = [harness.route_shard(cfg, x, router, bias) for x in shards]
    caps = torch.stack([r.counts.caps for r in routes]).amax(0).tolist()
    return cfg, router, bias, shards, routes, int(caps[0]), int(caps[1])


def _prepare_step(c, seed):
    dtype = torch.float32 if c["dtype"] == "f32" else torch.bfloat16
    cfg, router, bias, shards, routes, M, CAP = _routing(c, seed, dtype)
    W, H, F, E_l, T, k = cfg.world, cfg.hidden, cfg.ffn, cfg.e_local, cfg.tokens, cfg.topk
    recv = torch.empty((W, M, H), dtype=dtype, device=DEV)
    recv_counts = torch.stack([r.counts.send_counts[0] for r in routes]).contiguous()
    for s in range(W):
        harness.pack_for_dst(shards[s], routes[s], 0, M, out=recv[s])
    per_src = recv_counts.sum(1).tolist()
    S = sum(per_src)
    world = harness.World(cfg, router, bias, shards[0], routes[:1], M, CAP, recv, recv_counts, S)
    g = _gen(seed, 2)
    if c["dtype"] == "fp8":
        q, sc = ops.quantize_rows_fp8(recv.view(W * M, H))
        world.recv_q, world.recv_scale = q.view(W, M, H), sc.view(W, M)
        qs = [harness.quantize_weight_fp8(_weight(g, E_l, i, o, dtype)) for i, o in ((H, F), (H, F), (F, H))]
        ew = ExpertWeights.prepare_fp8(qs[0][0], qs[0][1], qs[1][0], qs[1][1], qs[2][0], qs[2][1])
    elif c["act"] == "swiglu":
        wg, wu, wd = _weight(g, E_l, H, F, dtype), _weight(g, E_l, H, F, dtype), _weight(g, E_l, F, H, dtype)
        ew = ExpertWeights.prepare("swiglu", wg, wd, wu)
    else:
        ew = ExpertWeights.prepare(c["act"], _weight(g, E_l, H, F, dtype), _weight(g, E_l, F, H, dtype))
    flat, gated = c["mode"] == "flat", c["mode"] == "gated"
    pipe = DispatchPipeline(
        world, ew, returned=_normal(_gen(seed, 3), (T * k, H) if flat else (W, M, H), dtype), gated=gated, padding_free=flat,
        recv_gate=torch.rand((W, M), generator=_gen(seed, 4), device=DEV) if gated else None,
        recv_flat=torch.cat([recv[s, :n] for s, n in enumerate(per_src)]) if flat else None)
    return {"pipe": pipe, "graph": pipe.capture() if c["launch"] == "graph" else None}


def _run_step(s):
    p = s["pipe"]
    if s["graph"] is not None:
        s["graph"].replay()
    else:
        p.step()
    sent = p.payload if p.padding_free else p.send_q if p.fp8_dispatch else p.send
    out = {"logits": p.logits, "idx": p.idx, "gate": p.gate, "counts": p.send_counts, "offsets": p.expert_offs, "sizes": p.dst_sizes,
           "starts": p.dst_offsets, "caps": p.caps, "pos": p.pos, "sent": sent, "expert_rows": p.expert_cnt,
           "ret": p.ret_flat if p.padding_free else p.ret, "out": p.out}
    if p.fp8_dispatch:
        out["sent_scale"] = p.send_scale
    if p.gated:
        out["sent_gate"] = p.send_gate
    return out


def _row_counts(S, E_l, skew, seed):
    """S rows spread over the local experts by a power law, in an order that depends on the seed."""
    p = torch.arange(1, E_l + 1, dtype=torch.float64) ** -skew
    p = p[torch.randperm(E_l, generator=torch.Generator().manual_seed(seed))] / p.sum()
    edge = torch.round(torch.cumsum(p, 0) * S).to(torch.int64)
    edge[-1] = S
    return torch.diff(edge, prepend=torch.zeros(1, dtype=torch.int64)).to(torch.int32).to(DEV)


def _prepare_train(c, seed):
    S, H, E_l, F, dt = c["rows"], c["hidden"], c["experts"], c["ffn"], torch.bfloat16
    g = _gen(seed, 2)
    w = [_weight(g, E_l, H, F, dt), _weight(g, E_l, F, H, dt)] + ([_weight(g, E_l, H, F, dt)] if c["act"] == "swiglu" else [])
    for t in w:
        t.requires_grad_()
    x = _normal(_gen(seed, 3), (S, H), dt).requires_grad_()
    dy = _normal(_gen(seed, 4), (S, H), dt, 0.01)
    return {"x": x, "dy": dy, "w": w, "ew": ExpertWeights.prepare(c["act"], *w), "cnt": _row_counts(S, E_l, c["skew"], seed),
            "lr": 1e-4 if c["update"] else None}


def _run_train(s):
    x, w = s["x"], s["w"]
    x.grad = None
    for t in w:
        t.grad = None
    y = expert_mlp(x, s["ew"], s["cnt"])
    y.backward(s["dy"])
    out = {"y": y.detach(), "dx": x.grad, "dw": [t.grad for t in w]}
    if s["lr"] is not None:
        with torch.no_grad():
            for t in w:
                t.add_(t.grad, alpha=-s["lr"])
        out["w"] = [t.detach() for t in w]
    return out


def _prepare_dispatch(c, seed):
    cfg, router, bias, shards, routes, M, _ = _routing(c, seed, torch.bfloat16)
    W, T, H = cfg.world, cfg.tokens, cfg.hidden
    return {"x": shards[0].requires_grad_(), "router": router, "bias": bias, "M": M, "W": W, "E": cfg.experts, "k": cfg.topk,
            "returned": _normal(_gen(seed, 3), (W, M, H), torch.bfloat16).requires_grad_(),
            "d_send": _normal(_gen(seed, 4), (W, M, H), torch.bfloat16), "d_out": _normal(_gen(seed, 5), (T, H), torch.bfloat16)}


def _run_dispatch(s):
    x, returned, e_l = s["x"], s["returned"], s["E"] // s["W"]
    x.grad = returned.grad = None
    idx, gate, logits = ops.route_topk(x.detach(), s["router"], s["k"], s["bias"])
    gate.requires_grad_()
    n = ops.count_and_offsets(idx, s["E"], s["W"])
    send = pack_fixed_m(x, idx, n.pos, n.dst_sizes, n.dst_offsets, e_l, s["M"])
    out = combine(returned, idx, n.pos, gate, n.dst_offsets, e_l)
    torch.autograd.backward([send, out], [s["d_send"], s["d_out"]])
    return {"logits": logits, "idx": idx, "gate": gate.detach(), "counts": n.send_counts, "sizes": n.dst_sizes, "pos": n.pos,
            "send": send.detach(), "out": out.detach(), "dx": x.grad, "d_returned": returned.grad, "d_gate": gate.grad}


def _prepare_flow(c, seed):
    W, E, k, H, dt = c["world"], c["experts"], c["topk"], c["hidden"], torch.bfloat16
    E_l = E // W
    _, router, _, shards, _, _, _ = _routing(c, seed, dt)
    world = SimulatedWorld(W, 0)
    counts = []
    for s, x in enumerate(shards):
        payload, n, starts, _ = route_and_pack_padding_free(x, router, k, W, E)
        counts.append(n)
        if s:
            world.post(s, payload, n, starts)
    cap = compute_capacity_from_pca(torch.stack(counts))
    cb, tb = alloc_counts_buffers(None, W, E_l), alloc_token_buffers(None, W, E_l, cap, H, dt)
    return {"x": shards[0], "router": router, "world": world, "cap": cap, "cb": cb, "tb": tb, "E": E, "W": W, "k": k,
            "w": _weight(_gen(seed, 2), E_l, H, c["ffn"], dt)}


def _run_flow(s):
    cb, tb = s["cb"], s["tb"]
    payload, n, starts, sizes = route_and_pack_padding_free(s["x"], s["router"], s["k"], s["W"], s["E"])
    with simulated_world(s["world"]):
        buf = custom_a2a(payload, n, starts, cb.pca, tb.token_buf, cb.counts_ready, tb.token_sync, cb.heap_bases, s["E"], s["cap"])
    rows = shuffle(buf, cb.pca, tb.token_sync)
    out = expert(rows, s["w"], cb.pca.sum(1, dtype=torch.int32), s["E"])
    return {"payload": payload, "counts": n, "starts": starts, "sizes": sizes, "pca": cb.pca, "buf": buf, "rows": rows, "out": out}


_PREPARE = {"step": _prepare_step, "train": _prepare_train, "dispatch": _prepare_dispatch, "flow": _prepare_flow}
_RUN = {"step": _run_step, "train": _run_train, "dispatch": _run_dispatch, "flow": _run_flow}


def prepare(case, seed):
    return dict(_PREPARE[case["kind"]](case, int(seed)), kind=case["kind"])


def run(state):
    return _RUN[state["kind"]](state)
