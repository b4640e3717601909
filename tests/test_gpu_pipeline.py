"""End to end on the two small workloads: every simulated rank's experts are run in turn on the one
GPU, the outputs returned and combined on rank 0, and the result compared with the dense closed
form  out[t] = sum_kk p[t, idx[t,kk]] * MLP_{idx[t,kk]}(x[t])  computed per token by the oracle."""
import numpy as np
import pytest
import torch

from helpers import O, assert_bits_equal, err_stats, to_np

pytestmark = pytest.mark.gpu

from iris_testing_amd import harness, ops  # noqa: E402
from iris_testing_amd.configs import CONFIGS, gen_expert_weights  # noqa: E402
from iris_testing_amd.layers.expert import expert_mlp  # noqa: E402

DEV = "cuda"


@pytest.mark.parametrize("name", ["plumbing", "small"])
def test_dispatch_expert_combine_matches_dense(name):
    cfg = CONFIGS[name]
    W, E_l = cfg.world, cfg.e_local
    world, shards = harness.build_world(cfg, DEV, keep_shards=True)
    M = world.M
    r0 = world.routes[0]

    # every destination rank d: receive, unpack, MLP with its own weights, pack the return buffer
    returned = torch.zeros((W, M, cfg.hidden), dtype=cfg.torch_dtype, device=DEV)
    raw_weights = []
    for d in range(W):
        recv = torch.stack([harness.pack_for_dst(shards[s], world.routes[s], d, M) for s in range(W)])
        rc = torch.stack([world.routes[s].counts.send_counts[d] for s in range(W)]).contiguous()
        S = int(rc.sum().item())
        rows, cnt = ops.unpack_expert_major(recv, rc, S)
        ew, raw, _ = harness.expert_weights(cfg, d, DEV)
        raw_weights.append(raw)
        y = expert_mlp(rows, ew, cnt)
        ret = ops.return_pack(y, rc, M)
        returned[d] = ret[0]  # the slot that goes back to source 0
    out = ops.combine(returned, r0.idx, r0.counts.pos, r0.gate, r0.counts.dst_offsets, E_l)

    # dense closed form on the CPU: every expert applied to the tokens that chose it
    x = to_np(shards[0])
    idx, gate = to_np(r0.idx), to_np(r0.gate)
    o_idx, o_gate, _ = O.route(x, to_np(world.router), cfg.topk, None)
    assert_bits_equal(idx, o_idx, "indices")
    want = np.zeros((cfg.tokens, cfg.hidden), dtype=np.float64)
    for ex in range(cfg.experts):
        d, el = divmod(ex, E_l)
        t_sel, k_sel = np.nonzero(o_idx == ex)
        if len(t_sel) == 0:
            continue
        w1, w2 = (to_np(w[el:el + 1]) for w in raw_weights[d])
        y = O.expert_mlp(x[t_sel], np.array([len(t_sel)]), w1, w2, cfg.act, cfg.dtype)
        want[t_sel] += o_gate[t_sel, k_sel][:, None].astype(np.float64) * y
    mx, mx_rms, rel = err_stats(to_np(out), want)
    print(f"{name}: end-to-end max-abs {mx:.3e}, max-abs/rms {mx_rms:.3e}, max-rel {rel:.3e}", flush=True)
    tol = 2.0 ** -6 if cfg.dtype == "bf16" else 1e-4
    assert mx_rms < tol * 4, f"end-to-end error {mx_rms} of rms"


@pytest.mark.parametrize("name,fused", [("small", False), ("small", True), ("zipf_k1", False)])
def test_graph_replay_equals_eager(name, fused):
    """The whole step captured as one HIP graph: every replay (with eager work and synchronisation in
    between, and outputs cleared before each replay) must reproduce the eager step bit for bit."""
    from iris_testing_amd.pipeline import DispatchPipeline
    cfg = CONFIGS[name]
    world = harness.build_world(cfg, DEV)
    ew, _, _ = harness.expert_weights(cfg, 0, DEV)
    pipe = DispatchPipeline(world, ew, fused=fused)
    pipe.returned.copy_(torch.randn(pipe.returned.shape, device=DEV).to(pipe.returned.dtype))
    pipe.step()
    torch.cuda.synchronize()
    names = ["idx", "gate", "send_counts", "pos", "send", "ret", "out"] + (["row_map"] if fused else ["rows", "y"])
    eager = {n: getattr(pipe, n).clone() for n in names}
    graph = pipe.capture()
    for rep in range(3):
        for n in names:
            getattr(pipe, n).zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for n in names:
            assert torch.equal(getattr(pipe, n), eager[n]), f"replay {rep}: {n} differs from the eager step"
        pipe.step()  # eager work between replays
        torch.cuda.synchronize()


@pytest.mark.parametrize("name,mode", [("plumbing", {}), ("small", dict(fused=False)), ("small", {}), ("small", dict(gated=True)),
                                       ("small", dict(padding_free=True)), ("zipf_k4", {}), ("zipf_k4", dict(fp8_dispatch=False)),
                                       ("zipf_k4", dict(gated=True)), ("zipf_k4", dict(padding_free=True))])
def test_step_as_one_call_equals_its_stages(name, mode):
    """step() is one library call; with events it runs stage by stage.  Every result must be the same bits."""
    from dataclasses import replace
    from iris_testing_amd.pipeline import DispatchPipeline
    cfg = CONFIGS[name]
    cfg = replace(cfg, tokens=min(cfg.tokens, 300))
    world = harness.build_world(cfg, DEV)
    ew, _, _ = harness.expert_weights(cfg, 0, DEV)
    if mode.get("gated"):
        mode = dict(mode, recv_gate=harness.recv_gates(world))
    if mode.get("padding_free"):
        mode = dict(mode, recv_flat=harness.recv_flat(world))
    pipe = DispatchPipeline(world, ew, **mode)
    pipe.returned.copy_(torch.randn(pipe.returned.shape, device=DEV).to(pipe.returned.dtype))
    names = [n for n in ("logits idx gate send_counts expert_offs dst_sizes dst_offsets caps pos row_token send send_gate payload send_q "
                         "send_scale expert_cnt row_map row_gate rows hidden y ret ret_flat xq xs hq hsc out").split()
             if isinstance(getattr(pipe, n, None), torch.Tensor)]
    def results(events):
        for n in names:
            getattr(pipe, n).zero_()
        pipe.step(events)
        torch.cuda.synchronize()
        return {n: getattr(pipe, n).clone() for n in names}
    one, stages = results(None), results([])
    for n in names:
        assert torch.equal(one[n], stages[n]), f"{n} differs"


@pytest.mark.parametrize("name,mode", [("plumbing", {}), ("small", dict(fused=False)), ("small", {}), ("small", dict(gated=True)),
                                       ("small", dict(padding_free=True)), ("zipf_k4", {}), ("zipf_k4", dict(fused=False)), ("zipf_k4", dict(fp8_dispatch=False)),
                                       ("zipf_k4", dict(gated=True)), ("zipf_k4", dict(padding_free=True))])
def test_step_of_a_rank_that_receives_nothing(name, mode):
    """No token of any rank chose an expert of this one: what it sends back is all padding, and its source side goes on as ever."""
    from dataclasses import replace
    from iris_testing_amd.pipeline import DispatchPipeline
    cfg = replace(CONFIGS[name], tokens=40)
    world = harness.build_world(cfg, DEV)
    ew, _, _ = harness.expert_weights(cfg, 0, DEV)
    world.recv_counts, world.S = torch.zeros_like(world.recv_counts), 0
    if mode.get("gated"):
        mode = dict(mode, recv_gate=harness.recv_gates(world))
    if mode.get("padding_free"):
        mode = dict(mode, recv_flat=harness.recv_flat(world))
    pipe = DispatchPipeline(world, ew, **mode)
    pipe.returned.copy_(torch.randn(pipe.returned.shape, device=DEV).to(pipe.returned.dtype))
    outs = []
    for events in (None, []):
        pipe.expert_cnt.fill_(7)
        if pipe.ret is not None:
            pipe.ret.fill_(3)
        pipe.out.zero_()
        pipe.step(events)
        torch.cuda.synchronize()
        outs.append(pipe.out.clone())
        assert not bool(pipe.expert_cnt.any()) and (pipe.ret is None or not bool(pipe.ret.any()))
    assert torch.equal(*outs) and bool(outs[0].any())


@pytest.mark.parametrize("T,H,E,k,W,F,act,cut", [(37, 128, 8, 2, 4, 260, "gelu", 0), (5, 36, 3, 1, 1, 100, "silu", 0), (300, 256, 130, 2, 65, 512, "silu", 3),
                                                 (2000, 132, 24, 4, 8, 200, "gelu", 40), (700, 512, 12, 2, 2, 1024, "silu", 1), (4, 64, 16, 1, 4, 64, "gelu", 0), (40, 252, 8, 2, 2, 130, "swiglu", -70)])
def test_fp32_rows_come_from_and_go_to_their_slots_in_the_gemms(T, H, E, k, W, F, act, cut):
    """In a step the GEMMs of fp32 experts move the rows; stage by stage copies stand before and behind them.  Tiles of 32 and 64 rows, one and
    two sets of waves, sources without rows, (cut > 0) rows past the pair capacity, which have no slot, (cut < 0) rows behind the total."""
    from iris_testing_amd.configs import MoEConfig
    from iris_testing_amd.pipeline import DispatchPipeline
    cfg = MoEConfig("case", T, T, H, "f32", E, k, W, F, act)
    world = harness.build_world(cfg, DEV)
    if cut < 0:
        world.S -= cut
    if cut > 0:
        M = max(world.M - cut, 1)
        world.M, world.recv = M, world.recv[:, :M].contiguous()
    ew, _, _ = harness.expert_weights(cfg, 0, DEV)
    pipe = DispatchPipeline(world, ew)
    names = "expert_cnt rows hidden y ret".split()

    def results(events):
        for n in names:
            getattr(pipe, n).fill_(3)
        pipe.step(events)
        torch.cuda.synchronize()
        return {n: getattr(pipe, n).clone() for n in names}
    one, stages = results(None), results([])
    for n in names:
        assert torch.equal(one[n], stages[n]), f"{n} differs"


@pytest.mark.parametrize("over", ["recv", "ret", "counts"])
def test_fp32_scratch_over_rows_that_are_done_with(over):
    """The hidden activation may lie where the received rows lay (they are unpacked first), and the returned buffer where the hidden activation
    or the counts per expert did: the step then keeps the copies."""
    from iris_testing_amd.configs import MoEConfig
    from iris_testing_amd.pipeline import DispatchPipeline
    cfg = MoEConfig("case", 7, 300, 256, "f32", 8, 2, 4, 128, "gelu")
    world = harness.build_world(cfg, DEV)
    ew, _, _ = harness.expert_weights(cfg, 0, DEV)
    pipe = DispatchPipeline(world, ew)
    pipe.step()
    torch.cuda.synchronize()
    want = {n: getattr(pipe, n).clone() for n in ("rows", "y", "ret")}
    if over == "counts":
        pipe.expert_cnt = pipe.ret.view(-1).view(torch.int32)[12:12 + cfg.e_local]
    else:
        pipe.hidden = (world.recv if over == "recv" else pipe.ret).view(-1)[:pipe.S * cfg.ffn].view(pipe.S, cfg.ffn)
    pipe.step()
    torch.cuda.synchronize()
    for n in want:
        assert torch.equal(getattr(pipe, n), want[n]), f"{n} differs"


@pytest.mark.parametrize("tokens,gated", [(40, False), (40, True), (1500, True)])
def test_rows_looped_back_on_one_rank_are_the_sent_ones(tokens, gated):
    """The receive side is prepared beside the ranking unless it reads what the source side writes: with one rank the received counts, rows and
    gates may be the sent buffers themselves, and the step has to give what it gives with copies of them."""
    from iris_testing_amd.configs import MoEConfig
    from iris_testing_amd.pipeline import DispatchPipeline
    cfg = MoEConfig("case", 5, tokens, 256, "bf16", 12, 2, 1, 256, "silu")
    world = harness.build_world(cfg, DEV)
    ew, _, _ = harness.expert_weights(cfg, 0, DEV)
    kw = dict(gated=True, recv_gate=harness.recv_gates(world)) if gated else {}
    pipe = DispatchPipeline(world, ew, **kw)
    names = "send_counts pos send expert_cnt row_map hidden ret".split()

    def results():
        for n in names:
            getattr(pipe, n).zero_()
        pipe.step()
        torch.cuda.synchronize()
        return {n: getattr(pipe, n).clone() for n in names}
    apart = results()
    assert torch.equal(apart["send"], world.recv) and torch.equal(apart["send_counts"], world.recv_counts)
    world.recv, world.recv_counts = pipe.send, pipe.send_counts
    if gated:
        pipe.recv_gate = pipe.send_gate
    back = results()
    for n in names:
        assert torch.equal(back[n], apart[n]), f"{n} differs"


@pytest.mark.parametrize("mode,shared", [("fp8", "rows counts scale"), ("fp8", "scale"), ("fp8", "counts"), ("fp8 gated", "rows counts scale gate"),
                                         ("fp8 gated", "gate"), ("gated", "gate"), ("flat", "rows counts"), ("flat", "counts"), ("fp8 flat", "rows counts")])
def test_one_rank_loops_some_of_its_buffers_back(mode, shared):
    """As above with fp8 rows and their scales, gates and padding-free payloads, all of them looped back or one alone; what the last step left in
    the shared buffers is wrong before each step."""
    from iris_testing_amd.configs import MoEConfig
    from iris_testing_amd.pipeline import DispatchPipeline
    fp8, gated, flat = "fp8" in mode, "gated" in mode, "flat" in mode
    cfg = MoEConfig("case", 5, 300, 256, "bf16", 12, 2, 1, 256, "swiglu" if fp8 else "silu", quant="fp8" if fp8 else "none")
    world = harness.build_world(cfg, DEV)
    ew, _, _ = harness.expert_weights(cfg, 0, DEV)
    kw = dict(gated=True, recv_gate=harness.recv_gates(world)) if gated else dict(padding_free=True, recv_flat=harness.recv_flat(world)) if flat else {}
    pipe = DispatchPipeline(world, ew, **kw)
    assert pipe.fp8_dispatch == (fp8 and not flat)
    names = [n for n in "send_counts pos send payload send_q send_scale send_gate expert_cnt row_map row_gate xs hidden ret ret_flat".split()
             if isinstance(getattr(pipe, n, None), torch.Tensor)]

    def results():
        for n in names:
            getattr(pipe, n).zero_()
        pipe.step()
        torch.cuda.synchronize()
        return {n: getattr(pipe, n).clone() for n in names}
    apart = results()
    for what in shared.split():
        if what == "counts":
            world.recv_counts = pipe.send_counts
        elif what == "scale":
            world.recv_scale = pipe.send_scale
        elif what == "gate":
            pipe.recv_gate = pipe.send_gate
        elif flat:
            pipe.recv_flat = pipe.payload
        else:
            world.recv_q = pipe.send_q
    back = results()
    for n in names:
        assert torch.equal(back[n], apart[n]), f"{n} differs"


@pytest.mark.parametrize("over", ["ret over send", "ret over recv", "ret over rows", "ret over counts and rows", "y over recv", "y over rows"])
def test_fp32_destination_buffers_that_take_each_others_place(over):
    """Scratch plans that stage by stage are right: a buffer where another lay that is done with by then."""
    from iris_testing_amd.configs import MoEConfig
    from iris_testing_amd.pipeline import DispatchPipeline
    cfg = MoEConfig("case", 7, 300, 256, "f32", 8, 2, 4, 128, "gelu")
    world = harness.build_world(cfg, DEV)
    ew, _, _ = harness.expert_weights(cfg, 0, DEV)
    pipe = DispatchPipeline(world, ew)
    pipe.step()
    torch.cuda.synchronize()
    names = ["hidden", "ret", "out"] + (["y"] if over[0] == "y" else [])
    want, recv, S = {n: getattr(pipe, n).clone() for n in names}, world.recv.clone(), pipe.S
    assert pipe.ret.numel() >= 64 + S * cfg.hidden
    if over == "ret over send":
        pipe.ret = pipe.send
    elif over == "ret over recv":
        pipe.ret = world.recv
    elif over == "y over recv":
        pipe.y = world.recv.view(-1)[:S * cfg.hidden].view(S, -1)
    elif over == "y over rows":
        pipe.y = pipe.rows
    else:
        if "counts" in over:
            pipe.expert_cnt = pipe.ret.view(-1).view(torch.int32)[:cfg.e_local]
        pipe.rows = pipe.ret.view(-1)[64:64 + S * cfg.hidden].view(S, -1)
    for _ in range(3):
        pipe.ret.fill_(5)
        pipe.y.fill_(5)
        world.recv.copy_(recv)
        pipe.step()
        torch.cuda.synchronize()
        for n in names:
            assert torch.equal(getattr(pipe, n), want[n]), f"{n} differs"


def test_entry_point_smoke_runs():
    """The smoke check of the repository's entry module (one small step against the oracle) must keep passing."""
    import importlib
    import os
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    if root not in sys.path:
        sys.path.insert(0, root)
    importlib.import_module("__graft_entry__").smoke()
