"""Up to some two thousand slots a step counts and packs in one launch, where every wave finds its token's rows from the expert ids alone.  Against the
stages one by one (the ranking, then the pack) on both sides of that line: every top-k form, odd worlds, rows that are dropped, all layouts."""
from dataclasses import replace

import pytest
import torch

pytestmark = pytest.mark.gpu

from iris_testing_amd import harness  # noqa: E402
from iris_testing_amd.configs import CONFIGS  # noqa: E402
from iris_testing_amd.pipeline import DispatchPipeline  # noqa: E402

DEV = "cuda"
NAMES = ("logits idx gate send_counts expert_offs dst_sizes dst_offsets caps pos row_token send send_gate send_q send_scale payload expert_cnt row_map row_gate rows "
         "hidden y ret ret_flat out status").split()


def _pipe(name, tokens, topk, experts, world, hidden=None, mode="fixed", slots=None):
    cfg = replace(CONFIGS[name], tokens=tokens, topk=topk, experts=experts, world=world, hidden=hidden or CONFIGS[name].hidden, ffn=128)
    w = harness.build_world(cfg, DEV)
    ew, _, _ = harness.expert_weights(cfg, 0, DEV)
    kw = dict(recv_gate=harness.recv_gates(w)) if mode == "gated" else dict(recv_flat=harness.recv_flat(w)) if mode == "flat" else {}
    if slots:
        w.M = max(1, int(w.M * slots))
        w.recv = w.recv[:, :w.M].contiguous()
        if mode == "gated":
            kw["recv_gate"] = kw["recv_gate"][:, :w.M].contiguous()
    p = DispatchPipeline(w, ew, gated=mode == "gated", padding_free=mode == "flat", **kw)
    p.returned.copy_(torch.randn(p.returned.shape, device=DEV).to(p.returned.dtype))
    return p


def _results(pipe, events, skip=()):
    names = [n for n in NAMES if isinstance(getattr(pipe, n, None), torch.Tensor) and n not in skip]
    for n in names:
        getattr(pipe, n).fill_(0 if n == "status" else 77)
    pipe.step(events)
    torch.cuda.synchronize()
    return {n: getattr(pipe, n).clone() for n in names}


@pytest.mark.parametrize("mode", ["fixed", "gated", "flat"])
@pytest.mark.parametrize("tokens,topk,experts,world,slots", [(1, 1, 8, 8, None), (2, 16, 16, 1, None), (65, 3, 27, 3, None), (32, 16, 64, 2, None), (33, 16, 64, 2, None),
                                                             (128, 8, 256, 8, 0.5), (129, 8, 256, 8, None), (512, 4, 20, 5, 0.3), (513, 4, 20, 5, None),
                                                             (1024, 2, 512, 8, None), (1025, 2, 8, 2, None), (2048, 1, 12, 4, 0.7), (2049, 1, 12, 4, None)])
def test_count_with_the_pack_equals_the_stages(tokens, topk, experts, world, slots, mode):
    pipe = _pipe("small", tokens, topk, experts, world, hidden=64 if topk == 1 else 1088, mode=mode, slots=slots if mode != "flat" else None)
    one, stages = _results(pipe, None), _results(pipe, [])
    for n in one:
        assert torch.equal(one[n], stages[n]), f"{n} differs"
    if slots and mode != "flat":
        assert one["status"].item() == 1


@pytest.mark.parametrize("tokens,topk,experts,world,hidden,mode", [(1, 1, 8, 8, 128, "fixed"), (33, 16, 64, 2, 1152, "fixed"), (100, 3, 27, 3, 2176, "gated"),
                                                                   (128, 8, 64, 8, 4224, "gated"), (512, 4, 20, 5, 256, "fixed"), (513, 4, 20, 5, 256, "fixed"),
                                                                   (1024, 2, 8, 2, 8320, "fixed"), (2048, 1, 12, 4, 128, "gated")])
def test_count_with_the_quantising_pack_equals_the_stages(tokens, topk, experts, world, hidden, mode):
    pipe = _pipe("zipf_k4", tokens, topk, experts, world, hidden=hidden, mode=mode)
    assert pipe.fp8_dispatch
    one, stages = _results(pipe, None), _results(pipe, [])
    for n in one:
        assert torch.equal(one[n], stages[n]), f"{n} differs"


@pytest.mark.parametrize("tokens,topk", [(1, 2), (100, 5), (1024, 2), (1025, 2)])
def test_count_with_the_pack_fp32(tokens, topk):
    pipe = _pipe("plumbing", tokens, topk, 8, 4)
    one, stages = _results(pipe, None), _results(pipe, [])
    for n in one:
        assert torch.equal(one[n], stages[n]) or n in ("rows", "hidden"), f"{n} differs"  # (scratch of the fp32 experts: rows in other places)


def test_a_rank_that_sends_to_itself():
    """The received counts are the sent ones: the receive side waits for the launch that counts and packs."""
    pipe = _pipe("small", 300, 2, 16, 1)
    w = pipe.world
    w.recv, w.recv_counts = pipe.send, pipe.send_counts
    one, stages = _results(pipe, None), _results(pipe, [])
    for n in one:
        assert torch.equal(one[n], stages[n]), f"{n} differs"


def test_count_beside_the_pack_only_where_their_buffers_are_apart():
    """The list of tokens in slot order, which no later stage of this layout reads, laid over the send buffer: the pack has the last word."""
    pipe = _pipe("small", 300, 2, 16, 4)
    want = _results(pipe, None)
    pipe.row_token = pipe.send.view(-1).view(torch.int32)[:600]
    got = _results(pipe, None, skip=("row_token",))
    for n in got:
        assert torch.equal(got[n], want[n]), f"{n} differs"
