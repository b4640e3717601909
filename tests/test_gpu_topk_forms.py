"""The router's selection and the pack have a form of their own for every usual top-k (1, 2, 4, 8, 16) and one for any: the first against the
oracle, the second against the slot-major gather, around the sizes of a wave's pass and of a row's runs of columns."""
import pytest
import torch

from helpers import O, assert_bits_equal, to_np

pytestmark = pytest.mark.gpu

from iris_testing_amd import ops  # noqa: E402

DEV = "cuda"


@pytest.mark.parametrize("k", [1, 2, 3, 4, 7, 8, 15, 16])
@pytest.mark.parametrize("T,H,E,W,dtype", [(1, 64, 16, 2, "bf16"), (65, 1032, 24, 3, "bf16"), (300, 132, 40, 4, "f32"), (130, 64, 264, 8, "bf16"),
                                           (2100, 72, 512, 8, "bf16")])
def test_selection_and_pack_for_every_topk(T, H, E, W, dtype, k):
    g = torch.Generator(device=DEV).manual_seed(T + k)
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    x, router = (torch.randn(s, device=DEV, generator=g).to(dt) for s in ((T, H), (H, E)))
    idx, gate, logits = ops.route_topk(x, router, k)
    assert_bits_equal(idx, O.topk_select(to_np(logits), k), "indices")
    # (E roundings in the sum, exp to 2 ulp and the difference in its argument rounded, one division; a value below the smallest normal number, 2^-126, is a few bits
    # of a subnormal one or 0: off by less than that number)
    far = (logits.amax(1) - logits.amin(1)).double()[:, None]
    p = torch.softmax(logits.double(), 1).gather(1, idx.long())
    assert ((gate.double() - p).abs() <= (E + 8 + 2 * far) * 2.0 ** -23 * p + 2.0 ** -126).all()
    n = ops.count_and_offsets(idx, E, W)
    for M in (int(n.caps[0]), max(1, int(n.caps[0]) // 2)):  # (all rows; the larger destinations' last ones dropped)
        status, st2 = (torch.zeros(1, dtype=torch.int32, device=DEV) for _ in range(2))
        want = ops.pack_fixed_m(x, n.row_token, n.dst_sizes, n.dst_offsets, M, status=status)
        send, send_gate = ops.pack_tokens(x, idx, n.pos, n.dst_sizes, n.dst_offsets, E // W, M, status=st2, gate=gate)
        assert torch.equal(send.view(torch.uint8), want.view(torch.uint8)) and status.item() == st2.item()
        want_gate = torch.zeros(W, M, device=DEV)
        d = idx.long() // (E // W)
        m = n.pos.long() - n.dst_offsets.long()[d]
        keep = m < M
        want_gate[d[keep], m[keep]] = gate[keep]
        assert torch.equal(send_gate, want_gate)
        if dtype == "bf16":
            q, scale = ops.pack_tokens_fp8(x, idx, n.pos, n.dst_sizes, n.dst_offsets, E // W, M)[:2]
            want_q, want_scale = ops.quantize_rows_fp8(want.view(W * M, H))
            assert torch.equal(q.view(torch.uint8).view(W * M, H), want_q.view(torch.uint8)) and torch.equal(scale.view(-1), want_scale.view(-1))
