"""GPU parity, integer/byte part of the path: route indices, counts, offsets, M/CAP, payload order,
packed [W,M,H], token_buf, expert-major rows, return buffer, combine -- all compared BIT-EXACTLY
with the CPU oracle on identical seeded inputs, through the C ABI (iris_testing_amd.ops)."""
import dataclasses

import numpy as np
import pytest
import torch

from helpers import O, assert_bits_equal, oracle_recv, oracle_world, to_np

pytestmark = pytest.mark.gpu

from iris_testing_amd import ops, utils  # noqa: E402
from iris_testing_amd.configs import CONFIGS, gen_router, gen_router_bias, gen_shard_tokens  # noqa: E402
from iris_testing_amd.layers import SimulatedWorld, custom_a2a, simulated_world  # noqa: E402

DEV = "cuda"

# (config name, tokens per shard or None for the full size)
ROUTE_CASES = [("plumbing", None), ("small", None), ("mixtral", 2048), ("mixtral", None), ("finegrained", 512),
               ("finegrained", None), ("zipf_k1", 1024), ("zipf_k2", None), ("zipf_k4", 1000), ("zipf_k8", None)]


def _cfg(name, tokens):
    cfg = CONFIGS[name]
    return cfg if tokens is None else dataclasses.replace(cfg, tokens=tokens)


def _inputs(cfg, shard=0):
    x = gen_shard_tokens(cfg, shard)
    w = gen_router(cfg)
    b = gen_router_bias(cfg)
    return x, w, b


@pytest.mark.parametrize("name,tokens", ROUTE_CASES)
def test_route_count_pack_bit_exact(name, tokens):
    cfg = _cfg(name, tokens)
    print(f"case {cfg}", flush=True)
    x, w, b = _inputs(cfg)
    xn, wn, bn = to_np(x), to_np(w), None if b is None else to_np(b)
    xd, wd = x.to(DEV), w.to(DEV)
    bd = None if b is None else b.to(DEV)

    idx, gate, logits = ops.route_topk(xd, wd, cfg.topk, bd)
    o_idx, o_gate, o_logits = O.route(xn, wn, cfg.topk, bn)
    assert_bits_equal(logits, o_logits, "router logits")
    assert_bits_equal(idx, o_idx, "top-k indices")
    np.testing.assert_allclose(to_np(gate), o_gate, rtol=1e-5, atol=1e-30, err_msg="softmax gates")

    c = ops.count_and_offsets(idx, cfg.experts, cfg.world)
    o_counts = O.send_counts(o_idx, cfg.world, cfg.experts)
    o_sizes, o_offs = O.dst_sizes_offsets(o_counts)
    o_pos, o_rt = O.payload_positions(o_idx, cfg.experts)
    assert_bits_equal(c.send_counts, o_counts, "send_counts")
    assert_bits_equal(c.expert_offs, O.build_expert_offsets(o_counts), "expert_offs")
    assert_bits_equal(c.dst_sizes, o_sizes, "dst_sizes")
    assert_bits_equal(c.dst_offsets, o_offs, "dst_offsets")
    assert_bits_equal(c.pos, o_pos, "pos")
    assert_bits_equal(c.row_token, o_rt, "row_token")
    caps = to_np(c.caps)
    assert caps[0] == O.pair_capacity(o_sizes) and caps[1] == O.compute_capacity_from_pca(o_counts)

    payload = ops.pack_payload(xd, c.row_token)
    o_payload = O.send_payload(xn, o_rt)
    assert_bits_equal(payload, o_payload, "send_payload")

    M = int(caps[0]) + 3  # a few rows of mandatory zero padding everywhere
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    send = ops.pack_fixed_m(xd, c.row_token, c.dst_sizes, c.dst_offsets, M, status=status)
    assert_bits_equal(send, O.pack_fixed_m(o_payload, o_offs, o_sizes, M), "send [W,M,H]")
    assert int(status.item()) == 0
    # the token-major writer of the same buffer (each token row read once), into a buffer full of garbage
    send2 = torch.full_like(send, 3.0)
    ops.pack_tokens(xd, idx, c.pos, c.dst_sizes, c.dst_offsets, cfg.e_local, M, out=send2, status=status)
    assert_bits_equal(send2, O.pack_fixed_m(o_payload, o_offs, o_sizes, M), "send [W,M,H], token-major")
    assert int(status.item()) == 0


def test_route_ties_prefer_lower_expert():
    # identical router columns -> identical logits: every tie must resolve to the lower expert id
    T, H, E, k = 130, 64, 40, 5
    g = torch.Generator().manual_seed(5)
    x = torch.randn(T, H, generator=g)
    col = torch.randn(H, 4, generator=g)
    w = col.repeat(1, E // 4)  # expert e has the same column as e % 4
    idx, gate, logits = ops.route_topk(x.to(DEV), w.to(DEV).contiguous(), k)
    o_idx, _, _ = O.route(x.numpy(), w.numpy(), k)
    assert_bits_equal(idx, o_idx, "tied top-k")
    # the best class appears with its k lowest ids (10 copies of each class, k = 5)
    cls = o_idx % 4
    assert (cls == cls[:, :1]).all() and (np.diff(o_idx, axis=1) == 4).all()


def test_route_zeros_of_either_sign_tie():
    """Products that underflow (1e-30 * +-1e-30) give logits of +0 or -0 by the sign of the router column: they compare
    equal, so the selection is the k lowest expert ids whatever the signs (the selection keys count -0 as +0), and
    every gate is 1 / E."""
    T, H, E, k = 70, 64, 24, 6
    x = torch.full((T, H), 1e-30)
    w = torch.full((H, E), 1e-30)
    w[:, ::3] = -1e-30   # every step of the chain adds -1e-60, which rounds to -0: these experts' logits are -0
    b = torch.full((E,), -0.0)
    idx, gate, logits = ops.route_topk(x.to(DEV), w.to(DEV).contiguous(), k, b.to(DEV))
    o_idx, o_gate, o_logits = O.route(x.numpy(), w.numpy(), k, b.numpy())
    assert_bits_equal(logits, o_logits, "signed-zero logits")
    lg = to_np(logits)
    assert np.signbit(lg[:, ::3]).all() and not np.signbit(lg[:, 1::3]).any(), "the case does not produce both zeros"
    assert_bits_equal(idx, o_idx, "top-k among zeros")
    assert (to_np(idx) == np.arange(k)[None, :]).all()
    np.testing.assert_allclose(to_np(gate), np.full((T, k), 1.0 / E, np.float32), rtol=1e-6)


@pytest.mark.parametrize("kind", ["wide", "subnormal", "cancel"])
@pytest.mark.parametrize("E", [8, 20, 200])
def test_route_logits_rounding_matches_fmaf_chain(kind, E):
    """The logits run on K = 1 fp32 matrix instructions; every step must round exactly like fmaf (one rounding,
    subnormals kept): operands spread over 40 binades, products in the subnormal range, and sums that cancel
    would each expose a multiply-then-add, a flush to zero or another summation order."""
    T, H, k = 130, 200, 3
    g = torch.Generator().manual_seed(E * 7 + len(kind))
    x = torch.randn(T, H, generator=g)
    w = torch.randn(H, E, generator=g)
    if kind == "wide":
        x = x * torch.pow(2.0, torch.randint(-20, 21, (T, H), generator=g).float())
        w = w * torch.pow(2.0, torch.randint(-20, 21, (H, E), generator=g).float())
    elif kind == "subnormal":
        x = x * 2.0 ** -70
        w = w * 2.0 ** -62
    else:
        x[:, 1::2] = -x[:, 0::2]  # consecutive terms nearly cancel
        w[1::2] = w[0::2] * (1 + 2.0 ** -12)
    idx, gate, logits = ops.route_topk(x.to(DEV), w.to(DEV).contiguous(), k)
    o_idx, _, o_logits = O.route(x.numpy(), w.numpy(), k)
    if kind == "subnormal":
        assert np.abs(o_logits).max() < 2.0 ** -126 and np.count_nonzero(o_logits) > o_logits.size // 2
    assert_bits_equal(logits, o_logits, f"logits ({kind})")
    assert_bits_equal(idx, o_idx, f"top-k ({kind})")


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("E", [3, 8, 16, 40, 130])
def test_route_block_shapes_for_many_tokens(E, dtype):
    """More than 2048 tokens take the block shapes with two token blocks per wave (one for fp32 tokens at 17 to 64
    experts), one per range of E: each of them, in both token dtypes, with a row length that is no multiple of the
    segment length, bit-exact against the oracle."""
    T, H, k = 2500, 200, min(3, E)
    g = torch.Generator().manual_seed(E)
    x = torch.randn(T, H, generator=g)
    w = torch.randn(H, E, generator=g) * H ** -0.5
    b = torch.randn(E, generator=g)
    if dtype == "bf16":
        x, w = x.bfloat16(), w.bfloat16()
    idx, gate, logits = ops.route_topk(x.to(DEV), w.to(DEV).contiguous(), k, b.to(DEV))
    o_idx, o_gate, o_logits = O.route(to_np(x), to_np(w), k, b.numpy())
    assert_bits_equal(logits, o_logits, f"logits E={E} {dtype}")
    assert_bits_equal(idx, o_idx, f"top-k E={E} {dtype}")
    np.testing.assert_allclose(to_np(gate), o_gate, rtol=1e-5, atol=1e-30)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("T,H,E,k,bias", [(2049, 8, 1, 1, True), (2111, 72, 2, 2, False), (2050, 4096, 8, 8, True), (2300, 520, 9, 9, False),
                                          (2177, 264, 13, 5, True), (3000, 8192, 16, 16, True), (2112, 64, 5, 1, False)])
def test_route_one_launch_edge_shapes(T, H, E, k, bias, dtype):
    """Up to 16 experts and more than 2048 tokens run logits and top-k in one launch: one token in the last workgroup, a single
    expert, as many selections as experts, rows shorter than one segment per wave (most chains empty), rows of 16 KB, expert counts
    on either side of the two-group / four-group split, with and without bias -- bit-exact against the oracle."""
    g = torch.Generator().manual_seed(T + 7 * E)
    x = torch.randn(T, H, generator=g)
    w = torch.randn(H, E, generator=g) * H ** -0.5
    b = torch.randn(E, generator=g) if bias else None
    if dtype == "bf16":
        x, w = x.bfloat16(), w.bfloat16()
    idx, gate, logits = ops.route_topk(x.to(DEV), w.to(DEV).contiguous(), k, None if b is None else b.to(DEV))
    o_idx, o_gate, o_logits = O.route(to_np(x), to_np(w), k, None if b is None else b.numpy())
    assert_bits_equal(logits, o_logits, f"logits T={T} H={H} E={E} {dtype}")
    assert_bits_equal(idx, o_idx, f"top-k T={T} H={H} E={E} k={k} {dtype}")
    np.testing.assert_allclose(to_np(gate), o_gate, rtol=1e-5, atol=1e-30)


@pytest.mark.parametrize("off", [1, 2, 4])
@pytest.mark.parametrize("T,H,E", [(2049, 136, 32), (600, 136, 128), (4200, 72, 256)])
def test_route_of_a_router_at_an_odd_address(T, H, E, off):
    """A router that is a slice of a flat buffer, at addresses where four experts' values do not lie at 8 bytes (off 4: they do):
    bit-exact against the oracle, for each form of the kernel for many tokens."""
    g = torch.Generator().manual_seed(T + E)
    x, w = torch.randn(T, H, generator=g).bfloat16(), (torch.randn(H, E, generator=g) * H ** -0.5).bfloat16()
    flat = torch.empty(H * E + off, dtype=torch.bfloat16, device=DEV)
    router = flat[off:].view(H, E)
    router.copy_(w)
    assert router.is_contiguous() and router.data_ptr() % 8 == 2 * off % 8
    idx, gate, logits = ops.route_topk(x.to(DEV), router, 4)
    o_idx, o_gate, o_logits = O.route(to_np(x), to_np(w), 4)
    assert_bits_equal(logits, o_logits, "logits")
    assert_bits_equal(idx, o_idx, "top-k")
    np.testing.assert_allclose(to_np(gate), o_gate, rtol=1e-5, atol=1e-30)


@pytest.mark.parametrize("E,k,W", [(8, 8, 4), (512, 16, 64), (6, 1, 3), (60, 7, 1), (40, 12, 4), (16, 16, 2)])  # (the last two: more selections than lanes per token)
def test_route_edge_shapes(E, k, W):
    T, H = 77, 72
    g = torch.Generator().manual_seed(E * 31 + k)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    w = (torch.randn(H, E, generator=g) / 8).to(torch.bfloat16)
    b = torch.randn(E, generator=g)
    idx, gate, logits = ops.route_topk(x.to(DEV), w.to(DEV), k, b.to(DEV))
    o_idx, o_gate, o_logits = O.route(to_np(x), to_np(w), k, b.numpy())
    assert_bits_equal(logits, o_logits, "logits")
    assert_bits_equal(idx, o_idx, "idx")
    np.testing.assert_allclose(to_np(gate), o_gate, rtol=1e-5)
    c = ops.count_and_offsets(idx, E, W)
    assert_bits_equal(c.send_counts, O.send_counts(o_idx, W, E), "send_counts")
    assert_bits_equal(c.pos, O.payload_positions(o_idx, E)[0], "pos")


def test_zero_tokens_and_overflow_flag():
    # zero routed tokens: all counts zero, capacities floor at 1 (reference utils.py:121,240-242)
    idx = torch.empty((0, 2), dtype=torch.int32, device=DEV)
    c = ops.count_and_offsets(idx, 8, 4)
    assert to_np(c.send_counts).sum() == 0 and to_np(c.caps).tolist() == [1, 1]
    # M smaller than a destination's rows -> status flag, rows beyond M dropped, no overrun
    cfg = CONFIGS["plumbing"]
    x, w, _ = _inputs(cfg)
    xd = x.to(DEV)
    idx, _, _ = ops.route_topk(xd, w.to(DEV), cfg.topk)
    c = ops.count_and_offsets(idx, cfg.experts, cfg.world)
    M = int(c.caps[0].item()) - 5
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    guard = torch.full((cfg.world * M + 4, cfg.hidden), 7.0, device=DEV)
    ops.pack_fixed_m(xd, c.row_token, c.dst_sizes, c.dst_offsets, M, out=guard[:cfg.world * M].view(cfg.world, M, -1),
                     status=status)
    assert int(status.item()) == 1
    assert (guard[cfg.world * M:] == 7.0).all()
    kept = guard[:cfg.world * M].clone()
    status.zero_()
    guard.fill_(7.0)
    ops.pack_tokens(xd, idx, c.pos, c.dst_sizes, c.dst_offsets, cfg.e_local, M,
                    out=guard[:cfg.world * M].view(cfg.world, M, -1), status=status)
    assert int(status.item()) == 1
    assert (guard[cfg.world * M:] == 7.0).all()
    assert torch.equal(guard[:cfg.world * M], kept), "token-major pack drops the same rows as the slot-major one"


def test_overflowed_pack_drops_rows_consistently_down_the_path():
    """M below the largest pair size: the pack raises the status word and drops the rows at and past M; every
    later stage must treat exactly those rows as absent (zero rows on the receive side, no slot on the way back,
    no contribution to the combine) and stay inside its buffers.  Bit-exact against the oracle's drop semantics;
    the copy-free destination side (row map with -1 entries, gathering / scattering GEMM) against the copies."""
    cfg = _cfg("zipf_k4", 512)
    W, E, E_l, k, H = cfg.world, cfg.experts, cfg.e_local, cfg.topk, cfg.hidden
    w = gen_router(cfg)
    b = gen_router_bias(cfg)
    xs = [gen_shard_tokens(cfg, s) for s in range(W)]
    xn = [to_np(x) for x in xs]
    shards, M_full, CAP = oracle_world(cfg, xn, to_np(w), to_np(b))
    M = M_full - 37
    assert all(int(sh["sizes"][0]) > M for sh in shards)  # every source overflows its slot on rank 0
    # source side of shard 0: both packs drop the same rows and raise the flag
    s0 = shards[0]
    x0 = xs[0].to(DEV)
    idx0, pos0 = torch.from_numpy(s0["idx"]).to(DEV), torch.from_numpy(s0["pos"]).to(DEV)
    sizes0, offs0 = torch.from_numpy(s0["sizes"]).to(DEV), torch.from_numpy(s0["offs"]).to(DEV)
    o_send0 = O.pack_fixed_m(O.send_payload(xn[0], s0["row_token"]), s0["offs"], s0["sizes"], M, drop=True)
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    send = ops.pack_tokens(x0, idx0, pos0, sizes0, offs0, E_l, M, status=status)
    assert int(status.item()) == 1
    assert_bits_equal(send, o_send0, "token-major pack with dropped rows")
    send2 = ops.pack_fixed_m(x0, torch.from_numpy(s0["row_token"]).to(DEV), sizes0, offs0, M)
    assert_bits_equal(send2, o_send0, "slot-major pack with dropped rows")
    # destination side of rank 0
    o_recv = np.stack([O.pack_fixed_m(O.send_payload(x, sh["row_token"]), sh["offs"], sh["sizes"], M, drop=True)[0]
                       for x, sh in zip(xn, shards)])
    o_rc = np.stack([sh["counts"][0] for sh in shards]).astype(np.int32)
    recv = torch.from_numpy(o_recv).to(cfg.torch_dtype).to(DEV)
    rc = torch.from_numpy(o_rc).to(DEV)
    S = int(o_rc.sum())
    o_rows = O.unpack_expert_major(o_recv, o_rc)
    n_dropped = int((np.abs(o_rows).sum(1) == 0).sum())
    assert n_dropped > 0
    rows, cnt = ops.unpack_expert_major(recv, rc, S)
    assert_bits_equal(rows, o_rows, "expert-major rows (dropped rows read as zeros)")
    status.zero_()
    tb, pca = ops.unpack_token_buf(recv, rc, CAP, status=status)
    assert int(status.item()) == 1
    assert_bits_equal(tb, O.recv_to_token_buf(o_recv, o_rc, CAP)[0], "token_buf")
    y = (rows * 2).contiguous()
    guard = torch.full((W * M + 8, H), 3.0, dtype=rows.dtype, device=DEV)
    ret = ops.return_pack(y, rc, M, out=guard[:W * M].view(W, M, H))
    assert_bits_equal(ret, O.return_pack(o_rows * 2, o_rc, M), "return buffer")
    assert (guard[W * M:] == 3.0).all()
    # the copy-free destination side: dropped rows carry -1 in the row map, read row 0 and store nothing
    row_map, cnt2 = ops.recv_row_map(rc, M, S)
    assert torch.equal(cnt, cnt2)
    rm = to_np(row_map)
    assert int((rm < 0).sum()) == n_dropped and rm.max() < W * M
    keep = rm >= 0
    assert_bits_equal(recv.view(W * M, H)[torch.from_numpy(rm[keep]).long().to(DEV)], o_rows[keep], "rows picked by the row map")
    rng = np.random.default_rng(5)
    N = 256
    wt = torch.from_numpy(O.bf16_round((rng.standard_normal((E_l, H, N)) * H ** -0.5).astype(np.float32))).to(torch.bfloat16).to(DEV)
    packed = ops.prepack_weights(wt)
    plain = torch.zeros((S, N), dtype=torch.bfloat16, device=DEV)
    ops.grouped_gemm_mapped(rows, None, packed, cnt, S, N, "none", plain)
    want = torch.full((W * M + 8, N), 3.0, dtype=torch.bfloat16, device=DEV)
    want[:W * M] = ops.return_pack(plain, rc, M).view(W * M, N)
    got = torch.full((W * M + 8, N), 3.0, dtype=torch.bfloat16, device=DEV)
    ops.grouped_gemm_mapped(recv.view(W * M, H), row_map, packed, cnt, S, N, "none", got, c_row_map=row_map)
    ops.zero_padding_rows(got[:W * M].view(W, M, N), rc)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16)), "gathering / scattering GEMM with dropped rows"
    # combine on shard 0: returned = 2 * what was sent; dropped slots contribute nothing; flag raised
    returned = torch.from_numpy(o_send0 * 2).to(cfg.torch_dtype).to(DEV)
    gate0 = torch.from_numpy(s0["gate"]).to(DEV)
    status.zero_()
    out = ops.combine(returned, idx0, pos0, gate0, offs0, E_l, status=status)
    assert int(status.item()) == 1
    assert_bits_equal(out, O.combine(o_send0 * 2, s0["idx"], s0["pos"], s0["gate"], s0["offs"], E_l, cfg.dtype), "combine")
    # an expert id outside the layout is skipped as well (no read outside the buffer)
    bad_idx = idx0.clone()
    bad_idx[3, 1] = E + 5 * E_l
    status.zero_()
    out = ops.combine(returned, bad_idx, pos0, gate0, offs0, E_l, status=status)
    assert int(status.item()) == 1
    o_bad = s0["idx"].copy()
    o_bad[3, 1] = E + 5 * E_l
    assert_bits_equal(out, O.combine(o_send0 * 2, o_bad, s0["pos"], s0["gate"], s0["offs"], E_l, cfg.dtype), "combine, bad id")
    # ... and by the token-major pack: the slot of the bad id stays as it was (its offset is never read), all others are written
    t_bad, m_bad = 3, int(s0["pos"][3, 1] - s0["offs"][s0["idx"][3, 1] // E_l])
    guard = torch.full((W * M + 8, H), 7.0, dtype=cfg.torch_dtype, device=DEV)
    ops.pack_tokens(x0, bad_idx, pos0, sizes0, offs0, E_l, M, out=guard[:W * M].view(W, M, H))
    want = o_send0.copy()
    d_bad = int(s0["idx"][t_bad, 1]) // E_l
    if m_bad < M:
        want[d_bad, m_bad] = 7.0
    assert_bits_equal(guard[:W * M].view(W, M, H), want, "token-major pack, bad id")
    assert (guard[W * M:] == 7.0).all()


UNPACK_CASES = [("plumbing", None), ("small", None), ("mixtral", 1024), ("finegrained", 512), ("zipf_k4", 1024)]


@pytest.mark.parametrize("name,tokens", UNPACK_CASES)
def test_unpack_return_combine_bit_exact(name, tokens):
    """All W shards routed on both sides; rank 0's receive buffer assembled; then token_buf, pca,
    expert-major rows, return buffer and combine compared bit for bit."""
    cfg = _cfg(name, tokens)
    print(f"case {cfg}", flush=True)
    w = gen_router(cfg)
    b = gen_router_bias(cfg)
    xs = [gen_shard_tokens(cfg, s) for s in range(cfg.world)]
    xn = [to_np(x) for x in xs]
    shards, M, CAP = oracle_world(cfg, xn, to_np(w), None if b is None else to_np(b))
    o_recv, o_rc = oracle_recv(cfg, xn, shards, M, 0)

    recv = torch.from_numpy(o_recv).to(cfg.torch_dtype).to(DEV)
    rc = torch.from_numpy(o_rc).to(DEV)
    S = int(o_rc.sum())

    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    tb, pca = ops.unpack_token_buf(recv, rc, CAP, status=status)
    o_tb, o_pca = O.recv_to_token_buf(o_recv, o_rc, CAP)
    assert_bits_equal(tb, o_tb, "token_buf")
    assert_bits_equal(pca, o_pca, "pca")
    assert int(status.item()) == 0

    sh, cnt = ops.shuffle_rows(tb, pca, S + 2)
    o_sh = O.shuffle(o_tb, o_pca)
    assert_bits_equal(sh[:S], o_sh, "shuffled")
    assert (to_np(sh[S:]) == 0).all()
    assert_bits_equal(cnt, O.expert_row_counts(o_pca), "expert_cnt")

    sh2, cnt2 = ops.unpack_expert_major(recv, rc, S)
    assert_bits_equal(sh2, O.unpack_expert_major(o_recv, o_rc), "unpack_expert_major")
    assert_bits_equal(cnt2, O.expert_row_counts(o_pca), "expert_cnt (fused)")

    # return path with a recognisable payload: y = 2 * shuffled (exact in every dtype, keeps +0 padding)
    y = (sh2 * 2).contiguous()
    ret = ops.return_pack(y, rc, M)
    o_ret = O.return_pack(o_sh * 2, o_rc, M)
    assert_bits_equal(ret, o_ret, "return buffer")
    # inverse property: the return buffer is 2 x the receive buffer, padding included
    assert_bits_equal(ret, o_recv * 2, "return == 2 * recv")

    # combine on rank 0 as a source: returned[d] is the slot dst d sends back = 2 * send_0[d]
    s0 = shards[0]
    o_send0 = O.pack_fixed_m(O.send_payload(xn[0], s0["row_token"]), s0["offs"], s0["sizes"], M)
    returned = torch.from_numpy(o_send0 * 2).to(cfg.torch_dtype).to(DEV)
    out = ops.combine(returned, torch.from_numpy(s0["idx"]).to(DEV), torch.from_numpy(s0["pos"]).to(DEV),
                      torch.from_numpy(s0["gate"]).to(DEV), torch.from_numpy(s0["offs"]).to(DEV), cfg.e_local)
    o_out = O.combine(o_send0 * 2, s0["idx"], s0["pos"], s0["gate"], s0["offs"], cfg.e_local, cfg.dtype)
    assert_bits_equal(out, o_out, "combine")


def test_capacity_overflow_flag_on_unpack():
    rc = torch.tensor([[3, 1], [0, 2]], dtype=torch.int32, device=DEV)
    recv = torch.arange(2 * 4 * 8, dtype=torch.float32, device=DEV).view(2, 4, 8)
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    tb, pca = ops.unpack_token_buf(recv, rc, 2, status=status)  # count 3 > CAP 2
    assert int(status.item()) == 1
    status.zero_()
    tb, pca = ops.unpack_token_buf(recv, rc, 3, status=status)
    assert int(status.item()) == 0
    assert_bits_equal(tb, O.recv_to_token_buf(to_np(recv), to_np(rc), 3)[0], "token_buf")


def test_kernels_reproduce_the_frozen_dispatch_vectors():
    """The committed vectors of tests/golden (every intermediate of route -> count -> pack -> unpack -> return ->
    combine on a tiny case) against the kernels, with no oracle call in between."""
    import os
    g = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "dispatch_small.npz"))
    W, E, k = 3, 12, 3
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    router, bias = dev(g["router"]), dev(g["bias"])
    M, CAP = int(g["M"]), int(g["CAP"])
    for s in range(W):
        x = dev(g[f"x{s}"])
        idx, gate, logits = ops.route_topk(x, router, k, bias)
        assert_bits_equal(logits, g[f"logits{s}"], f"logits of shard {s}")
        assert_bits_equal(idx, g[f"idx{s}"], f"top-k of shard {s}")
        np.testing.assert_allclose(to_np(gate), g[f"gate{s}"], rtol=1e-5)
        c = ops.count_and_offsets(idx, E, W)
        assert_bits_equal(c.send_counts, g[f"counts{s}"], "send_counts")
        assert_bits_equal(c.pos, g[f"pos{s}"], "pos")
        assert_bits_equal(c.row_token, g[f"row_token{s}"], "row_token")
        if s == 0:
            assert_bits_equal(ops.pack_tokens(x, idx, c.pos, c.dst_sizes, c.dst_offsets, E // W, M), g["send0"], "send [W,M,H]")
            assert_bits_equal(ops.pack_fixed_m(x, c.row_token, c.dst_sizes, c.dst_offsets, M), g["send0"], "send [W,M,H]")
            c0, idx0 = c, idx
    recv, rc = dev(g["recv"]), dev(g["recv_counts"])
    tb, pca = ops.unpack_token_buf(recv, rc, CAP)
    assert_bits_equal(tb, g["token_buf"], "token_buf")
    assert_bits_equal(pca, g["pca"], "pca")
    S = int(g["rows"].shape[0])
    rows, _ = ops.unpack_expert_major(recv, rc, S)
    assert_bits_equal(rows, g["rows"], "expert-major rows")
    assert_bits_equal(ops.shuffle_rows(tb, pca, S)[0], g["rows"], "shuffled rows")
    assert_bits_equal(ops.return_pack(rows * 2.0, rc, M), g["ret"], "return buffer")
    out = ops.combine(dev(g["send0"]) * 2.0, idx0, c0.pos, dev(g["gate0"]), c0.dst_offsets, E // W)
    assert_bits_equal(out, g["combined"], "combined output")


@pytest.mark.parametrize("T,H,E,k,W,slack", [(90, 64, 12, 3, 4, 2), (700, 2048, 60, 8, 4, 0), (300, 7168, 16, 1, 8, 5), (64, 16384, 8, 2, 2, 1)])
def test_pack_tokens_fp8_is_the_quantised_send_buffer(T, H, E, k, W, slack):
    """Quantise-and-pack against the oracle (quantize_rows_fp8 of every row of the bf16 send buffer): codes and scales
    bit-exact, padding slots codes 0 / scale 1; and against the kernels' own two-step path (pack, then quantise)."""
    rng = np.random.default_rng(T + H)
    x = O.bf16_round((rng.standard_normal((T, H)) * rng.uniform(0.1, 4.0, (T, 1))).astype(np.float32))
    x[3] = 0.0
    idx = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    counts = O.send_counts(idx, W, E)
    sizes, offs = O.dst_sizes_offsets(counts)
    pos, row_token = O.payload_positions(idx, E)
    M = O.pair_capacity(sizes) + slack
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    xt = torch.from_numpy(x).bfloat16().to(DEV)
    q = torch.full((W, M, H), 0xAB, dtype=torch.uint8, device=DEV)
    sc = torch.full((W, M), -3.0, dtype=torch.float32, device=DEV)
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    ops.pack_tokens_fp8(xt, dev(idx), dev(pos), dev(sizes), dev(offs), E // W, M, out_q=q, out_scale=sc, status=status)
    want_q, want_s = O.pack_fixed_m_fp8(O.send_payload(x, row_token), offs, sizes, M)
    assert_bits_equal(q, want_q, "fp8 send codes")
    assert_bits_equal(sc, want_s, "fp8 send scales")
    assert int(status.item()) == 0
    send = ops.pack_tokens(xt, dev(idx), dev(pos), dev(sizes), dev(offs), E // W, M)
    q2, s2 = ops.quantize_rows_fp8(send.view(W * M, H))
    assert torch.equal(q.view(W * M, H), q2) and torch.equal(sc.view(-1), s2)


def test_pack_tokens_fp8_drops_what_the_bf16_pack_drops():
    """An undersized M: the same rows are dropped, the status word is raised, nothing is written outside the buffers."""
    rng = np.random.default_rng(12)
    T, H, E, k, W = 200, 256, 8, 2, 4
    x = O.bf16_round(rng.standard_normal((T, H)).astype(np.float32))
    idx = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    counts = O.send_counts(idx, W, E)
    sizes, offs = O.dst_sizes_offsets(counts)
    pos, row_token = O.payload_positions(idx, E)
    M = int(sizes.max()) - 7
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    q, sc = ops.pack_tokens_fp8(torch.from_numpy(x).bfloat16().to(DEV), dev(idx), dev(pos), dev(sizes), dev(offs), E // W, M, status=status)
    want_q, want_s = O.pack_fixed_m_fp8(O.send_payload(x, row_token), offs, sizes, M, drop=True)
    assert_bits_equal(q, want_q, "fp8 send codes (overflow)")
    assert_bits_equal(sc, want_s, "fp8 send scales (overflow)")
    assert int(status.item()) == 1


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("k", [3, 7, 16])
def test_pack_and_combine_at_other_top_k(k, dtype):
    """top-k values without a compiled-in variant (the kernels then loop over a run-time k): pack, both ways, and
    combine, bit-exact against the oracle."""
    rng = np.random.default_rng(k)
    T, H, E, W = 130, 72, 48, 4
    E_l = E // W
    x = rng.standard_normal((T, H)).astype(np.float32)
    if dtype == "bf16":
        x = O.bf16_round(x)
    idx = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    gate = rng.random((T, k)).astype(np.float32)
    counts = O.send_counts(idx, W, E)
    sizes, offs = O.dst_sizes_offsets(counts)
    pos, row_token = O.payload_positions(idx, E)
    M = O.pair_capacity(sizes) + 1
    tdt = torch.float32 if dtype == "f32" else torch.bfloat16
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    xt = torch.from_numpy(x).to(tdt).to(DEV)
    want = O.pack_fixed_m(O.send_payload(x, row_token), offs, sizes, M)
    send = ops.pack_tokens(xt, dev(idx), dev(pos), dev(sizes), dev(offs), E_l, M)
    assert_bits_equal(send, want, "send (token-major pack)")
    assert_bits_equal(ops.pack_fixed_m(xt, dev(row_token), dev(sizes), dev(offs), M), want, "send (slot-major pack)")
    ret = O.bf16_round(rng.standard_normal((W, M, H)).astype(np.float32)) if dtype == "bf16" else rng.standard_normal((W, M, H)).astype(np.float32)
    out = ops.combine(torch.from_numpy(ret).to(tdt).to(DEV), dev(idx), dev(pos), dev(gate), dev(offs), E_l)
    assert_bits_equal(out, O.combine(ret, idx, pos, gate, offs, E_l, dtype), "combine")


@pytest.mark.parametrize("T", [1, 64, 65, 1024, 1025, 2049])
@pytest.mark.parametrize("E,W,k", [(2, 2, 1), (60, 4, 3), (512, 8, 8)])
def test_counts_and_positions_at_block_edges(T, E, W, k):
    """The single-workgroup count (up to 1024 tokens) and the two-launch one, around the edges of their blocks of 64 and 1024."""
    rng = np.random.default_rng(T + E)
    p = rng.random(E) ** 4 + 1e-6
    idx = np.stack([rng.choice(E, k, replace=False, p=p / p.sum()) for _ in range(T)]).astype(np.int32)
    c = ops.count_and_offsets(torch.from_numpy(idx).to(DEV), E, W)
    counts = O.send_counts(idx, W, E)
    sizes, offs = O.dst_sizes_offsets(counts)
    pos, row_token = O.payload_positions(idx, E)
    assert_bits_equal(c.send_counts, counts, "send_counts")
    assert_bits_equal(c.expert_offs, O.build_expert_offsets(counts), "expert_offs")
    assert_bits_equal(c.dst_sizes, sizes, "dst_sizes")
    assert_bits_equal(c.dst_offsets, offs, "dst_offsets")
    assert_bits_equal(c.pos, pos, "pos")
    assert_bits_equal(c.row_token, row_token, "row_token")
    assert c.caps.tolist() == [max(1, int(sizes.max())), max(1, int(counts.max()))]


@pytest.mark.parametrize("T,E,W,k", [(14080, 512, 8, 4), (14081, 512, 8, 4), (14400, 511, 7, 1), (65600, 73, 1, 2), (81001, 17, 1, 3), (330000, 1, 1, 1)])
def test_counts_and_positions_of_many_tokens(T, E, W, k):
    """Either side of where the ranking workgroups' own sums over the histogram give way to a scan (6 M cells read in all), which takes
    16 experts to a workgroup and 64 slices of groups of 4 blocks of tokens."""
    rng = np.random.default_rng(T + E)
    p = rng.random(E) ** 4 + 1e-6
    # (k distinct experts per token, drawn in proportion to p: the smallest of exponential times)
    idx = np.concatenate([np.argsort(rng.exponential(size=(min(8192, T - t), E)) / p, axis=1)[:, :k] for t in range(0, T, 8192)]).astype(np.int32)
    c = ops.count_and_offsets(torch.from_numpy(idx).to(DEV), E, W)
    counts = O.send_counts(idx, W, E)
    sizes, offs = O.dst_sizes_offsets(counts)
    pos, row_token = O.payload_positions(idx, E)
    assert_bits_equal(c.send_counts, counts, "send_counts")
    assert_bits_equal(c.expert_offs, O.build_expert_offsets(counts), "expert_offs")
    assert_bits_equal(c.dst_sizes, sizes, "dst_sizes")
    assert_bits_equal(c.dst_offsets, offs, "dst_offsets")
    assert_bits_equal(c.pos, pos, "pos")
    assert_bits_equal(c.row_token, row_token, "row_token")
    assert c.caps.tolist() == [max(1, int(sizes.max())), max(1, int(counts.max()))]


@pytest.mark.parametrize("T,E,W,k", [(16384, 64, 8, 2), (10923, 60, 4, 3), (4681, 511, 7, 7), (1027, 1, 1, 1)])
def test_counts_of_slots_that_every_workgroup_counts(T, E, W, k):
    """Either side of where the ranking workgroups count all slots themselves (32768), an index that 16-byte loads cannot start at, and
    expert ids that are none, which count nowhere."""
    test_counts_and_positions_of_many_tokens(T, E, W, k)
    idx = torch.stack([torch.randperm(max(E, k), generator=torch.Generator().manual_seed(t))[:k] for t in range(T + 1)]).to(torch.int32)
    idx[:: 97, 0] = -1
    idx[1:: 89, k - 1] = E
    both = [ops.count_and_offsets(i, E, W) for i in (idx.to(DEV)[1:], idx[1:].to(DEV))]
    want = torch.bincount(idx[1:][(idx[1:] >= 0) & (idx[1:] < E)], minlength=E).view(W, -1).to(torch.int32)
    placed = ((idx[1:] >= 0) & (idx[1:] < E)).to(DEV)
    for c in both:
        assert torch.equal(c.send_counts.cpu(), want)
    assert torch.equal(both[0].pos[placed], both[1].pos[placed])
    assert torch.equal(both[0].row_token[:int(want.sum())], both[1].row_token[:int(want.sum())])


@pytest.mark.parametrize("T,H,k", [(1, 520, 1), (5, 4096, 3), (33, 1032, 8), (700, 264, 2), (2050, 2056, 4)])
def test_row_copies_and_sums_cut_into_column_runs(T, H, k):
    """Rows cut into runs of columns (whole, ragged, single) where tokens are few, and for the sums where rows are long; pack, combine and the gradient of combine."""
    rng = np.random.default_rng(T)
    E, W = 16, 4
    E_l = E // W
    x = O.bf16_round(rng.standard_normal((T, H)).astype(np.float32))
    idx = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    gate = rng.random((T, k)).astype(np.float32)
    sizes, offs = O.dst_sizes_offsets(O.send_counts(idx, W, E))
    pos, row_token = O.payload_positions(idx, E)
    M = O.pair_capacity(sizes) + 1
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    bf = lambda a: torch.from_numpy(a).bfloat16().to(DEV)  # noqa: E731
    send = ops.pack_tokens(bf(x), dev(idx), dev(pos), dev(sizes), dev(offs), E_l, M)
    assert_bits_equal(send, O.pack_fixed_m(O.send_payload(x, row_token), offs, sizes, M), "send")
    ret = O.bf16_round(rng.standard_normal((W, M, H)).astype(np.float32))
    out = ops.combine(bf(ret), dev(idx), dev(pos), dev(gate), dev(offs), E_l)
    assert_bits_equal(out, O.combine(ret, idx, pos, gate, offs, E_l, "bf16"), "combine")
    d_out = O.bf16_round(rng.standard_normal((T, H)).astype(np.float32))
    want = np.zeros((W, M, H), np.float32)
    want_g = np.zeros((T, k), np.float64)
    for t in range(T):
        for j in range(k):
            d = idx[t, j] // E_l
            m = pos[t, j] - offs[d]
            want[d, m] = O.bf16_round(gate[t, j] * d_out[t])
            want_g[t, j] = (d_out[t].astype(np.float64) * ret[d, m]).sum()
    for known in (dev(sizes), None):  # (None: the sizes follow from the starts)
        d_ret, d_gate = ops.combine_backward(bf(d_out), bf(ret), dev(idx), dev(pos), dev(gate), known, dev(offs), E_l)
        assert_bits_equal(d_ret, want, "d returned")
        np.testing.assert_allclose(to_np(d_gate), want_g, rtol=1e-4, atol=1e-3)


# (the segment kernel below the token limits and at 33 to 64 experts; one segment per workgroup; all segments in one workgroup;
# rows of 8 to 63 chunks of eight, so that segments end inside and at the end of slabs, some of them empty)
@pytest.mark.parametrize("T,H,E,k,bias", [(65, 520, 250, 8, True), (130, 72, 300, 3, False), (511, 72, 72, 2, True), (513, 264, 68, 8, False), (2049, 504, 20, 1, True), (2177, 1032, 32, 4, False),
                                          (2050, 296, 60, 2, True), (8192, 136, 260, 8, True), (4200, 8, 256, 2, False), (16385, 328, 100, 4, False)])
def test_router_tiles_are_bit_exact(T, H, E, k, bias):
    rng = np.random.default_rng(T)
    x = O.bf16_round(rng.standard_normal((T, H)).astype(np.float32))
    w = O.bf16_round(rng.standard_normal((H, E)).astype(np.float32))
    b = rng.standard_normal(E).astype(np.float32) if bias else None
    dev = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    idx, gate, logits = ops.route_topk(dev(x).bfloat16(), dev(w).bfloat16(), k, None if b is None else dev(b))
    o_idx, o_gate, o_logits = O.route(x, w, k, b)
    assert_bits_equal(logits, o_logits, "router logits")
    assert_bits_equal(idx, o_idx, "top-k indices")
    np.testing.assert_allclose(to_np(gate), o_gate, rtol=1e-5, atol=1e-30)


@pytest.mark.parametrize("T,H,E,k,bias", [(14337, 136, 200, 8, True), (28673, 1032, 68, 2, False), (14500, 40, 132, 3, True)])
def test_router_of_very_many_tokens_in_finished_logits(T, H, E, k, bias):
    """Two tiles of 64 tokens x 128 experts for every compute unit: all segments in one workgroup, whatever the rows' length (empty and
    partly filled segments among them)."""
    test_router_tiles_are_bit_exact(T, H, E, k, bias)


@pytest.mark.parametrize("T,H,E,k,bias", [(4033, 264, 140, 8, True), (4097, 504, 130, 2, False), (7000, 72, 68, 4, True), (517, 40, 68, 2, True)])
def test_router_segments_two_and_four_to_a_compute_unit(T, H, E, k, bias):
    """One slab of LDS and four workgroups to a compute unit, or two and two, by what the rounds come to."""
    test_router_tiles_are_bit_exact(T, H, E, k, bias)


@pytest.mark.parametrize("T,H,E,k,bias", [(2050, 264, 256, 8, True), (8191, 72, 68, 2, False), (4097, 1032, 132, 4, True), (2048, 8, 252, 2, False), (2113, 40, 256, 3, True)])
def test_router_segments_by_two_sets_of_waves(T, H, E, k, bias):
    """Tiles of 64 x 64 whose segments two sets of waves share: empty and partly filled segments in either set, ragged tiles."""
    test_router_tiles_are_bit_exact(T, H, E, k, bias)


@pytest.mark.parametrize("H", [1024, 1032, 2040, 2048, 2056])
def test_copies_of_many_rows_two_and_four_to_a_wave(H):
    """Rows of 2 to 4 KB are copied two to a wave when there are many.  A copy moves columns without
    looking at them: the first 64 of every output are those of the same copy of 64-column rows, which go one by one."""
    T, E, W, k, E_l = 2051, 24, 4, 2, 6
    g = torch.Generator(device=DEV).manual_seed(H)
    x = torch.randn(T, H, generator=g, device=DEV).bfloat16()
    idx = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:k] for t in range(T)]).to(torch.int32).to(DEV)
    n = ops.count_and_offsets(idx, E, W)
    M, counts, S, cap = int(n.caps[0]) - 3, n.send_counts, T * k, int(n.caps[1]) - 1  # (three rows of a pair and one of an expert have no place)
    status = lambda: torch.zeros(1, dtype=torch.int32, device=DEV)  # noqa: E731

    def chain(rows, C):
        cols = lambda *s: torch.full((*s, C), 3.0, dtype=torch.bfloat16, device=DEV)  # noqa: E731
        payload = ops.pack_payload(rows, n.row_token)
        recv = ops.pack_fixed_m(rows, n.row_token, n.dst_sizes, n.dst_offsets, M, status=status())
        buf, pca = ops.unpack_token_buf(recv, counts, cap, cols(E_l, W, cap), status=status())
        flat = ops.reorder_flat(payload, counts, cap, cols(E_l, W, cap), status=status())
        er = ops.unpack_expert_major(recv, counts, S)[0]
        back = ops.return_pack(er, counts, M)
        pca_cut = counts.T.clamp(max=cap).contiguous()
        sh = ops.shuffle_rows(flat, pca_cut, int(pca_cut.sum()))[0]
        return [payload, recv, buf, flat, er, back, sh, ops.shuffle_rows_backward(sh, pca_cut, cap)]

    for i, (a, b) in enumerate(zip(chain(x, H), chain(x[:, :64].contiguous(), 64))):
        assert torch.equal(a[..., :64].view(torch.int16), b.view(torch.int16)), i
        assert a.numel() // H >= 4096 or i in (2, 3, 6, 7)
    assert torch.equal(chain(x, H)[0].view(torch.int16), x[n.row_token.long()].view(torch.int16))


@pytest.mark.parametrize("H", [8, 768, 1024, 1032, 2048, 2056])
def test_exchange_of_many_rows(H, cap=641):
    """The exchange by one and two rows to a wave, with a source that sends nothing, one whose payload ends early, and an
    odd number of rows."""
    W, E_l = 5, 3
    g = torch.Generator(device=DEV).manual_seed(H)
    counts = torch.randint(0, cap + 1, (W, E_l), generator=torch.Generator().manual_seed(H)).to(torch.int32)
    counts[0, 0], counts[1, 2] = cap, 0
    world, rows = SimulatedWorld(W, rank=0), []
    for s in range(W):
        before, size = 7 * s, int(counts[s].sum())
        rows.append(torch.randn(before + size, H, generator=g, device=DEV).bfloat16())
        full = torch.zeros(W, E_l, dtype=torch.int32)
        full[0] = counts[s]
        if s != 3:
            world.post(s, rows[s], full.to(DEV), torch.tensor([before] + [0] * (W - 1), dtype=torch.int32, device=DEV))
    bufs = utils.alloc_shmem_buffers(None, W, E_l, cap, H, torch.bfloat16)
    bufs.token_buf.fill_(9.0)
    with simulated_world(world):
        out = custom_a2a(*world.sends[0], bufs.pca, bufs.token_buf, bufs.counts_ready, bufs.token_sync, None, W * E_l, cap)
    assert E_l * W * cap >= 8192
    for s in range(W):
        at = 7 * s
        for e in range(E_l):
            c = 0 if s == 3 else int(counts[s, e])
            assert torch.equal(out[e, s, :c], rows[s][at:at + c]) and not bool(out[e, s, c:].any()), (s, e)
            at += c


@pytest.mark.parametrize("H,cap", [(8, 3281), (640, 3277), (648, 3277), (504, 3276)])
def test_exchange_of_very_many_short_rows(H, cap):
    """Either side of where four rows go to a wave: 49152 slots, rows of 1280 bytes."""
    test_exchange_of_many_rows(H, cap)
