"""The reference-named operators (utils / baseline / layers) on the GPU: same call signatures,
return types, in-place behaviour and exceptions as the reference, results equal to the oracle."""
import numpy as np
import pytest
import torch

from helpers import O, assert_bits_equal, to_np

pytestmark = pytest.mark.gpu

from iris_testing_amd import utils  # noqa: E402
from iris_testing_amd.baseline import reorder_flat_to_token_buf  # noqa: E402
from iris_testing_amd.layers import SimulatedWorld, custom_a2a, expert, shuffle, simulated_world  # noqa: E402

DEV = "cuda"


def test_route_and_pack_padding_free_matches_oracle():
    # the reference's own generator conventions (utils.py:142-173): rand tokens, 0.001*randn router
    T, H, E, k, W = 192, 128, 8, 2, 4
    tokens = utils.gen_local_tokens(1, T, H, torch.float32, DEV, 0, 0)
    router = utils.gen_router(H, E, torch.float32, DEV, 0)
    payload, counts, offs, sizes = utils.route_and_pack_padding_free(tokens, router, k, W, E)
    o_payload, o_counts, o_offs, o_sizes = O.route_and_pack_padding_free(to_np(tokens), to_np(router), k, W, E)
    assert counts.dtype == torch.int32 and offs.dtype == torch.int32 and sizes.dtype == torch.int32
    assert_bits_equal(counts, o_counts, "send_counts")
    assert_bits_equal(offs, o_offs, "dst_offsets")
    assert_bits_equal(sizes, o_sizes, "dst_sizes")
    assert_bits_equal(payload, o_payload, "send_payload")
    assert_bits_equal(utils.build_expert_offsets(counts), O.build_expert_offsets(o_counts), "expert_offs")
    assert utils.compute_capacity_from_pca(counts) == O.compute_capacity_from_pca(o_counts)
    # agreement with the library routines the reference itself calls, on the same fp32 inputs
    p = torch.softmax(tokens.cpu() @ router.cpu(), dim=-1)
    ref_idx = torch.topk(p, k, dim=-1).indices
    same = (np.sort(ref_idx.numpy(), 1) == np.sort(O.route(to_np(tokens), to_np(router), k)[0], 1)).all(1).mean()
    print(f"top-k sets equal to torch.topk(softmax(x@W)) on {100 * same:.2f}% of tokens", flush=True)
    assert same > 0.99


def test_route_and_pack_errors_and_empty():
    tokens = torch.zeros((0, 64), dtype=torch.float32, device=DEV)
    router = torch.zeros((64, 8), dtype=torch.float32, device=DEV)
    payload, counts, offs, sizes = utils.route_and_pack_padding_free(tokens, router, 2, 4, 8)
    assert payload.shape == (0, 64) and int(counts.sum()) == 0
    with pytest.raises(AssertionError):
        utils.route_and_pack_padding_free(torch.zeros((4, 64), device=DEV), router, 2, 3, 8)  # 8 % 3 != 0
    with pytest.raises(AssertionError):
        utils.route_and_pack_padding_free(torch.zeros((4, 64)), router, 2, 4, 8)  # CPU tokens
    with pytest.raises(AssertionError):
        utils.build_expert_offsets(torch.zeros((4, 2), dtype=torch.int64, device=DEV))


@pytest.mark.parametrize("e_local,hidden_dim,cap", [(2, 128, 32), (4, 256, 16)])
def test_custom_a2a_uniform_pattern(e_local, hidden_dim, cap):
    """The reference's placement test (unit_tests.py:126-220) on a simulated 8-rank world: every src
    sends exactly `cap` rows to every (dst, expert); every block must land exactly.  Values are
    integer codes in fp32 (the reference's bf16 codes collide)."""
    W = 8
    experts = e_local * W
    dest_counts = torch.full((W, e_local), cap, device=DEV, dtype=torch.int32)
    dst_offsets = (torch.arange(W, device=DEV, dtype=torch.int32) * (e_local * cap)).contiguous()

    def payload_of(rank):
        rows = torch.arange(W * e_local * cap, device=DEV, dtype=torch.float32)
        return (rank * 1_000_000 + rows)[:, None].expand(-1, hidden_dim).contiguous()

    world = SimulatedWorld(W, rank=3)
    for src in range(W):
        if src != 3:
            world.post(src, payload_of(src), dest_counts, dst_offsets)
    bufs = utils.alloc_shmem_buffers(None, W, e_local, cap, hidden_dim, torch.float32)
    with simulated_world(world):
        out = custom_a2a(payload_of(3), dest_counts, dst_offsets, bufs.pca, bufs.token_buf, bufs.counts_ready,
                         bufs.token_sync, bufs.heap_bases, experts, cap)
    assert out.data_ptr() == bufs.token_buf.data_ptr()
    assert (bufs.pca == cap).all() and int(bufs.counts_ready) == W and (bufs.token_sync == W).all()
    for e in range(e_local):
        for src in range(W):
            start = 3 * (e_local * cap) + e * cap  # dst_offsets[rank] + e * cap
            assert torch.equal(out[e, src], payload_of(src)[start:start + cap]), (e, src)
    # shuffle removes nothing here (no padding) and orders by (expert, src, row)
    sh = shuffle(out, bufs.pca, bufs.token_sync)
    assert torch.equal(sh, out.reshape(-1, hidden_dim))
    with pytest.raises(RuntimeError):
        shuffle(out, bufs.pca, torch.zeros_like(bufs.token_sync))
    with pytest.raises(AssertionError):
        custom_a2a(payload_of(3), dest_counts, dst_offsets, bufs.pca, bufs.token_buf, bufs.counts_ready,
                   bufs.token_sync, None, experts + 1, cap)


@pytest.mark.parametrize("W,e_local,H,cap", [(2, 1, 8, 1), (4, 15, 520, 7), (70, 3, 2056, 5)])
def test_custom_a2a_ragged_world(W, e_local, H, cap):
    """Ragged and empty blocks, a silent source, more sources than one launch takes; an overflow raises and writes nothing."""
    rng = np.random.default_rng(W)
    counts = rng.integers(0, cap + 1, size=(W, W, e_local)).astype(np.int32)  # [src, dst, e]
    counts[0, 0, 0], counts[-1] = cap, 0
    rank, silent = W // 2, 0 if W > 2 else None
    world, rows = SimulatedWorld(W, rank=rank), {}
    for s in range(W):
        sizes = counts[s].sum(1)
        start = (np.cumsum(sizes) - sizes).astype(np.int32)
        rows[s] = torch.randn((int(sizes.sum()), H), device=DEV).bfloat16()
        if s != silent:
            world.post(s, rows[s], torch.from_numpy(counts[s]).to(DEV), torch.from_numpy(start).to(DEV))
    bufs = utils.alloc_shmem_buffers(None, W, e_local, cap, H, torch.bfloat16)
    bufs.token_buf.fill_(9.0)
    want_pca = counts[:, rank].T.copy()
    if silent is not None:
        want_pca[:, silent] = 0
    args = lambda c: (*world.sends[rank], bufs.pca, bufs.token_buf[:, :, :c], bufs.counts_ready, bufs.token_sync,  # noqa: E731
                      bufs.heap_bases, e_local * W, c)
    with simulated_world(world):
        if want_pca.max() == cap and cap > 1:
            small = bufs.token_buf[:, :, : cap - 1].contiguous()
            with pytest.raises(ValueError, match="capacity overflow"):
                custom_a2a(*world.sends[rank], bufs.pca, small, bufs.counts_ready, bufs.token_sync, None, e_local * W, cap - 1)
            assert (small == 9.0).all()
            for t in (bufs.pca, bufs.counts_ready, bufs.token_sync):
                assert not bool(t.any()), "an exchange that raises must not count or signal"
        custom_a2a(*args(cap))
    assert_bits_equal(bufs.pca, want_pca, "pca")
    assert int(bufs.counts_ready) == W and (bufs.token_sync == W).all()
    want = torch.zeros_like(bufs.token_buf)
    for s in range(W):
        sizes = counts[s].sum(1)
        at = int((np.cumsum(sizes) - sizes)[rank])
        for e in range(e_local):
            n = int(want_pca[e, s])
            want[e, s, :n] = rows[s][at:at + n]
            at += int(counts[s, rank, e])
    assert torch.equal(bufs.token_buf, want)
    assert torch.equal(shuffle(bufs.token_buf, bufs.pca, bufs.token_sync),
                       torch.cat([want[e, s, : int(want_pca[e, s])] for e in range(e_local) for s in range(W)]))


@pytest.mark.parametrize("W,over", [(4, 1), (64, 63), (70, 3), (70, 69), (130, 70)])
def test_custom_a2a_overflow_of_one_source_writes_nothing(W, over):
    """One source sends a row more than the capacity, all others fit: with more sources than a launch takes, its launch is one of
    several, and none of them may write."""
    cap, H = 2, 8
    counts = torch.ones((W, W), dtype=torch.int32)
    counts[over, 0] = cap + 1
    world, dev = SimulatedWorld(W, rank=0), lambda t: t.to(torch.int32).to(DEV)  # noqa: E731
    for s in range(W):
        n = counts[s]
        world.post(s, torch.full((int(n.sum()), H), float(s), device=DEV), dev(n[:, None]), dev(torch.cumsum(n, 0) - n))
    bufs = utils.alloc_shmem_buffers(None, W, 1, cap, H, torch.float32)
    args = lambda c, buf: (*world.sends[0], bufs.pca, buf, bufs.counts_ready, bufs.token_sync, None, W, c)  # noqa: E731
    bufs.token_buf.fill_(9.0)
    with simulated_world(world):
        with pytest.raises(ValueError, match="capacity overflow"):
            custom_a2a(*args(cap, bufs.token_buf))
        torch.cuda.synchronize()
        assert bool((bufs.token_buf == 9.0).all())
        for t in (bufs.pca, bufs.counts_ready, bufs.token_sync):
            assert not bool(t.any()), "an exchange that raises must not count or signal"
        with pytest.raises(ValueError, match="mismatch"):
            custom_a2a(*args(cap + 1, bufs.token_buf))
        out = custom_a2a(*args(cap + 1, torch.full((1, W, cap + 1, H), 9.0, device=DEV)))
    assert torch.equal(bufs.pca[0], dev(counts[:, 0])) and int(bufs.counts_ready) == W
    want = torch.arange(W, device=DEV)[:, None] * (torch.arange(cap + 1, device=DEV)[None] < counts[:, :1].to(DEV))
    assert torch.equal(out[0, :, :, 0], want.float()) and torch.equal(out[..., 0], out[..., H - 1])


def test_custom_a2a_payloads_at_odd_addresses():
    """A payload that is a slice of a flat buffer, at an address where no 16-byte load may start."""
    W, H = 3, 8
    counts = torch.tensor([[2], [1], [3]], dtype=torch.int32, device=DEV)
    starts = torch.tensor([0, 2, 3], dtype=torch.int32, device=DEV)
    flat = torch.randn(1 + 6 * H, device=DEV).bfloat16()
    world = SimulatedWorld(W, rank=1)
    for s in range(W):
        world.post(s, flat[1:].view(6, H), counts, starts)
    bufs = utils.alloc_shmem_buffers(None, W, 1, 3, H, torch.bfloat16)
    with simulated_world(world):
        out = custom_a2a(*world.sends[1], bufs.pca, bufs.token_buf, bufs.counts_ready, bufs.token_sync, None, W, 3)
    for s in range(W):
        assert torch.equal(out[0, s, :1], flat[1:].view(6, H)[2:3]) and bool((out[0, s, 1:] == 0).all())


def test_reorder_flat_to_token_buf_and_errors():
    rng = np.random.default_rng(0)
    W, E_l, H, CAP = 4, 3, 32, 9
    rc = rng.integers(0, CAP + 1, size=(W, E_l)).astype(np.int32)
    rc[1, 2] = 0
    flat = rng.standard_normal((int(rc.sum()), H)).astype(np.float32)
    tb = torch.full((E_l, W, CAP, H), 5.0, device=DEV)
    out = reorder_flat_to_token_buf(torch.from_numpy(flat).to(DEV), torch.from_numpy(rc).to(DEV), CAP, tb)
    want = O.reorder_flat_to_token_buf(flat, rc, CAP, np.empty((E_l, W, CAP, H), np.float32))
    assert out.data_ptr() == tb.data_ptr()
    assert_bits_equal(out, want, "token_buf")
    f, c = torch.from_numpy(flat).to(DEV), torch.from_numpy(rc).to(DEV)
    with pytest.raises(ValueError):
        reorder_flat_to_token_buf(f, c, CAP, torch.zeros((E_l, W, CAP + 1, H), device=DEV))  # wrong shape
    with pytest.raises(ValueError):
        reorder_flat_to_token_buf(f, c, int(rc.max()) - 1, torch.zeros((E_l, W, int(rc.max()) - 1, H), device=DEV))
    with pytest.raises(RuntimeError):
        reorder_flat_to_token_buf(f[:-1], c, CAP, tb)  # rows consumed != rows given
    with pytest.raises(ValueError):
        reorder_flat_to_token_buf(f, c.to(torch.int64), CAP, tb)
    with pytest.raises(ValueError):
        reorder_flat_to_token_buf(f.cpu(), c, CAP, tb)


def test_expert_layer_signature():
    rng = np.random.default_rng(1)
    cnt = np.array([17, 0, 40, 5, 66], dtype=np.int32)
    x = rng.standard_normal((int(cnt.sum()), 128)).astype(np.float32)
    w = rng.standard_normal((5, 128, 128)).astype(np.float32)
    out = expert(torch.from_numpy(x).to(DEV), torch.from_numpy(w).to(DEV), torch.from_numpy(cnt).to(DEV), 40)
    want = O.grouped_gemm(x, w, cnt, "f32")
    np.testing.assert_allclose(to_np(out), want, rtol=1e-2, atol=1e-3)  # the reference's intended rtol (unit_tests.py:237)
    np.testing.assert_allclose(to_np(out), want, rtol=1e-4, atol=1e-4)


def test_expert_layer_bf16_reuses_retiled_weights_until_they_change():
    """bf16 weights are re-tiled once per tensor version: a second call gives the same bits, an in-place update of
    the weights is seen by the next call, and the result is the oracle's."""
    import importlib
    expert_mod = importlib.import_module("iris_testing_amd.layers.expert")  # (the package re-exports the function under this name)
    rng = np.random.default_rng(2)
    cnt = np.array([300, 0, 45, 130], dtype=np.int32)
    S = int(cnt.sum())
    x = O.bf16_round(rng.standard_normal((S + 2, 256)).astype(np.float32))
    w = O.bf16_round((rng.standard_normal((4, 256, 192)) / 16).astype(np.float32))
    xt, wt = torch.from_numpy(x).bfloat16().to(DEV), torch.from_numpy(w).bfloat16().to(DEV)
    ct = torch.from_numpy(cnt).to(DEV)
    out1 = expert(xt, wt, ct, 4)
    n_cached = len(expert_mod._PACKED)
    out2 = expert(xt, wt, ct, 4)
    assert len(expert_mod._PACKED) == n_cached and torch.equal(out1, out2)
    want = O.grouped_gemm(x[:S], w, cnt, "bf16")
    got = to_np(out1)
    rms = float(np.sqrt((want.astype(np.float64) ** 2).mean()))
    assert (np.abs(got[:S] - want) <= 2.0 ** -7 * np.abs(want) + 2.0 ** -7 * rms).all()
    assert (got[S:] == 0).all()
    wt.mul_(2.0)  # exact in bf16: the product doubles exactly
    out3 = expert(xt, wt, ct, 4)
    assert torch.equal(out3, out1 * 2), "an in-place weight update must reach the kernel"


def test_benchmark_driver_point_and_overflow_report(capsys):
    """The environment-variable driver (the reference's benchmark.py knobs): one point with a CAPACITY smaller
    than the largest per-expert count prints the skip notice, still times, and its correctness report (fixed-M
    route against the padding-free flat route into token_buf) passes."""
    from iris_testing_amd import benchmark
    res = benchmark.run_point({"WORLD_SIZE": 4, "BATCH": 1, "SEQ": 320, "HIDDEN": 256, "TOPK": 2, "E_LOCAL": 3,
                               "CAPACITY": 8, "SEED": 7})
    out = capsys.readouterr().out
    assert "[SKIP] max_recv_count=" in out and "=== Correctness Report ===" in out and out.rstrip().endswith("PASS")
    assert res["ok"] and res["world"] == 4 and res["e_local"] == 3 and res["cap"] > 8
    assert res["source_ms"] > 0 and res["dest_ms"] > 0 and res["dest_direct_ms"] > 0


def test_benchmark_driver_point_is_the_oracles_layout():
    """The driver's CHECK compares two device routes with each other; here the buffers of the same point are held to
    the CPU oracle: pca, the zero-padded token_buf and the receive buffer it was filled from, bit for bit."""
    from iris_testing_amd import benchmark
    from iris_testing_amd.configs import gen_router, gen_shard_tokens
    res = benchmark.run_point({"WORLD_SIZE": 4, "BATCH": 1, "SEQ": 320, "HIDDEN": 256, "TOPK": 2, "E_LOCAL": 3,
                               "CAPACITY": 8, "SEED": 7}, keep=True)
    assert res["ok"] and res["baseline_agrees"]
    cfg = res["world_obj"].cfg
    xs = [to_np(gen_shard_tokens(cfg, s)) for s in range(cfg.world)]
    router = to_np(gen_router(cfg))
    shards = []
    for x in xs:
        idx = O.route(x, router, cfg.topk)[0]
        counts = O.send_counts(idx, cfg.world, cfg.experts)
        sizes, offs = O.dst_sizes_offsets(counts)
        shards.append((counts, sizes, offs, O.payload_positions(idx, cfg.experts)[1]))
    M = O.pair_capacity(np.stack([s[1] for s in shards]))
    assert M == res["M"]
    o_recv = np.stack([O.pack_fixed_m(O.send_payload(x, s[3]), s[2], s[1], M)[0] for x, s in zip(xs, shards)])
    o_rc = np.stack([s[0][0] for s in shards]).astype(np.int32)
    assert_bits_equal(res["recv"], o_recv, "receive buffer")
    assert_bits_equal(res["recv_counts"], o_rc, "recv_counts")
    o_tb, o_pca = O.recv_to_token_buf(o_recv, o_rc, res["cap"])
    assert_bits_equal(res["pca"], o_pca, "pca")
    assert_bits_equal(res["token_buf"], o_tb, "token_buf")


def test_benchmark_sweep_prints_the_figure_tables(capsys, monkeypatch):
    """One pass of SWEEP=topk at a small shape: one detailed row and one figure-style row per top-k value, the
    library baseline moving the same bytes as the kernels at every point."""
    from iris_testing_amd import benchmark
    for k, v in {"WORLD_SIZE": "4", "BATCH": "1", "SEQ": "256", "HIDDEN": "256", "E_LOCAL": "4", "SEED": "3"}.items():
        monkeypatch.setenv(k, v)
    monkeypatch.setattr(benchmark, "WARMUP", 1)
    monkeypatch.setattr(benchmark, "ITERS", 2)
    rows = benchmark.run_sweep("topk")
    out = capsys.readouterr().out.splitlines()
    assert [v for v, _ in rows] == [1, 2, 4, 8] and all(r["baseline_agrees"] for _, r in rows)
    head = [i for i, l in enumerate(out) if l.startswith("=== all2all_topk_change")]
    assert len(head) == 1
    fig = out[head[0] + 2: head[0] + 6]
    assert [int(l.split()[0]) for l in fig] == [1, 2, 4, 8]
    for l in fig:
        cols = l.split()
        assert len(cols) == 5 and float(cols[1]) > 0 and float(cols[2]) > 0 and cols[3].endswith("x") and cols[4] == "yes"
    detail = [l for l in out[:head[0]] if l.split() and l.split()[0].isdigit()]
    assert len(detail) == 4 and all(len(l.split()) == 9 for l in detail)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_shuffle_backward_puts_rows_back_and_zeroes_the_padding(dtype):
    """Gradient of the expert-major unpack (empty in the reference, token_shuffle.py:58-60): the shuffle is a row
    permutation that drops the padding, so the gradient of token_buf[e, src, j] is the gradient of the row it
    went to, and zero in the padding -- exact, whatever the dtype."""
    rng = np.random.default_rng(11)
    E_l, W, CAP, H = 3, 4, 9, 64
    pca = rng.integers(0, CAP + 1, size=(E_l, W)).astype(np.int32)
    pca[1, 2] = 0
    S = int(pca.sum())
    tb = torch.from_numpy(rng.standard_normal((E_l, W, CAP, H)).astype(np.float32)).to(DEV).to(dtype).requires_grad_(True)
    out = shuffle(tb, torch.from_numpy(pca).to(DEV), None)
    assert out.shape == (S, H)
    g = torch.from_numpy(rng.standard_normal((S, H)).astype(np.float32)).to(DEV).to(dtype)
    out.backward(g)
    want = np.zeros((E_l, W, CAP, H), np.float32)
    gn, r = to_np(g), 0
    for e in range(E_l):
        for s in range(W):
            want[e, s, :pca[e, s]] = gn[r:r + pca[e, s]]
            r += pca[e, s]
    assert_bits_equal(tb.grad, want if dtype == torch.float32 else torch.from_numpy(want).to(dtype), "grad of token_buf")
    # nothing received: the gradient is all padding
    tb0 = torch.zeros((2, 2, 3, 64), device=DEV, dtype=dtype, requires_grad=True)
    out0 = shuffle(tb0, torch.zeros((2, 2), dtype=torch.int32, device=DEV), None)
    out0.backward(torch.zeros_like(out0))
    assert out0.shape == (0, 64) and bool((tb0.grad == 0).all())


@pytest.mark.parametrize("dtype,H,F,cnt", [(torch.float32, 96, 72, (70, 0, 45)), (torch.bfloat16, 128, 192, (70, 0, 45)),
                                           (torch.bfloat16, 256, 320, (300, 17, 0, 129))])
def test_expert_backward_matches_float64_autograd(dtype, H, F, cnt):
    """Gradients of the grouped GEMM layer (not implemented in the reference, layers/expert.py:62-64) against
    float64 autograd of  out[rows of g] = tokens[rows of g] @ weights[g]  on the CPU -- parity unpinned by the
    reference, pinned by the mathematics.  Rows past the counted total take no part and get a zero gradient."""
    rng = np.random.default_rng(H + F)
    cnt = np.array(cnt, dtype=np.int32)
    S = int(cnt.sum()) + 5
    x = torch.from_numpy(rng.standard_normal((S, H)).astype(np.float32)).to(dtype)
    w = torch.from_numpy((rng.standard_normal((len(cnt), H, F)) * H ** -0.5).astype(np.float32)).to(dtype)
    g = torch.from_numpy(rng.standard_normal((S, F)).astype(np.float32)).to(dtype)
    xd, wd = x.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    out = expert(xd, wd, torch.from_numpy(cnt).to(DEV), int(cnt.sum()))
    out.backward(g.to(DEV))
    x64, w64 = x.double().requires_grad_(True), w.double().requires_grad_(True)
    parts, r = [], 0
    for e, c in enumerate(cnt):
        parts.append(x64[r:r + c] @ w64[e])
        r += c
    ref = torch.cat(parts + [torch.zeros((S - r, F), dtype=torch.float64)])
    ref.backward(g.double())
    tol = 1e-4 if dtype == torch.float32 else 2.0 ** -6
    for name, got, want in (("d tokens", xd.grad, x64.grad), ("d weights", wd.grad, w64.grad)):
        got, want = got.double().cpu(), want
        scale = float(want.abs().max()) + 1e-30
        err = float((got - want).abs().max()) / scale
        print(f"{name}: max error / max |gradient| = {err:.2e}", flush=True)
        assert err < tol, f"{name}: {err}"
    assert bool((xd.grad[int(cnt.sum()):] == 0).all()) and bool((wd.grad[cnt == 0] == 0).all())
