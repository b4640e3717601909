"""GPU parity, floating-point part of the path: grouped GEMM, expert MLP (GELU / SiLU / SwiGLU,
fp32 / bf16 / fp8) and the end-to-end combine.  Tolerances are stated per test; max-abs and
relative errors are printed."""
import dataclasses

import numpy as np
import pytest
import torch

from helpers import O, assert_bits_equal, err_stats, gemm_parts, to_np

pytestmark = pytest.mark.gpu

from iris_testing_amd import ops  # noqa: E402
from iris_testing_amd.layers.expert import ExpertWeights, expert_mlp  # noqa: E402

DEV = "cuda"

# bf16 outputs: the GPU and the oracle round the same fp32-accumulated value to bf16; they can differ
# by accumulation order only, i.e. by at most one bf16 rounding step (at most 2^-7 of the value) plus the
# propagated rounding of the hidden activation.  Bound used: |err| <= BF16_RTOL*|ref| + BF16_ATOL*rms(ref).
BF16_RTOL, BF16_ATOL = 2.0 ** -7, 2.0 ** -7
F32_RTOL, F32_ATOL = 1e-4, 1e-5
# fp8 end to end (see test_expert_mlp_fp8): a one-bit difference in a hidden row's amax re-codes a few
# per cent of that row in fp8 (steps of 2^-3 relative), so single outputs may move by ~0.1 rms.
FP8_RTOL, FP8_ATOL = 2.0 ** -4, 2.0 ** -3


def _check(got, want, rtol, atol, what):
    mx, mx_rms, rel = err_stats(got, want)
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    print(f"{what}: max-abs {mx:.3e}  max-abs/rms {mx_rms:.3e}  max-rel(|ref|>rms/8) {rel:.3e}", flush=True)
    bound = rtol * np.abs(want) + atol * rms
    bad = np.abs(got.astype(np.float64) - want) > bound
    assert not bad.any(), f"{what}: {bad.sum()} of {bad.size} outside tolerance (max-abs {mx}, rms {rms})"


def _groups(rng, E_l, S_target, with_zero=True):
    cnt = rng.multinomial(S_target, rng.dirichlet(np.ones(E_l))).astype(np.int32)
    if with_zero and E_l > 2:
        cnt[1] = 0
    return cnt


def _randn(rng, *shape, scale=1.0, dtype="bf16"):
    a = (rng.standard_normal(shape) * scale).astype(np.float32)
    return O.bf16_round(a) if dtype == "bf16" else a


def _t(a, dtype):
    return torch.from_numpy(a).to({"bf16": torch.bfloat16, "f32": torch.float32}[dtype]).to(DEV)


@pytest.mark.parametrize("dtype,E_l,K,N,S", [("bf16", 2, 128, 256, 300), ("bf16", 5, 192, 328, 777),
                                              ("bf16", 1, 4096, 512, 1500), ("bf16", 32, 256, 256, 3000),
                                              ("bf16", 3, 64, 264, 1000),  # K = one pair of LDS ring stages
                                              ("f32", 2, 24, 48, 99), ("f32", 5, 128, 128, 333)])
def test_grouped_gemm(dtype, E_l, K, N, S):
    """expert(tokens, weights, cnt): one GEMM per group, the shapes the reference meant to test
    ((2,24,48), (5,128,128), unit_tests.py:247-248) and MFMA-sized ones."""
    rng = np.random.default_rng(E_l * 1000 + K)
    cnt = _groups(rng, E_l, S)
    S_tot = int(cnt.sum())
    x = _randn(rng, S_tot + 3, K, dtype=dtype)
    w = _randn(rng, E_l, K, N, scale=K ** -0.5, dtype=dtype)
    out = ops.grouped_gemm(_t(x, dtype), _t(w, dtype), torch.from_numpy(cnt).to(DEV))
    want = O.grouped_gemm(x, w, cnt, dtype)
    r, a = (BF16_RTOL, BF16_ATOL) if dtype == "bf16" else (F32_RTOL, F32_ATOL)
    _check(to_np(out)[:S_tot], want[:S_tot].astype(np.float64), r, a, f"grouped_gemm {dtype}")
    assert (to_np(out)[S_tot:] == 0).all(), "rows past sum(cnt) must stay untouched"


@pytest.mark.parametrize("act,H,F,S", [("silu", 20, 33, 70), ("swiglu", 127, 66, 65), ("gelu", 132, 260, 31),
                                       ("swiglu", 260, 1100, 2300), ("gelu", 97, 1026, 3100)])
def test_fp32_expert_at_tile_edges(act, H, F, S):
    """Both tile sizes of the fp32 GEMM (32 x 32 for few tiles, 64 x 64 for many), rows, K and N that fill no tile, slab or 16-byte
    unit, and an expert without rows."""
    rng = np.random.default_rng(H + F)
    E_l = 3
    cnt = _groups(rng, E_l, S)
    cnt[1] = 0
    S_tot = int(cnt.sum())
    x = _randn(rng, S_tot, H, dtype="f32")
    w1, w2 = _randn(rng, E_l, H, F, scale=H ** -0.5, dtype="f32"), _randn(rng, E_l, F, H, scale=F ** -0.5, dtype="f32")
    wu = _randn(rng, E_l, H, F, scale=H ** -0.5, dtype="f32") if act == "swiglu" else None
    c = torch.from_numpy(cnt).to(DEV)
    hid = ops.grouped_gemm(_t(x, "f32"), _t(w1, "f32"), c)
    _check(to_np(hid), O.grouped_gemm(x, w1, cnt, "f32").astype(np.float64), F32_RTOL, F32_ATOL, "fp32 GEMM")
    if H % 4 == 0 and F % 4 == 0:
        ew = ExpertWeights.prepare(act, _t(w1, "f32"), _t(w2, "f32"), None if wu is None else _t(wu, "f32"))
        y = expert_mlp(_t(x, "f32"), ew, c)
        _check(to_np(y), O.expert_mlp(x, cnt, w1, w2, act, "f32", w_up=wu).astype(np.float64), F32_RTOL, F32_ATOL, "fp32 MLP")


def test_grouped_gemm_identity_is_exact():
    """Identity / one-hot weights: the GEMM must reproduce (permute) its input bit for bit."""
    rng = np.random.default_rng(3)
    E_l, K = 3, 256
    cnt = np.array([130, 0, 259], dtype=np.int32)
    x = _randn(rng, int(cnt.sum()), K)
    perm = rng.permutation(K)
    w = np.zeros((E_l, K, K), dtype=np.float32)
    w[0] = np.eye(K)
    w[1] = np.eye(K)
    w[2][perm, np.arange(K)] = 1.0  # out[:, j] = x[:, perm[j]]
    out = to_np(ops.grouped_gemm(_t(x, "bf16"), _t(w, "bf16"), torch.from_numpy(cnt).to(DEV)))
    assert_bits_equal(out[:130], x[:130], "identity expert")
    assert_bits_equal(out[130:], x[130:][:, perm], "permutation expert")


MLP_CASES = [
    # dtype, act, E_l, H, F, S
    ("f32", "gelu", 2, 256, 512, 512),      # plumbing workload's expert
    ("f32", "swiglu", 3, 64, 96, 200),
    ("bf16", "silu", 2, 2048, 4096, 443),   # small workload's expert at its real shape
    ("bf16", "gelu", 4, 256, 512, 900),
    ("bf16", "swiglu", 1, 4096, 1792, 1300),  # Mixtral-style expert, F cut to 1/8 for CPU time
    ("bf16", "swiglu", 32, 7168, 256, 2500),  # fine-grained: 32 small groups, F cut to 1/8
    ("bf16", "swiglu", 15, 2048, 1408, 3000),
]


@pytest.mark.parametrize("dtype,act,E_l,H,F,S", MLP_CASES)
def test_expert_mlp(dtype, act, E_l, H, F, S):
    rng = np.random.default_rng(H + F + E_l)
    cnt = _groups(rng, E_l, S)
    S_tot = int(cnt.sum())
    x = _randn(rng, S_tot, H, dtype=dtype)
    w1 = _randn(rng, E_l, H, F, scale=H ** -0.5, dtype=dtype)
    w2 = _randn(rng, E_l, F, H, scale=F ** -0.5, dtype=dtype)
    wu = _randn(rng, E_l, H, F, scale=H ** -0.5, dtype=dtype) if act == "swiglu" else None
    ew = ExpertWeights.prepare(act, _t(w1, dtype), _t(w2, dtype), None if wu is None else _t(wu, dtype))
    out = to_np(expert_mlp(_t(x, dtype), ew, torch.from_numpy(cnt).to(DEV)))
    want = O.expert_mlp(x, cnt, w1, w2, act, dtype, w_up=wu)
    r, a = (BF16_RTOL, BF16_ATOL) if dtype == "bf16" else (F32_RTOL, F32_ATOL)
    _check(out, want.astype(np.float64), r, a, f"expert_mlp {dtype} {act} E_l={E_l} H={H} F={F}")


@pytest.mark.parametrize("E_l,K,N,S,act", [(3, 128, 264, 900, "none"), (4, 256, 512, 1500, "swiglu"),
                                           # more tiles than workgroups, short K: the ring runs on from tile to tile (K = 192,
                                           # 320: six and ten stages, so consecutive tiles start in different ring slots) or,
                                           # with four stages (K = 128), every tile is set up on its own
                                           (3, 128, 2048, 9000, "none"), (2, 192, 2048, 9500, "none"), (5, 320, 1024, 17000, "swiglu"),
                                           (2, 64, 2048, 9100, "none")])  # two stages per tile: the shortest K
def test_grouped_gemm_mapped(E_l, K, N, S, act):
    """Row indirection on both sides: logical row r is read from a scattered row of a larger buffer and its
    result is written to a scattered row of a larger output.  The result must be bit for bit what the plain
    kernel produces on the gathered rows (same arithmetic), rows outside the map stay untouched, and the
    plain kernel itself is held to the oracle."""
    from iris_testing_amd import _lib as L
    rng = np.random.default_rng(K + N + E_l)
    cnt = _groups(rng, E_l, S)
    S_tot = int(cnt.sum())
    n_in, n_out = S_tot + 500, S_tot + 300
    a_map = rng.permutation(n_in)[:S_tot].astype(np.int32)
    c_map = rng.permutation(n_out)[:S_tot].astype(np.int32)
    base = _randn(rng, n_in, K)
    w = _randn(rng, E_l, K, N, scale=K ** -0.5)
    wu = _randn(rng, E_l, K, N, scale=K ** -0.5) if act == "swiglu" else None
    packed = ops.prepack_weights(_t(w, "bf16"), None if wu is None else _t(wu, "bf16"))
    cnt_t = torch.from_numpy(cnt).to(DEV)
    base_t = _t(base, "bf16")
    gathered = base_t[torch.from_numpy(a_map).long().to(DEV)].contiguous()
    plain = torch.empty((S_tot, N), dtype=torch.bfloat16, device=DEV)
    L.check(L.lib().moe_grouped_gemm_packed(L.ptr(gathered), L.ptr(packed), L.ptr(cnt_t), S_tot, K, N, E_l, L.ACT[act],
                                            L.ptr(plain), L.stream_ptr()))
    out = torch.full((n_out, N), -7.0, dtype=torch.bfloat16, device=DEV)
    ops.grouped_gemm_mapped(base_t, torch.from_numpy(a_map).to(DEV), packed, cnt_t, S_tot, N, act, out,
                            torch.from_numpy(c_map).to(DEV))
    torch.cuda.synchronize()
    got = out[torch.from_numpy(c_map).long().to(DEV)]
    assert torch.equal(got.view(torch.int16), plain.view(torch.int16)), "mapped GEMM differs from the plain one"
    untouched = np.setdiff1d(np.arange(n_out), c_map)
    assert bool((out[torch.from_numpy(untouched).to(DEV)] == -7.0).all()), "rows outside the map were written"
    if act == "none":
        _check(to_np(plain), O.grouped_gemm(base[a_map], w, cnt, "bf16"), BF16_RTOL, BF16_ATOL, "gathered GEMM")
    # argument checks happen before any launch
    lib = L.lib()
    rc = lib.moe_grouped_gemm_mapped(L.ptr(base_t), n_in, None, L.ptr(packed), L.ptr(cnt_t), S_tot, K + 8, N, E_l, 0,
                                     L.ptr(out), n_out, None, None, 0, L.stream_ptr())
    assert rc != 0 and b"K" in lib.moe_last_error()
    rc = lib.moe_grouped_gemm_mapped(L.ptr(base_t), 1 << 30, L.ptr(torch.from_numpy(a_map).to(DEV)), L.ptr(packed),
                                     L.ptr(cnt_t), S_tot, K, N, E_l, 0, L.ptr(out), n_out, None, None, 0, L.stream_ptr())
    assert rc != 0 and b"4 GiB" in lib.moe_last_error()


def test_grouped_gemm_counts_that_claim_more_rows_than_there_are():
    """Row counts are device data the kernels cannot trust: a group that claims rows past S_rows is cut there (its tiles
    beyond have no rows and are skipped by the walk), the groups after it get nothing, and nothing is read or written
    past row S_rows."""
    rng = np.random.default_rng(77)
    E_l, K, N, S_rows = 3, 256, 1024, 700
    cnt = np.array([300, 5000, 40], dtype=np.int32)
    x = _randn(rng, S_rows, K)
    w = _randn(rng, E_l, K, N, scale=K ** -0.5)
    packed = ops.prepack_weights(_t(w, "bf16"))
    out = torch.full((S_rows + 300, N), -7.0, dtype=torch.bfloat16, device=DEV)
    ops.grouped_gemm_mapped(_t(x, "bf16"), None, packed, torch.from_numpy(cnt).to(DEV), S_rows, N, "none", out)
    torch.cuda.synchronize()
    want = O.grouped_gemm(x, w, np.array([300, 400, 0], dtype=np.int32), "bf16")
    _check(to_np(out[:S_rows]), want, BF16_RTOL, BF16_ATOL, "clamped groups")
    assert bool((out[S_rows:] == -7.0).all()), "rows past S_rows were written"


@pytest.mark.parametrize("E_l,K,N,rows,act", [(2, 512, 1024, (200, 150), "none"), (2, 2048, 4096, (230, 213), "silu"),
                                              (3, 1024, 512, (300, 0, 77), "swiglu"), (1, 4096, 2048, (443,), "gelu"),
                                              (1, 1024, 4096, (20836,), "swiglu"),
                                              # cut into parts: few tiles, and the last round of a launch of large ones
                                              (2, 4096, 512, (70, 33), "swiglu"), (3, 8192, 256, (40, 0, 5), "none"),
                                              (1, 4096, 2048, (8448,), "silu")])
def test_grouped_gemm_k_split_of_the_last_round(E_l, K, N, rows, act):
    """With a partial-sum workspace the small tiles that a launch, or its last round, comes to are cut along K where rows are long, and the
    last part of a tile to finish adds the sums.  The result must be the oracle's within the bf16 bar, within a bf16 rounding step of
    the unsplit kernel's (only the fp32 summation order differs), identical from call to call, and rows outside the map stay
    untouched."""
    rng = np.random.default_rng(K + N + len(rows))
    cnt = np.array(rows, dtype=np.int32)
    height, whole, parts = gemm_parts(cnt, K, N, act)
    assert (parts > 1) == (K >= 4096) and (height >= 128) == (whole > 0) and gemm_parts(cnt, K, N, act, workspace=False)[2] == 1
    S_tot = int(cnt.sum())
    x = _randn(rng, S_tot, K)
    w = _randn(rng, E_l, K, N, scale=K ** -0.5)
    wu = _randn(rng, E_l, K, N, scale=K ** -0.5) if act == "swiglu" else None
    packed = ops.prepack_weights(_t(w, "bf16"), None if wu is None else _t(wu, "bf16"))
    cnt_t, x_t = torch.from_numpy(cnt).to(DEV), _t(x, "bf16")
    c_map = torch.from_numpy(rng.permutation(S_tot + 64)[:S_tot].astype(np.int32)).to(DEV)
    ws = ops.gemm_part_workspace(DEV)
    ws.fill_(float("nan"))  # stale contents must not matter
    plain = torch.full((S_tot + 64, N), -7.0, dtype=torch.bfloat16, device=DEV)
    ops.grouped_gemm_mapped(x_t, None, packed, cnt_t, S_tot, N, act, plain, c_map)
    split = torch.full((S_tot + 64, N), -7.0, dtype=torch.bfloat16, device=DEV)
    ops.grouped_gemm_mapped(x_t, None, packed, cnt_t, S_tot, N, act, split, c_map, part_ws=ws)
    again = torch.full((S_tot + 64, N), -7.0, dtype=torch.bfloat16, device=DEV)
    ws.fill_(3.0)
    ops.grouped_gemm_mapped(x_t, None, packed, cnt_t, S_tot, N, act, again, c_map, part_ws=ws)
    torch.cuda.synchronize()
    assert torch.equal(split.view(torch.int16), again.view(torch.int16)), "the K split is not reproducible"
    a, b = split.float(), plain.float()
    assert bool(torch.isfinite(a).all())
    step = 2.0 ** -7 * torch.maximum(a.abs(), b.abs()) + 1e-6  # one bf16 rounding step either way
    assert bool(((a - b).abs() <= 2 * step).all()), "split and unsplit sums differ by more than a rounding step"
    untouched = np.setdiff1d(np.arange(S_tot + 64), to_np(c_map))
    assert bool((split[torch.from_numpy(untouched).to(DEV)] == -7.0).all()), "rows outside the map were written"
    got = to_np(split[c_map.long()])
    if act == "none":
        _check(got, O.grouped_gemm(x, w, cnt, "bf16"), BF16_RTOL, BF16_ATOL, "K-split GEMM")
    differs = int((split.view(torch.int16) != plain.view(torch.int16)).sum().item())
    print(f"K split: {differs} of {split.numel()} outputs differ in the last bits from the unsplit kernel", flush=True)


@pytest.mark.parametrize("E_l,K,N,rows,act", [(3, 256, 384, (300, 0, 77), "swiglu"), (2, 512, 256, (70, 333), "gelu"),
                                              (1, 1024, 2048, (443,), "silu"), (1, 1024, 4096, (20836,), "swiglu"),
                                              (2, 4096, 512, (60, 40), "swiglu"), (1, 4096, 256, (33,), "gelu")])
@pytest.mark.parametrize("split", [False, True], ids=["whole_tiles", "k_split"])
def test_grouped_gemm_act_keep_also_stores_the_pre_activations(E_l, K, N, rows, act, split):
    """The launch that keeps the values before the activation for the backward pass: its output is bit for bit that
    of the ordinary launch, and what it keeps is bit for bit what a launch without activation produces (SwiGLU: in
    the fused gate / up column order) -- with and without the K split, which long rows get."""
    rng = np.random.default_rng(K + N + len(rows))
    cnt = np.array(rows, dtype=np.int32)
    assert (gemm_parts(cnt, K, N, act, workspace=split)[2] > 1) == (split and K >= 4096)
    S_tot = int(cnt.sum())
    x = _randn(rng, S_tot, K)
    w = _randn(rng, E_l, K, N, scale=K ** -0.5)
    wu = _randn(rng, E_l, K, N, scale=K ** -0.5) if act == "swiglu" else None
    packed = ops.prepack_weights(_t(w, "bf16"), None if wu is None else _t(wu, "bf16"))
    cnt_t, x_t = torch.from_numpy(cnt).to(DEV), _t(x, "bf16")
    ws = ops.gemm_part_workspace(DEV) if split else None
    NP = 2 * N if act == "swiglu" else N
    plain = torch.full((S_tot, N), -7.0, dtype=torch.bfloat16, device=DEV)
    ops.grouped_gemm_mapped(x_t, None, packed, cnt_t, S_tot, N, act, plain, part_ws=ws)
    pre_ref = torch.full((S_tot, NP), -7.0, dtype=torch.bfloat16, device=DEV)
    ops.grouped_gemm_mapped(x_t, None, packed, cnt_t, S_tot, NP, "none", pre_ref, part_ws=ws)
    out = torch.full((S_tot, N), -7.0, dtype=torch.bfloat16, device=DEV)
    pre = torch.full((S_tot, NP), -7.0, dtype=torch.bfloat16, device=DEV)
    ops.grouped_gemm_act_keep(x_t, packed, cnt_t, S_tot, N, act, out, pre, part_ws=ws)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), plain.view(torch.int16)), "the output changed with the second store"
    assert torch.equal(pre.view(torch.int16), pre_ref.view(torch.int16)), "kept pre-activations differ from a launch without activation"
    # and they are the oracle's product
    want = O.grouped_gemm(x, w, cnt, "bf16")
    got = to_np(pre)
    if act == "swiglu":  # fused order: 32 gate columns, their 32 up columns, ...
        got = got.reshape(S_tot, N // 32, 2, 32)[:, :, 0, :].reshape(S_tot, N)
    _check(got, want, BF16_RTOL, BF16_ATOL, "kept pre-activations")


@pytest.mark.parametrize("W,E_l,M,H,F,fill", [(4, 3, 300, 128, 256, "ragged"), (8, 5, 64, 256, 128, "empty"),
                                              (2, 1, 40, 128, 128, "full")])
def test_copy_free_destination_equals_operator_chain(W, E_l, M, H, F, fill):
    """unpack -> GEMM -> GEMM -> return pack against row map -> gathering GEMM -> scattering GEMM -> zeroed
    padding rows, on receive buffers with empty (source, expert) segments, with nothing received at all,
    and with every slot full: identical returned buffers, bit for bit."""
    rng = np.random.default_rng(W * 100 + E_l)
    if fill == "empty":
        rc = np.zeros((W, E_l), np.int32)
    else:
        rc = np.zeros((W, E_l), np.int32)
        for s_ in range(W):
            tot = M if fill == "full" else int(rng.integers(0, M + 1))
            rc[s_] = rng.multinomial(tot, rng.dirichlet(np.ones(E_l)))
        if fill == "ragged":
            rc[1, :] = 0      # a source that sent nothing
            rc[:, 0] = 0      # an expert that got nothing
    S = int(rc.sum())
    recv = _t(_randn(rng, W, M, H), "bf16")
    rc_t = torch.from_numpy(rc).to(DEV)
    w1 = _t(_randn(rng, E_l, H, F, scale=H ** -0.5), "bf16")
    w2 = _t(_randn(rng, E_l, F, H, scale=F ** -0.5), "bf16")
    p1, p2 = ops.prepack_weights(w1), ops.prepack_weights(w2)
    S_rows = max(S, 1)
    from iris_testing_amd import _lib as L
    # operator chain
    rows, cnt = ops.unpack_expert_major(recv, rc_t, S_rows)
    hid = torch.zeros((S_rows, F), dtype=torch.bfloat16, device=DEV)
    y = torch.zeros((S_rows, H), dtype=torch.bfloat16, device=DEV)
    lib = L.lib()
    L.check(lib.moe_grouped_gemm_packed(L.ptr(rows), L.ptr(p1), L.ptr(cnt), S, H, F, E_l, L.ACT["gelu"], L.ptr(hid), L.stream_ptr()))
    L.check(lib.moe_grouped_gemm_packed(L.ptr(hid), L.ptr(p2), L.ptr(cnt), S, F, H, E_l, 0, L.ptr(y), L.stream_ptr()))
    want = ops.return_pack(y, rc_t, M)
    # copy-free chain
    row_map, cnt2 = ops.recv_row_map(rc_t, M, S)
    hid2 = torch.zeros((S_rows, F), dtype=torch.bfloat16, device=DEV)
    got = torch.full((W, M, H), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.grouped_gemm_mapped(recv.view(W * M, H), row_map, p1, cnt2, S, F, "gelu", hid2)
    ops.grouped_gemm_mapped(hid2, None, p2, cnt2, S, H, "none", got.view(W * M, H), row_map)
    ops.zero_padding_rows(got, rc_t)
    torch.cuda.synchronize()
    assert torch.equal(cnt, cnt2)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("R,C", [(5, 64), (300, 2048), (77, 1408), (40, 4096), (33, 7168), (9, 16384)])  # every register-held row length and the streamed one
def test_quantize_rows_fp8_bit_exact(R, C):
    rng = np.random.default_rng(R)
    x = _randn(rng, R, C, scale=3.0)
    x[1] = 0.0  # an all-zero row -> scale 1, codes 0
    q, s = ops.quantize_rows_fp8(_t(x, "bf16"))
    oq, osc = O.quantize_rows_fp8(x)
    assert_bits_equal(s, osc, "row scales")
    assert_bits_equal(q, oq, "fp8 codes")


def _hidden_codes_close(hq_gpu, hsc_gpu, hq_want, hsc_want, what, min_same=0.995):
    """The GPU's block-quantised hidden activation against the oracle's: fp32 sums in another order (and the hardware's exp /
    reciprocal) move a value that sits on an e4m3 rounding boundary to the neighbouring code, and a block maximum that sits on a
    power-of-two boundary to the neighbouring scale; everything else must be identical.  Bounds: at least `min_same` of the
    codes and 99.9 % of the scale bytes identical, no scale byte off by more than one, every dequantised value within one
    e4m3 step of the oracle's or within 2^-12 of its block's maximum."""
    same_b = hsc_gpu == hsc_want
    assert same_b.mean() >= 0.999, f"{what}: only {same_b.mean():.5f} of the block scales agree"
    assert np.abs(hsc_gpu.astype(np.int32) - hsc_want.astype(np.int32)).max() <= 1, f"{what}: a block scale is off by more than one"
    same_q = (hq_gpu == hq_want) & np.repeat(same_b, 32, axis=1)
    got, want = O.dequantize_blocks_fp8(hq_gpu, hsc_gpu).astype(np.float64), O.dequantize_blocks_fp8(hq_want, hsc_want).astype(np.float64)
    # (a value far below its block's maximum is a sum that nearly cancels: its fp32 summation noise, relative to the block
    # maximum 448 X, is what bounds it -- 2^-12 of that, a few dozen of the block's smallest steps)
    step = 2.0 ** -3 * np.abs(want) + 2.0 ** -12 * 448.0 * np.repeat(np.exp2(hsc_want.astype(np.float64) - 127.0), 32, axis=1)
    bad = np.abs(got - want) > step + 1e-30
    print(f"{what}: {same_q.mean():.6f} of the codes identical, {same_b.mean():.6f} of the block scales", flush=True)
    assert same_q.mean() >= min_same, f"{what}: only {same_q.mean():.5f} of the codes agree"
    if bad.any():
        at = np.argwhere(bad)[:5]
        detail = "; ".join(f"[{r},{c}] codes {hq_gpu[r, c]:#04x} / {hq_want[r, c]:#04x}, scale byte {hsc_want[r, c // 32]}, "
                           f"values {got[r, c]:.6g} / {want[r, c]:.6g}" for r, c in at)
        raise AssertionError(f"{what}: {int(bad.sum())} hidden activations are more than an e4m3 step from the oracle's: {detail}")


@pytest.mark.parametrize("E_l,H,F,S", [(2, 256, 384, 400), (15, 2048, 1408, 2500), (1, 128, 128, 700)])
def test_expert_mlp_fp8(E_l, H, F, S):
    """The two GEMMs are checked separately: the first one's block-quantised hidden activation (codes and scale bytes)
    against the oracle's, identical but for values on a rounding boundary; the second one with the tight bf16 bound
    against the oracle fed with the GPU's own codes and scales.  End to end the bound is looser on purpose: a hidden
    value that takes the neighbouring e4m3 code moves the outputs of its row, which is a property of the quantisation,
    not of the kernels."""
    rng = np.random.default_rng(H + F)
    cnt = _groups(rng, E_l, S)
    S_tot = int(cnt.sum())
    x = _randn(rng, S_tot, H)
    wg = _randn(rng, E_l, H, F, scale=H ** -0.5)
    wu = _randn(rng, E_l, H, F, scale=H ** -0.5)
    wd = _randn(rng, E_l, F, H, scale=F ** -0.5)
    (gq, gs), (uq, us), (dq, ds) = (O.quantize_cols_fp8(w) for w in (wg, wu, wd))
    tq = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    ew = ExpertWeights.prepare_fp8(tq(gq), tq(gs), tq(uq), tq(us), tq(dq), tq(ds))
    ws = ops.fp8_workspace(S_tot, H, F, DEV)
    sg, su, sd = ew.scales
    out = to_np(ops.grouped_mlp_fp8(_t(x, "bf16"), torch.from_numpy(cnt).to(DEV), F, ew.w1, sg, su, ew.w2, sd, ws=ws))
    hq_gpu, hsc_gpu = to_np(ws["hq"]), to_np(ws["hsc"])
    hq_want, hsc_want = O.expert_up_fp8(x, cnt, gq, gs, uq, us)
    _hidden_codes_close(hq_gpu, hsc_gpu, hq_want, hsc_want, f"fp8 gate/up GEMM + SwiGLU + block quantisation E_l={E_l} H={H} F={F}")
    assert torch.equal(ops.dequantize_hidden_fp8(ws["hq"], ws["hsc"]).cpu(), torch.from_numpy(O.dequantize_blocks_fp8(hq_gpu, hsc_gpu)))
    y_from_gpu_h = O.expert_down_fp8(hq_gpu, hsc_gpu, cnt, dq, ds)
    _check(out, y_from_gpu_h.astype(np.float64), BF16_RTOL, BF16_ATOL, f"fp8 down GEMM E_l={E_l} H={H} F={F}")
    # the gate of the gated return, folded into the channel scale
    gate = rng.random(S_tot).astype(np.float32)
    out_g = to_np(ops.grouped_mlp_fp8(_t(x, "bf16"), torch.from_numpy(cnt).to(DEV), F, ew.w1, sg, su, ew.w2, sd, ws=ws,
                                      row_gate=torch.from_numpy(gate).to(DEV)))
    _check(out_g, O.expert_down_fp8(to_np(ws["hq"]), to_np(ws["hsc"]), cnt, dq, ds, row_gate=gate).astype(np.float64), BF16_RTOL,
           BF16_ATOL, f"fp8 down GEMM with row gates E_l={E_l} H={H} F={F}")
    want = O.expert_mlp_fp8(x, cnt, gq, gs, uq, us, dq, ds)
    _check(out, want.astype(np.float64), FP8_RTOL, FP8_ATOL, f"expert_mlp_fp8 end to end E_l={E_l} H={H} F={F}")
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    tight = np.abs(out - want) <= BF16_RTOL * np.abs(want) + BF16_ATOL * rms
    print(f"fraction of outputs within the bf16 bound end to end: {tight.mean():.6f}", flush=True)
    assert tight.mean() > 0.99
    # against the unquantised fp32 MLP, to show what the quantisation itself costs (reported only)
    ref = O.expert_mlp(x, cnt, wg, wd, "swiglu", "f32", w_up=wu)
    print("fp8 vs unquantised fp32 MLP (max-abs, max-abs / rms, max-rel):", err_stats(out, ref.astype(np.float64)), flush=True)


@pytest.mark.parametrize("E_l,H,F,rows", [(2, 2048, 1408, (300, 220)), (1, 512, 1024, (450,)), (3, 1024, 2048, (130, 0, 260)),
                                           (1, 4096, 512, (90,)), (2, 512, 4096, (130, 60)), (1, 4096, 4096, (40,))])
def test_expert_mlp_fp8_k_split_of_the_last_round(E_l, H, F, rows):
    """The fp8 GEMMs with the partial-sum workspace: few tiles with long rows (4096 and more) are cut along K, and the last part of a tile
    adds the sums and applies the same scales, epilogue and block quantisation.  Each GEMM is held to the oracle on
    its own inputs (as in test_expert_mlp_fp8), the result is reproducible from call to call whatever the workspace held,
    and the hidden activation is that of the unsplit kernels but for values on a rounding boundary."""
    rng = np.random.default_rng(H + F + E_l)
    cnt = np.array(rows, dtype=np.int32)
    assert [gemm_parts(cnt, *a, fp8=True)[2] > 1 for a in ((H, F, "swiglu"), (F, H, "none"))] == [H >= 4096, F >= 4096]
    S_tot = int(cnt.sum())
    x = _randn(rng, S_tot, H)
    wg, wu = _randn(rng, E_l, H, F, scale=H ** -0.5), _randn(rng, E_l, H, F, scale=H ** -0.5)
    wd = _randn(rng, E_l, F, H, scale=F ** -0.5)
    (gq, gs), (uq, us), (dq, ds) = (O.quantize_cols_fp8(w) for w in (wg, wu, wd))
    tq = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    ew = ExpertWeights.prepare_fp8(tq(gq), tq(gs), tq(uq), tq(us), tq(dq), tq(ds))
    sg, su, sd = ew.scales
    cnt_t, x_t = torch.from_numpy(cnt).to(DEV), _t(x, "bf16")
    plain_ws = ops.fp8_workspace(S_tot, H, F, DEV)
    plain = ops.grouped_mlp_fp8(x_t, cnt_t, F, ew.w1, sg, su, ew.w2, sd, ws=plain_ws)
    part = ops.gemm_part_workspace(DEV)
    outs = []
    for fill in (float("nan"), 3.0):
        part.fill_(fill)
        ws = ops.fp8_workspace(S_tot, H, F, DEV)
        outs.append((ops.grouped_mlp_fp8(x_t, cnt_t, F, ew.w1, sg, su, ew.w2, sd, ws=ws, part_ws=part).clone(), ws))
    torch.cuda.synchronize()
    (split, ws1), (again, _) = outs
    assert torch.equal(split.view(torch.int16), again.view(torch.int16)), "the fp8 K split is not reproducible"
    assert bool(torch.isfinite(split.float()).all())
    hq_gpu, hsc_gpu = to_np(ws1["hq"]), to_np(ws1["hsc"])
    hq_want, hsc_want = O.expert_up_fp8(x, cnt, gq, gs, uq, us)
    _hidden_codes_close(hq_gpu, hsc_gpu, hq_want, hsc_want, "fp8 gate/up, K split")
    _check(to_np(split), O.expert_down_fp8(hq_gpu, hsc_gpu, cnt, dq, ds).astype(np.float64), BF16_RTOL, BF16_ATOL, "fp8 down, K split")
    # against the unsplit kernels: the same codes but for fp32 sums in another order
    _hidden_codes_close(hq_gpu, hsc_gpu, to_np(plain_ws["hq"]), to_np(plain_ws["hsc"]), "fp8 gate/up, K split against unsplit")
    assert bool(torch.isfinite(plain.float()).all())
