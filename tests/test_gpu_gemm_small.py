"""The small-tile grouped GEMM (csrc/gemm_small.hip) at the edges of its tiles, stages and parts, against fp32 products of the
same operands.  The sizes are ones the dispatch gives to it: few rows, or few columns, or both."""
import numpy as np
import pytest
import torch

from helpers import O
from iris_testing_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _close(got, ref, what):
    err = (got.float() - ref).abs()
    bar = 2.0 ** -7 * ref.abs() + 2.0 ** -8 * ref.abs().amax()
    assert bool(torch.isfinite(got.float()).all()) and bool((err <= bar).all()), f"{what}: {float((err - bar).max())} over the bar"


# (rows per group, K, N, activation): one row; a tile's edge on either side; one pair of stages and an odd number of pairs;
# a partly filled group of 32 columns, a partly filled tile; K ranges long enough to be cut into parts; more groups than lanes
CASES = [((1,), 64, 8, "none"), ((31, 32, 33), 192, 136, "none"), ((63, 0, 64, 65), 320, 96, "swiglu"), ((5, 130), 64, 264, "gelu"),
         ((17,), 8192, 256, "none"), ((40, 3), 4096, 512, "swiglu"), ((64,), 7168, 1032, "silu"), (tuple([1, 0, 2] * 30), 128, 128, "none"),
         # launches of large tiles (128 and 256 rows) whose last round of tiles is handed to small ones
         ((4701,), 2048, 4096, "none"), ((8900, 0, 1000), 3072, 2528, "swiglu")]


@pytest.mark.parametrize("cnt,K,N,act", CASES, ids=[f"{len(c[0])}g_{sum(c[0])}x{c[1]}x{c[2]}_{c[3]}" for c in CASES])
@pytest.mark.parametrize("workspace", [False, True], ids=["whole", "parts"])
def test_small_gemm_edges(cnt, K, N, act, workspace):
    rng = np.random.default_rng(K + N)
    E_l, S = len(cnt), sum(cnt)
    base = torch.from_numpy(rng.standard_normal((S + 9, K)).astype(np.float32)).to(DEV).bfloat16()
    w, wu = (torch.from_numpy((rng.standard_normal((E_l, K, N)) * K ** -0.5).astype(np.float32)).to(DEV).bfloat16() for _ in range(2))
    packed = ops.prepack_weights(w, wu if act == "swiglu" else None)
    a_map, c_map = (torch.from_numpy(rng.permutation(S + 9)[:S].astype(np.int32)).to(DEV) for _ in range(2))
    if S > 4:
        c_map[3] = -1  # a row without a place in the output
    cnt_t = torch.tensor(cnt, dtype=torch.int32, device=DEV)
    ws = ops.gemm_part_workspace(DEV) if workspace else None
    if workspace:
        ws.fill_(float("nan"))
    out = torch.full((S + 9, N), -7.0, dtype=torch.bfloat16, device=DEV)
    run = lambda: ops.grouped_gemm_mapped(base, a_map, packed, cnt_t, S, N, act, out, c_map, part_ws=ws)  # noqa: E731
    run()
    x, ref, r0 = base[a_map.long()].float().cpu(), torch.empty(S, N), 0
    for e, c in enumerate(cnt):
        g = x[r0:r0 + c] @ w[e].float().cpu()
        if act == "swiglu":
            g = torch.nn.functional.silu(g) * (x[r0:r0 + c] @ wu[e].float().cpu())
        elif act != "none":
            g = getattr(torch.nn.functional, act)(g)
        ref[r0:r0 + c] = g
        r0 += c
    kept = (c_map >= 0).cpu()
    first = out.clone()
    _close(first.cpu()[c_map.cpu().long()[kept]], ref[kept], f"{cnt} {K} {N} {act}")
    rest = torch.ones(S + 9, dtype=torch.bool)
    rest[c_map.cpu().long()[kept]] = False
    assert bool((first.cpu()[rest] == -7.0).all()), "a row outside the map was written"
    # the same bits again: called again, and replayed from a graph (the counters of the parts are left as a launch finds them)
    for _ in range(2):
        run()
        assert torch.equal(out.view(torch.int16), first.view(torch.int16))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    for _ in range(3):
        out.fill_(-7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), first.view(torch.int16))


# two sets of waves to a tile (every tile a compute unit to itself, 54 stages of K or more): odd and even numbers of pairs of stages, whole and in parts
@pytest.mark.parametrize("cnt,K,N,act", [((33, 31), 1728, 200, "silu"), ((64, 0, 17), 1856, 96, "swiglu"), ((70,), 1792, 1032, "none"), ((100, 28), 4160, 136, "gelu")])
@pytest.mark.parametrize("workspace", [False, True], ids=["whole", "parts"])
def test_small_gemm_two_sets_of_waves(cnt, K, N, act, workspace):
    test_small_gemm_edges(cnt, K, N, act, workspace)


@pytest.mark.parametrize("cnt,H,F", [((40,), 3456, 3584), ((65, 9), 4224, 128)])
@pytest.mark.parametrize("workspace", [False, True], ids=["whole", "parts"])
def test_small_fp8_mlp_two_sets_of_waves(cnt, H, F, workspace):
    test_small_fp8_mlp_edges(cnt, H, F, workspace)


@pytest.mark.parametrize("cnt,H,F", [((1,), 128, 128), ((33, 0, 64), 384, 256), ((65,), 4096, 640), ((20, 7), 2048, 2176),
                                     ((6000,), 2048, 1408)])  # (the last: large tiles with 8 left over)
@pytest.mark.parametrize("workspace", [False, True], ids=["whole", "parts"])
def test_small_fp8_mlp_edges(cnt, H, F, workspace):
    rng = np.random.default_rng(H + F)
    E_l, S = len(cnt), sum(cnt)
    x = torch.from_numpy((rng.standard_normal((S, H)) * rng.uniform(0.3, 3.0, (S, 1))).astype(np.float32)).to(DEV).bfloat16()
    (gq, gs), (uq, us), (dq, ds) = [tuple(torch.from_numpy(t).to(DEV) for t in O.quantize_cols_fp8((rng.standard_normal(sh) * sc).astype(np.float32)))
                                    for sh, sc in (((E_l, H, F), H ** -0.5), ((E_l, H, F), H ** -0.5), ((E_l, F, H), F ** -0.5))]
    ws = ops.fp8_workspace(S, H, F, DEV)
    part = ops.gemm_part_workspace(DEV) if workspace else None
    y = ops.grouped_mlp_fp8(x, torch.tensor(cnt, dtype=torch.int32, device=DEV), F, ops.prepack_weights_fp8(gq, uq), gs, us,
                            ops.prepack_weights_fp8(dq), ds, ws=ws, part_ws=part)
    dec = lambda t: t.view(torch.float8_e4m3fn).float().cpu()  # noqa: E731
    xd, hd, r0 = dec(ws["xq"]), ops.dequantize_hidden_fp8(ws["hq"], ws["hsc"]).cpu(), 0
    for e, c in enumerate(cnt):
        if c:
            sx = ws["xs"][r0:r0 + c, None].cpu()
            h = torch.nn.functional.silu((xd[r0:r0 + c] @ dec(gq[e])) * sx * gs[e].cpu()) * ((xd[r0:r0 + c] @ dec(uq[e])) * sx * us[e].cpu())
            # a code is at most half a step of its block's grid away (one step where a sum sits on a boundary)
            blk = h.view(c, -1, 32).abs().amax(-1, keepdim=True)
            err = (hd[r0:r0 + c] - h).abs().view(c, -1, 32)
            assert bool((err <= h.abs().view(c, -1, 32) * 2.0 ** -3.9 + blk * 2.0 ** -14 + 1e-6).all()), f"hidden of group {e}"
            _close(y[r0:r0 + c].cpu(), (hd[r0:r0 + c] @ dec(dq[e])) * ds[e].cpu(), f"down, group {e}")
        r0 += c


BIG = 2 ** 31 - 1


@pytest.mark.parametrize("S,E_l,K,N", [(40, 3, 64, 128), (64, 130, 4096, 256), (443, 3, 2048, 512), (9900, 3, 3072, 2528)])
@pytest.mark.parametrize("at", [0, 1])
def test_counts_that_claim_far_too_much(S, E_l, K, N, at):
    """Counts whose sum passes 2^31 are cut at the rows there are, one after the other, in every grouped GEMM: small tiles with and without
    parts, large ones with a last round of small ones, fp32, and the weight gradients."""
    g = torch.Generator(device=DEV).manual_seed(S)
    claimed = torch.zeros(E_l, dtype=torch.int32)
    claimed[0], claimed[at], claimed[at + 1], claimed[-1] = 7, BIG, BIG, BIG
    cut, left = torch.zeros_like(claimed), S
    for e in range(E_l):
        cut[e] = min(int(claimed[e]), left)
        left -= int(cut[e])
    claimed, cut = claimed.to(DEV), cut.to(DEV)
    x = (torch.randn(S, K, generator=g, device=DEV) / 8).bfloat16()
    w = (torch.randn(E_l, K, N, generator=g, device=DEV) / 8).bfloat16()
    packed = ops.prepack_weights(w)
    for ws in (None, ops.gemm_part_workspace(DEV)):
        got, want = (torch.full((S, N), -7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        ops.grouped_gemm_mapped(x, None, packed, claimed, S, N, "none", got, part_ws=ws)
        ops.grouped_gemm_mapped(x, None, packed, cut, S, N, "none", want, part_ws=ws)
        assert torch.equal(got, want) and not bool((got == -7.0).all(1).any())
    dy = (torch.randn(S, N, generator=g, device=DEV) / 8).bfloat16()
    assert torch.equal(ops.grouped_gemm_dw(x, dy, claimed), ops.grouped_gemm_dw(x, dy, cut))
    if S < 1000:
        xf, wf, dyf = x.float(), w.float(), dy.float()
        assert torch.equal(ops.grouped_gemm(xf, wf, claimed), ops.grouped_gemm(xf, wf, cut))
        assert torch.equal(ops.grouped_gemm_dw(xf, dyf, claimed), ops.grouped_gemm_dw(xf, dyf, cut))
    if K % 128 == 0 and S < 1000:
        F = 256
        q = lambda *s: torch.randint(0, 120, s, generator=g, device=DEV, dtype=torch.uint8)  # noqa: E731  (finite e4m3 codes)
        one = lambda n: torch.full((E_l, n), 2.0 ** -12, device=DEV)  # noqa: E731
        up, down = ops.prepack_weights_fp8(q(E_l, K, F), q(E_l, K, F)), ops.prepack_weights_fp8(q(E_l, F, K))
        for ws in (None, ops.gemm_part_workspace(DEV)):
            got, want = (ops.grouped_mlp_fp8(x, c, F, up, one(F), one(F), down, one(K), part_ws=ws) for c in (claimed, cut))
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)) and bool(got.float().abs().amax(1).gt(0).all())


def test_counts_that_claim_far_too_much_of_very_many_rows():
    """Beyond 2^25 rows even cut counts would wrap a sum of 64 of them: the same rule, one count at a time."""
    S = (1 << 25) + 77
    g = torch.Generator(device=DEV).manual_seed(1)
    x, w = torch.randn(S, 4, generator=g, device=DEV), torch.randn(66, 4, 4, generator=g, device=DEV)
    claimed = torch.full((66,), BIG, dtype=torch.int32, device=DEV)
    claimed[0], claimed[64] = 1 << 25, 5
    claimed[1:60] = 1
    got = ops.grouped_gemm(x, w, claimed)
    at = 1 << 25
    assert torch.allclose(got[:at], x[:at] @ w[0], rtol=1e-5, atol=1e-5)  # (four products each)
    for e in range(1, 60):
        assert torch.allclose(got[at + e - 1], x[at + e - 1] @ w[e], rtol=1e-5, atol=1e-5)
    assert torch.allclose(got[at + 59:], x[at + 59:] @ w[60], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("cnt,K,N", [((33, 0, 31), 128, 36), ((1, 64), 129, 32), ((32, 5), 240, 33), ((40,), 256, 7), ((17, 65), 257, 100),
                                     ((256, 256), 512, 256), ((3,), 1000, 64)])
@pytest.mark.parametrize("act", ["none", "swiglu"])
def test_f32_sums_by_one_and_two_sets_of_waves(cnt, K, N, act):
    """Few tiles and more than one slab's K: a tile's sums are made in two halves.  Against float64, with the bound of any order of
    K fp32 products and additions, (K + 1) 2^-24 of the sum of their magnitudes; a gated product adds its activation's rounding."""
    g = torch.Generator(device=DEV).manual_seed(K + N)
    S, E_l = sum(cnt), len(cnt)
    x = torch.randn(S, K, generator=g, device=DEV)
    w, wu = (torch.randn(E_l, K, N, generator=g, device=DEV) * K ** -0.5 for _ in range(2))
    c = torch.tensor(cnt, dtype=torch.int32, device=DEV)
    eye = torch.eye(N, K, device=DEV).expand(E_l, N, K).contiguous()
    got = ops.grouped_gemm(x, w, c) if act == "none" else ops.grouped_mlp(x, c, "swiglu", w, eye, wu)[:, :N]
    r0 = 0
    for e, n in enumerate(cnt):
        xd, a, b = x[r0:r0 + n].double(), w[e].double(), wu[e].double()
        s, mag = xd @ a, xd.abs() @ a.abs()
        bar = (K + 1) * 2.0 ** -24 * mag
        if act == "swiglu":
            u = xd @ b
            # |silu'| < 1.1; exp, division and product: 8 roundings; the product with the identity adds none
            bar = 1.1 * bar * u.abs() + torch.nn.functional.silu(s).abs() * (K + 1) * 2.0 ** -24 * (xd.abs() @ b.abs()) + 2.0 ** -21 * (s * u).abs()
            s = torch.nn.functional.silu(s) * u
        assert bool(((got[r0:r0 + n].double() - s).abs() <= bar + 1e-30).all()), (e, float(((got[r0:r0 + n].double() - s).abs() / (bar + 1e-30)).max()))
        r0 += n
