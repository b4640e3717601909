"""CPU-side checks of the product: the C-ABI library loads and exports every symbol the header
declares, the host layer rejects CPU tensors the way the reference does, and nothing in the
package reaches for the oracle."""
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    text = open(os.path.join(ROOT, "include", "moe_gfx950.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(moe_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from iris_testing_amd import _lib as L
    lib = L.lib()
    declared = _declared()
    assert len(declared) >= 20
    for name in declared:
        assert hasattr(lib, name), f"{name} declared in include/moe_gfx950.h but not exported"
    assert sorted(L.exported_symbols()) == declared, "ctypes table and header disagree"
    assert lib.moe_abi_version() == 3
    assert lib.moe_last_error() == b""


def test_argument_errors_are_reported_without_a_gpu():
    # calls that fail validation before any HIP call
    from iris_testing_amd import _lib as L
    lib = L.lib()
    rc = lib.moe_count_and_offsets(None, 4, 2, 9, 4, None, None, None, None, None, None, None, None, 0, None)
    assert rc == -1 and b"divisible" in lib.moe_last_error()
    rc = lib.moe_route_topk(None, None, None, 0, 4, 64, 8, 9, None, None, None, None, 0, None)
    assert rc == -1 and b"topk" in lib.moe_last_error()
    rc = lib.moe_route_topk(None, None, None, 1, 4, 60, 8, 2, None, None, None, None, 0, None)
    assert rc == -1 and b"16-byte" in lib.moe_last_error()
    with pytest.raises(L.MoeLibraryError):
        L.check(lib.moe_pack(None, 7, 1, 64, None, None, None, 4, 4, None, None, None, None))
    assert lib.moe_count_workspace_bytes(1000, 2, 8) == 4 * (2 * 8 * 16 + 2 * 8 + 1)


def test_argument_errors_of_the_fused_variants_and_diagnostics_without_a_gpu():
    """The gated / flat-payload / fp8 entry points and the diagnostics validate before they touch the GPU."""
    from iris_testing_amd import _lib as L
    lib = L.lib()
    # gates and their output buffer go together
    rc = lib.moe_pack_tokens_gated(None, 1, 4, 64, None, None, 1, 2, 2, None, None, 2, 4, None, None, None, None)
    assert rc == -1 and b"go together" in lib.moe_last_error()
    rc = lib.moe_recv_row_map_gated(None, 2, 2, 4, 8, 1, None, None, None, None)
    assert rc == -1
    rc = lib.moe_recv_row_map_flat(None, 0, 2, 8, None, None, None)
    assert rc == -1
    # the gated down projection needs its gates; bf16 GEMMs need K % 64 == 0
    rc = lib.moe_grouped_gemm_mapped_gated(1, 8, None, 1, 1, 8, 64, 64, 1, None, 1, 8, None, None, 0, None)
    assert rc == -1 and b"null pointer" in lib.moe_last_error()
    rc = lib.moe_grouped_gemm_mapped_gated(1, 8, None, 1, 1, 8, 48, 64, 1, 1, 1, 8, None, None, 0, None)
    assert rc == -2 and b"K %" in lib.moe_last_error()
    # fp8 expert: H and F in multiples of 128
    rc = lib.moe_grouped_mlp_fp8_q_mapped(1, 1, 8, None, 1, 8, 256, 96, 1, 1, 1, 1, 1, 1, 1, 1, 1, None, 1, 8, None, None, 0, None)
    assert rc == -2 and b"multiples of 128" in lib.moe_last_error()
    rc = lib.moe_grouped_mlp_fp8_mapped(1, 8, None, 1, 8, 200, 128, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, None, 1, 8, None, None, 0, None)
    assert rc == -2 and b"multiples of 128" in lib.moe_last_error()
    # time stamps need a buffer of the advertised size; switching them off needs none
    assert lib.moe_diag_gemm_trace_words() >= 128 + 4096
    rc = lib.moe_diag_gemm_trace(1, 16, 0)
    assert rc == -3 and b"words" in lib.moe_last_error()
    assert lib.moe_diag_gemm_trace(None, 0, 0) == 0
    assert lib.moe_diag_mfma_loop_flops(0, 1, 1) == 2.0 * 4 * 128 * 128 * 32


def test_operands_that_wide_loads_cannot_start_at_are_refused_without_a_gpu():
    """Weights in the reference layout (and payloads) go through 16-byte loads: an entry point that has no other way refuses them before
    it launches anything; moe_grouped_gemm re-tiles them if it is given room for that."""
    import ctypes
    from iris_testing_amd import _lib as L
    lib = L.lib()
    for layout in (L.W_TILED, L.W_RAW, L.W_RAW_T):
        assert lib.moe_expert_forward(16, 18, layout, 16, 4, 64, 64, 1, 16, None, 0, None) == -1 and b"16-byte aligned" in lib.moe_last_error()
    for w1, w_up, w2 in ((18, 16, 16), (16, 8, 16), (16, 16, 2)):
        rc = lib.moe_mlp_train_forward(16, 16, 4, 64, 64, 1, L.ACT["swiglu"], L.W_RAW, w1, w_up, w2, 16, 16, 16, None, 0, None)
        assert rc == -1 and b"16-byte aligned" in lib.moe_last_error()
        rc = lib.moe_mlp_train_backward(16, 16, 16, 16, 16, 4, 64, 64, 1, L.ACT["swiglu"], L.W_RAW_T, w1, w_up, w2, 16, 16, 16, 16, 16, 16, None, 0, None)
        assert rc == -1 and b"16-byte aligned" in lib.moe_last_error()
    assert lib.moe_grouped_gemm(16, 18, 16, L.MOE_BF16, 4, 64, 64, 1, 16, None, 0, None) == -3 and b"workspace" in lib.moe_last_error()
    block = (L.A2aSource * 2)()
    block[1].payload, block[1].counts, block[1].start, block[1].rows = 24, 16, 16, 3
    assert lib.moe_a2a_place(block, L.MOE_BF16, 2, 1, 4, 8, 16, 16, None, 0, None, 0, None) == -1 and b"16 bytes" in lib.moe_last_error()
    assert ctypes.sizeof(L.A2aSource) == 32


def test_static_scratch_count_rejects_oversized_inputs_without_a_gpu():
    """The allocation-free counting entry point checks its size limit before it touches the GPU."""
    from iris_testing_amd import _lib as L
    lib = L.lib()
    cap = lib.moe_count_static_scratch_bytes()
    assert cap == 4 << 20
    assert lib.moe_count_workspace_bytes(1 << 17, 2, 512) > cap
    rc = lib.moe_count_and_offsets_static(None, 1 << 17, 2, 512, 8, None, None, None, None, None, None, None, None)
    assert rc == -3 and b"scratch" in lib.moe_last_error()
    assert lib.moe_count_and_offsets_static(None, 64, 0, 8, 4, None, None, None, None, None, None, None, None) == -1


def test_host_layer_rejects_cpu_tensors_like_the_reference():
    from iris_testing_amd import utils
    from iris_testing_amd.baseline import reorder_flat_to_token_buf
    with pytest.raises(AssertionError, match="Expect CUDA tokens"):  # reference utils.py:193
        utils.route_and_pack_padding_free(torch.zeros(4, 8), torch.zeros(8, 4), 1, 2, 4)
    with pytest.raises(AssertionError, match="must be CUDA"):  # reference utils.py:16
        utils.build_expert_offsets(torch.zeros((2, 2), dtype=torch.int32))
    with pytest.raises(ValueError, match="CUDA"):  # reference baseline.py:10-12
        reorder_flat_to_token_buf(torch.zeros(2, 4), torch.zeros((1, 1), dtype=torch.int32), 2, torch.zeros(1, 1, 2, 4))


def test_product_never_imports_the_oracle():
    pkg = os.path.join(ROOT, "iris_testing_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h")):
                text = open(os.path.join(dirpath, f)).read()
                assert "oracle" not in text.lower() or f == "harness.py" and "moe_oracle" not in text, \
                    f"{f} mentions the oracle"


def test_configs_and_generators_are_deterministic():
    from iris_testing_amd.configs import CONFIGS, gen_router, gen_router_bias, gen_shard_tokens
    cfg = CONFIGS["plumbing"]
    a, b = gen_shard_tokens(cfg, 1), gen_shard_tokens(cfg, 1)
    assert torch.equal(a, b) and not torch.equal(a, gen_shard_tokens(cfg, 2))
    assert gen_router(cfg).shape == (256, 8)
    z = gen_router_bias(CONFIGS["zipf_k2"])
    assert z.shape == (60,) and torch.all(z[:-1] > z[1:])  # expert 0 hottest
    assert abs(float(torch.exp(z).sum()) - 1) < 1e-5
    for name, c in CONFIGS.items():
        assert c.experts % c.world == 0 and c.topk <= c.experts, name


def test_gemm_split_plan_covers_every_tile_and_every_k_stage_once():
    """The plan of moe_gemm_split_plan (whole tiles, then the tiles of an under-filled last round cut along K; kept for its
    callers, the launches follow moe_gemm_launch_plan): every tile appears, the parts of a split tile tile its K range
    exactly, every part has an even, non-zero number of stages, and the part tiles fit the workspace."""
    import ctypes
    import random
    from iris_testing_amd import _lib as L
    lib = L.lib()
    out = (ctypes.c_int32 * 4)()
    rnd = random.Random(3)
    split_seen = 0
    for _ in range(3000):
        grid = rnd.choice([256, 256, 304, 64, 8])
        total = rnd.randint(0, 4 * grid + 5)
        nk = 2 * rnd.randint(1, 400)
        max_units = rnd.choice([grid, grid // 2, 3, 1, 0])
        assert lib.moe_gemm_split_plan(total, grid, nk, max_units, out) == 0
        full, P, nkp, units = out[0], out[1], out[2], out[3]
        tail = total - full
        assert 0 <= full <= total and P >= 1 and units == full + tail * P
        if P == 1:
            assert full == total
            continue
        split_seen += 1
        assert tail == total % grid and 4 * tail <= grid and tail * P <= min(grid, max_units) and P <= 16
        assert nkp % 2 == 0 and nkp >= 8
        stages = [min(nkp, nk - part * nkp) for part in range(P)]
        assert sum(stages) == nk and all(s >= 2 and s % 2 == 0 for s in stages)
    assert split_seen > 100
    # the shapes of the bench workloads: Mixtral-style down GEMM (2064 tiles, 448 stages) and the small config's GEMMs
    for total, nk, want in [(2064, 448, (2048, 16, 28)), (14448, 128, (14448, 1, 128)), (64, 64, (0, 4, 16)), (32, 128, (0, 8, 16))]:
        lib.moe_gemm_split_plan(total, 256, nk, 256, out)
        assert (out[0], out[1], out[2]) == want
    assert lib.moe_gemm_split_plan(10, 0, 8, 4, out) != 0 and lib.moe_gemm_split_plan(10, 8, 7, 4, out) != 0


def _launch_plan(S, E_l, K, N, act="none", fp8=False, cus=256, ws=None, tiles=0):
    import ctypes
    from iris_testing_amd import _lib as L
    out = (ctypes.c_int32 * 4)()
    ws = L.lib().moe_gemm_part_workspace_bytes() if ws is None else ws
    assert L.lib().moe_gemm_launch_plan(S, E_l, K, N, L.ACT[act], fp8, cus, ws, tiles, out) == 0
    return tuple(out)


def test_launch_plan_covers_every_tile_and_every_k_stage_once():
    """What the launches and kernels decide by (the same functions): a large tile is taken whole or left, with the rest of a part-filled last
    round, to small ones; the parts of a small tile tile its K range exactly, in pairs of stages, 32 or more of them but for the last,
    and fit the workspace and the chip."""
    import random
    from iris_testing_amd import _lib as L
    rnd, ctr = random.Random(5), 16384
    seen = {"tail": 0, "whole": 0, "parts": 0, "cut_short": 0}
    for _ in range(4000):
        fp8, cus, act = rnd.random() < 0.4, rnd.choice([256, 256, 304, 64]), rnd.choice(["none", "swiglu"])
        S, E_l = int(2 ** rnd.uniform(0, 16)), rnd.choice([1, 2, 8, 32])
        K, N = 128 * int(2 ** rnd.uniform(0, 7)), 64 * int(2 ** rnd.uniform(0, 8))
        room = rnd.choice([0, 1, 2, 7, 64, 256])
        ws = ctr + room * 64 * 128 * 4 if room else 0
        nk = K * (1 if fp8 else 2) // 64
        bm = _launch_plan(S, E_l, K, N, act, fp8, cus, ws)[0]
        cols = 2 * N if act == "swiglu" else N
        tiles = rnd.randint(1, max(1, (-(-S // bm) + E_l) * -(-cols // (256 if bm >= 128 else 128))))
        again, whole, P, nkp = _launch_plan(S, E_l, K, N, act, fp8, cus, ws, tiles)
        assert again == bm and bm in (32, 64, 128, 256) and 1 <= P <= 16
        if bm >= 128:
            assert whole in (tiles, tiles - tiles % cus)
            seen["tail" if whole < tiles else "whole"] += 1
        else:
            assert whole == 0
        small = (tiles - whole) * (2 * (bm // 64) if bm >= 128 else 1)
        if P == 1:
            assert nkp == nk
            continue
        seen["parts"] += 1
        assert ws and nkp % 2 == 0 and nkp >= 32
        stages = [min(nkp, nk - i * nkp) for i in range(P)]
        assert sum(stages) == nk and all(s >= 2 and s % 2 == 0 for s in stages)
        seen["cut_short"] += stages[-1] < nkp
        assert small * P <= min(cus, room * (2 if bm == 32 else 1))
    assert min(seen.values()) > 30, seen
    # one group: the host knows what is left over, and keeps the second launch for rounds it is quicker in
    assert _launch_plan(8192, 1, 4096, 14336, "swiglu", tiles=32 * 112)[:2] == (256, 32 * 112)
    assert _launch_plan(8192 + 256, 1, 4096, 14336, "swiglu", tiles=33 * 112)[1] in (33 * 112, 14 * 256)
    out = (__import__("ctypes").c_int32 * 4)()
    assert L.lib().moe_gemm_launch_plan(0, 1, 64, 64, 0, 0, 256, 0, 1, out) == -1 and L.lib().moe_gemm_launch_plan(1, 1, 64, 64, 9, 0, 256, 0, 1, out) == -1


def test_tile_rule_counts_on_parts_only_where_there_is_room_for_them():
    """The height of a launch's tiles is chosen with the K split in mind; without a workspace nothing is split, and the choice must be
    the one of a launch that cannot be split (which short rows are anyway, workspace or not)."""
    from iris_testing_amd import _lib as L
    ctr, unit = 16384, 64 * 128 * 4
    full = L.lib().moe_gemm_part_workspace_bytes()
    differ = split = 0
    for S in (1, 24, 64, 300, 443, 1003, 4096, 20000):
        for E_l in (1, 2, 8, 32):
            for N, act in ((256, "none"), (2048, "swiglu"), (7168, "none")):
                for K in (512, 1024, 1920, 1984, 2048, 4096, 14336):
                    for fp8 in (False, True):
                        none = _launch_plan(S, E_l, K, N, act, fp8, ws=0, tiles=3)
                        some = _launch_plan(S, E_l, K, N, act, fp8, tiles=3)
                        assert none[2] == 1 and none == _launch_plan(S, E_l, K, N, act, fp8, ws=ctr, tiles=3)
                        if K * (1 if fp8 else 2) < L.MOE_SPLIT_MIN_K_BYTES:
                            assert some == none
                        differ, split = differ + (some[0] != none[0]), split + (some[2] > 1)
                        # room for one part tile is room for none
                        assert _launch_plan(S, E_l, K, N, act, fp8, ws=ctr + unit // 2, tiles=3)[0] == none[0]
    assert full == ctr + (8 << 20) and differ > 20 and split > 100


def test_fp32_launch_moves_rows_or_refuses():
    """A launch of the fp32 GEMM that cannot move rows (large tiles; an activation on the way to the slots) says so and is not launched
    without them; one that can covers every tile of any distribution of the rows."""
    import ctypes
    import random
    from iris_testing_amd import _lib as L
    rnd, out, seen = random.Random(7), (ctypes.c_int32 * 4)(), {"big": 0, "split": 0, "one": 0}
    for _ in range(3000):
        S, E_l, K, N = int(2 ** rnd.uniform(0, 15)), rnd.choice([1, 2, 15, 64, 130]), int(2 ** rnd.uniform(0, 12)), int(2 ** rnd.uniform(0, 12))
        act, cus = rnd.choice(["none", "gelu", "silu", "swiglu"]), rnd.choice([256, 256, 304, 64])
        args = (S, E_l, K, N, L.ACT[act])
        assert L.lib().moe_gemm_f32_plan(*args, 0, cus, out) == 0
        tile, sets, cols, rows = plan = tuple(out)
        assert tile in (32, 64) and sets in (1, 2) and cols * tile >= N and (sets == 1 or tile == 32 and K > 128)
        seen["big" if tile == 64 else "split" if sets == 2 else "one"] += 1
        cnt = [0] * E_l
        for _ in range(20):
            cnt[rnd.randrange(E_l)] += S // 20
        cnt[rnd.randrange(E_l)] += S - sum(cnt)
        assert sum(-(-c // tile) for c in cnt) <= rows
        for side in (1, 2):
            refused = tile == 64 or (side == 1 and act != "none")
            assert L.lib().moe_gemm_f32_plan(*args, side, cus, out) == (-2 if refused else 0)
            assert refused or tuple(out) == plan
    assert min(seen.values()) > 100, seen
    assert L.lib().moe_gemm_f32_plan(0, 1, 4, 4, 0, 0, 256, out) == -1 and L.lib().moe_gemm_f32_plan(1, 1, 4, 4, 0, 3, 256, out) == -1


def test_fp32_tiles_get_two_sets_of_waves_while_they_are_one_round():
    """A compute unit holds one workgroup of two sets: with rows spread over the groups at random, they are taken where the tiles
    are about as many as the compute units or fewer, and only there."""
    import ctypes
    import random
    from iris_testing_amd import _lib as L
    rnd, out, seen = random.Random(11), (ctypes.c_int32 * 4)(), [0, 0]
    for _ in range(2000):
        S, E_l, K, N, cus = int(2 ** rnd.uniform(0, 12)), rnd.choice([1, 2, 15, 32, 64]), rnd.choice([64, 128, 129, 400, 2000]), int(2 ** rnd.uniform(5, 11)), rnd.choice([256, 304, 64])
        L.check(L.lib().moe_gemm_f32_plan(S, E_l, K, N, L.ACT["none"], 0, cus, out))
        tile, sets, cols, _ = out
        if tile != 32:
            continue
        tiles = 0
        for _ in range(8):
            cnt = [0] * E_l
            for _ in range(S):
                cnt[rnd.randrange(E_l)] += 1
            tiles += cols * sum(-(-c // 32) for c in cnt) / 8
        slack = 1.0 if E_l == 1 else 1.2
        if sets == 2:
            assert K > 128 and tiles <= slack * cus, (S, E_l, K, N, cus, tiles)
        elif K > 128:
            assert slack * tiles > cus, (S, E_l, K, N, cus, tiles)
        seen[sets - 1] += K > 128
    assert min(seen) > 200, seen


def test_results_in_one_allocation_do_not_share_a_version_counter():
    """What a caller changes in place must not look changed elsewhere: autograd refuses to use a saved tensor whose counter moved."""
    from iris_testing_amd import ops
    parts = ops._i32_parts("cpu", (3, 5), (7,), (1, 1))
    for i, t in enumerate(parts):
        t.fill_(i)
    parts[1].clamp_(max=0)
    assert [t._version for t in parts] == [1, 2, 1] and [int(t.max()) for t in parts] == [0, 0, 2]
    assert [tuple(t.shape) for t in parts] == [(3, 5), (7,), (1, 1)] and all(t.is_contiguous() and t.data_ptr() % 16 == 0 for t in parts)


def test_bench_refuses_more_than_one_gpu():
    """This build has no collectives: bench.py --gpus 2 must say so and exit non-zero without touching a GPU."""
    import subprocess
    import sys
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 2 and "--gpus must be 1" in r.stderr and r.stdout.strip() == ""


def test_ctypes_table_has_the_argument_count_of_every_declaration():
    """Every entry of the ctypes signature table has as many arguments as the header's declaration of that symbol."""
    from iris_testing_amd import _lib as L
    text = re.sub(r"/\*.*?\*/", "", open(os.path.join(ROOT, "include", "moe_gfx950.h")).read(), flags=re.S)
    for name, (_, args) in L._SIGNATURES.items():
        m = re.search(r"\b" + name + r"\s*\(([^;]*?)\)\s*;", text, re.S)
        assert m, f"{name} is not declared"
        params = [x for x in m.group(1).split(",") if x.strip() and x.strip() != "void"]
        assert len(params) == len(args), f"{name}: header declares {len(params)} arguments, the ctypes table {len(args)}"


@pytest.mark.parametrize("kind,mode", [("f32", {}), ("bf16", {}), ("bf16", dict(gated=True)), ("bf16", dict(padding_free=True)),
                                       ("fp8", {}), ("fp8", dict(fp8_dispatch=False)), ("fp8", dict(gated=True)), ("fp8", dict(padding_free=True))])
def test_step_takes_the_buffers_of_the_moment(monkeypatch, kind, mode):
    """Every field of the step's argument block is what its name says, and a buffer that the caller has replaced, or given other
    memory, is the one the next step gets.  (CPU tensors; the library call is replaced by a look at its argument.)"""
    import types
    from iris_testing_amd import _lib as L
    from iris_testing_amd.configs import MoEConfig
    from iris_testing_amd.harness import World
    from iris_testing_amd.layers import ExpertWeights
    from iris_testing_amd.pipeline import DispatchPipeline
    T, H, E, k, W, F, M, S = 6, 128, 8, 2, 4, 256, 5, 11
    cfg = MoEConfig("case", 0, T, H, "f32" if kind == "f32" else "bf16", E, k, W, F, "swiglu" if kind == "fp8" else "silu")
    dt, e_l = cfg.torch_dtype, cfg.e_local
    world = World(cfg, torch.empty(H, E, dtype=dt), torch.empty(E), torch.empty(T, H, dtype=dt), [], M, 3, torch.empty(W, M, H, dtype=dt),
                  torch.empty(W, e_l, dtype=torch.int32), S)
    w1, w2 = torch.empty(e_l, H, F, dtype=dt), torch.empty(e_l, F, H, dtype=dt)
    if kind == "fp8":
        world.recv_q, world.recv_scale = torch.empty(W, M, H, dtype=torch.uint8), torch.empty(W, M)
        ew = ExpertWeights("swiglu", H, F, e_l, torch.uint8, w1, w2, scales=tuple(torch.empty(e_l, n) for n in (F, F, H)))
    else:
        ew = ExpertWeights("silu", H, F, e_l, dt, w1, w2)
    pipe = DispatchPipeline(world, ew, recv_gate=torch.empty(W, M) if mode.get("gated") else None,
                            recv_flat=torch.empty(S, H, dtype=dt) if mode.get("padding_free") else None, **mode)
    seen = {}
    stub = types.SimpleNamespace(moe_step=lambda a, s: seen.update({n: getattr(a, n) or 0 for n, _ in L.StepArgs._fields_}) or 0)
    monkeypatch.setattr(L, "lib", lambda: stub)
    monkeypatch.setattr(L, "stream_ptr", lambda: 0)

    def want():
        flat, q = pipe.padding_free, pipe.fp8_dispatch
        out = dict(tokens=T, hidden=H, experts=E, topk=k, world=W, ffn=F, act=L.ACT[ew.act], dtype=pipe.code, M=M, S=S, fused=pipe.fused,
                   flat=flat, gated=pipe.gated, quant=kind == "fp8", q_dispatch=q, f32_weights=kind == "f32",
                   route_ws_bytes=pipe.route_ws_bytes, count_ws_bytes=pipe.count_ws_bytes, part_ws_bytes=pipe.part_ws_bytes)
        t = dict(x=world.x0, router=world.router, bias=world.bias, recv_counts=world.recv_counts, recv_scale=world.recv_scale,
                 recv=world.recv_q if q else pipe.recv_flat if flat else world.recv, w1=ew.w1, w_up=ew.w_up, w2=ew.w2,
                 s1=ew.scales and ew.scales[0], s_up=ew.scales and ew.scales[1], s2=ew.scales and ew.scales[2],
                 send=pipe.send_q if q else pipe.payload if flat else pipe.send, ret=pipe.ret_flat if flat else pipe.ret,
                 hidden_ws=pipe.hidden, hscale=pipe.hsc)
        t.update({n: getattr(pipe, n, None) for n, _ in L.StepArgs._fields_ if n not in out and n not in t})
        out.update({n: 0 if v is None else v.data_ptr() for n, v in t.items()})
        return {n: int(v) for n, v in out.items()}

    pipe.step()
    assert seen == want()
    for n in [n for n, v in vars(pipe).items() if isinstance(v, torch.Tensor)]:
        setattr(pipe, n, torch.empty_like(getattr(pipe, n)))  # (the old one is freed)
        pipe.step()
        assert seen == want(), n
    keep = pipe.out.clone()
    pipe.out.data = keep
    pipe.step()
    assert seen["out"] == keep.data_ptr()


# What the launches of a step that may go beside one another read and write (names of moe_step_args): the receive side's preparation, and the
# source side from the counting to the packing; the two GEMMs of fp32 experts with the copies of the rows in them.
PREPARE = ("recv_counts recv_gate recv_scale", "row_map expert_cnt row_gate xs ret")
SOURCE = ("idx x gate", "send_counts expert_offs dst_sizes dst_offsets caps pos row_token count_ws send send_scale send_gate status")
F32_UP = ("recv recv_counts w1 w_up", "rows expert_cnt hidden_ws")
F32_DOWN = ("hidden_ws expert_cnt recv_counts w2", "y ret")
NOT_BESIDE = "router bias logits route_ws s1 s_up s2 xq hq hscale unpack_map ret_map part_ws returned zero_off out"  # other launches alone


@pytest.mark.parametrize("mode", ["f32", "f32 swiglu", "bf16", "gated", "flat", "fp8", "fp8 gated", "fp8 rows"])
def test_step_keeps_launches_apart_whose_buffers_meet(mode):
    """Every pair of a step's buffers laid over one another, by all and by one value: where one launch writes what another that would go
    beside it reads or writes, the step goes stage by stage; next to each other they may lie."""
    import ctypes
    from iris_testing_amd import _lib as L
    T, H, E, k, W, F, M, S = 24, 64, 12, 2, 3, 96, 17, 41
    e_l, f32 = E // W, mode.startswith("f32")
    flat, gated, q, quant = mode == "flat", "gated" in mode, mode in ("fp8", "fp8 gated"), "fp8" in mode
    act = L.ACT["swiglu" if quant or "swiglu" in mode else "silu"]
    B, slots, R = 4 if f32 else 2, W * M, T * k
    size = dict(x=T * H * B, idx=R * 4, gate=R * 4, send_counts=E * 4, expert_offs=E * 4, dst_sizes=W * 4, dst_offsets=W * 4, caps=8, pos=R * 4,
                row_token=R * 4, count_ws=4096, send=R * H * B if flat else slots * H * (1 if q else B), status=4, recv_counts=E * 4,
                recv=S * H * B if flat else slots * H * (1 if q else B), expert_cnt=e_l * 4, ret=(S if flat else slots) * H * B)
    size.update(dict(send_scale=slots * 4, recv_scale=slots * 4) if q else {}, **(dict(send_gate=slots * 4, recv_gate=slots * 4, row_gate=S * 4) if gated else {}))
    if f32:
        size.update(rows=S * H * 4, hidden_ws=S * F * 4, y=S * H * 4, w1=e_l * H * F * 4, w2=e_l * H * F * 4,
                    **({"w_up": e_l * H * F * 4} if act == L.ACT["swiglu"] else {}))
    else:
        size.update(row_map=S * 4, **({"xs": S * 4} if quant else {}))
    pointers = [n for n, t in L.StepArgs._fields_ if t is ctypes.c_void_p]
    known = " ".join((*PREPARE, *SOURCE, *F32_UP, *F32_DOWN, NOT_BESIDE)).split()
    assert set(known) == set(pointers), "a buffer of moe_step_args that this test does not know: say which launches use it"
    at = {n: (i + 1) << 32 for i, n in enumerate(pointers) if n in size or n in NOT_BESIDE.split()}
    out = (ctypes.c_int32 * 2)()

    def plan(**moved):
        a = L.StepArgs(tokens=T, hidden=H, experts=E, topk=k, world=W, ffn=F, act=act, dtype=L.MOE_F32 if f32 else L.MOE_BF16, M=M, S=S, fused=not f32,
                       flat=flat, gated=gated, quant=quant, q_dispatch=q, f32_weights=f32, count_ws_bytes=size["count_ws"], **{**at, **moved})
        L.check(L.lib().moe_step_plan(ctypes.byref(a), out))
        return out[1 if f32 else 0]

    used = lambda names: [n for n in names.split() if n in size and not (n == "xs" and not q) and not (n == "ret" and flat)]  # noqa: E731
    bad = set()
    if f32:
        for reads, writes in (map(used, F32_UP), map(used, F32_DOWN)):
            bad |= {frozenset((w, n)) for w in writes for n in reads + writes if n != w}
    else:
        (pr, pw), (sr, sw) = map(used, PREPARE), map(used, SOURCE)
        bad |= {frozenset((p, s)) for p in pw for s in sr + sw} | {frozenset((p, s)) for p in pr for s in sw}
    both_read = {frozenset((p, s)) for p in used(PREPARE[0]) for s in used(SOURCE[0])}  # (either way is right)
    assert plan() == 1 and len(bad) > 10
    for p in size:
        for q_ in size:
            if p == q_:
                continue
            pair = frozenset((p, q_))
            for over in (at[p], at[p] + size[p] - 4):
                got = plan(**{q_: over})
                assert got == 0 if pair in bad else got == 1 or pair in both_read, (p, q_)
            assert plan(**{q_: at[p] + size[p]}) == 1, (p, q_)
    for n in NOT_BESIDE.split():
        assert all(plan(**{n: at[p]}) == 1 for p in size), n


def test_step_plan_refuses_what_a_step_refuses():
    import ctypes
    from iris_testing_amd import _lib as L
    out = (ctypes.c_int32 * 2)()
    a = L.StepArgs(experts=8, world=4, fused=1)
    assert L.lib().moe_step_plan(ctypes.byref(a), out) == 0 and L.lib().moe_step_plan(ctypes.byref(a), None) == -1 and L.lib().moe_step_plan(None, out) == -1
    for wrong in (dict(world=0), dict(world=3), dict(experts=0), dict(flat=1, gated=1), dict(q_dispatch=1), dict(fused=0, flat=1)):
        b = L.StepArgs(**{**dict(experts=8, world=4, fused=1), **wrong})
        assert L.lib().moe_step_plan(ctypes.byref(b), out) == -1, wrong


def test_no_load_to_lds_takes_a_scalar_register_too_early():
    """The loads to LDS stand in inline assembly, where nobody counts the five wait states that a scalar register written by a vector
    instruction needs before a load takes it: no load of the built library comes too early, and one that did would be found."""
    from iris_testing_amd.csrc import build as B
    seen, early = B.early_loads(B.disassemble(B.LIB))
    assert seen > 3000 and not early, early[:5]

    def program(*lines):  # four bytes each, from 0x100 on
        return "0000000000000100 <f>:\n" + "".join(f"\t{x.split('//')[0]:60} // {0x100 + 4 * i:012X}: 00000000 {x.split('//')[1] if '//' in x else ''}\n"
                                                  for i, x in enumerate(lines))
    reload, load, buf = "v_readlane_b32 s5, v254, 39", "global_load_lds_dwordx4 v72, s[4:5]", "buffer_load_dwordx4 v70, s[4:7], 0 offen lds"
    for lines, bad in (((reload, "s_mov_b32 m0, s60", "s_nop 0", load), 1), ((reload, "s_add_u32 m0, s9, 0", "s_nop 3", load), 0),
                       ((reload, "s_add_u32 m0, s9, 0", "s_nop 2", load), 1), ((reload, "s_addc_u32 s5, s47, s5", load), 0),
                       ((reload, "s_cmp_lt_i32 s5, 3", load), 1), ((reload, "s_mov_b32 s4, s8", load), 1), (("v_readlane_b32 s6, v254, 39", load), 0),
                       (("v_readfirstlane_b32 s6, v3", "s_nop 1", buf), 1), (("v_add_co_u32_e64 v0, s[4:5], v1, v2", load), 1),
                       (("s_nop 7", load, "s_nop 7", reload, "s_branch 65532//<f+0x4>"), 1), (("s_nop 7", load, reload, "s_nop 4", "s_branch 65532//<f+0x4>"), 0)):
        got = B.early_loads(program(*lines))
        assert got[0] == 1 and len(got[1]) == bad, (lines, got)
