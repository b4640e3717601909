// Persistent grouped expert GEMM / MLP on gfx950 MFMA (bf16 and OCP fp8) with LDS-staged tiles,
// plus an fp32 path for the plumbing-size workload.
//
// Replaces the reference's intended expert layer (layers/expert.py:31-60) and grouped_gemm kernel
// (kernels.py:240-289): out[rows of group g] = tokens[rows of g] @ weights[g], fp32 accumulate,
// persistent grid walking a tile list that spans all groups.  Differences in kind, not a port:
//   * tiles are 256 x 256, four wave64s each owning a 128 x 128 block of 16x16x32 (bf16) MFMAs with the accumulators in the
//     accumulation registers, or eight with 64 x 128 of 32x32x64 (fp8); tiles of 128 x 256 are gemm_duo.hip's;
//   * operands go HBM -> LDS directly (global_load_lds, 16 bytes per lane) through a ring of four
//     64-byte K stages, activations two stages (a cache line of every row) at a time; the loads are spread over the MFMA
//     blocks, one to two blocks ahead; an XOR swizzle of the 16-byte chunks keeps MFMA fragment reads bank-conflict free;
//   * one MFMA block per stage: fragment reads and loads are interleaved one by one between its MFMAs;
//   * weights are re-tiled once into a K-contiguous layout (gate/up interleaved for SwiGLU) so both
//     MFMA operands are read as 128-bit fragments;
//   * ragged group tails are masked (the reference assumes full tiles, kernels.py:270,282);
//   * the tile walk is XCD-aware: the 32 workgroups that share an L2 take a compact 4 x 8 patch of
//     a 16 x 16 super-tile;
//   * the tiles of a last round of the persistent grid that fills less than about half of it go to a second launch of
//     small tiles (gemm_small.hip), which fills the chip with them.
#include "gg_common.h"
#include <algorithm>
#include <type_traits>

namespace moe_gg {

#ifndef GG_BIG_NWM
#define GG_BIG_NWM 2  // waves along M of the 256-row tile (x 2 along N)
#endif
#ifndef GG_FP8_NWM
#define GG_FP8_NWM 4  // fp8: 4 x 2 waves of 64 x 128 each, two per SIMD (measured 3.5 to 7 % faster over the fp8 workloads than 2 x 2
                      // waves of 128 x 128; the same shape costs bf16 5 %)
#endif

#ifndef GG_FP8_BSA_NWM
#define GG_FP8_BSA_NWM 4  // the fp8 down projection (block-scaled activations): waves along M, as for the other fp8 GEMM
#endif


// moe_gemm_split_plan: a last round of large tiles cut along K, tiles [0, full) whole, tiles [full, total) in P parts each.
constexpr int GG_MIN_PART_STAGES = 8;  // K stages per part at least (64 bytes of K each)
struct GgPlan {
    int total, full, P, nkp, units;
};
static GgPlan gg_plan(int total, int grid, int nk, bool split, int max_units) {
    GgPlan pl;
    pl.total = total; pl.full = total; pl.P = 1; pl.nkp = nk;
    const int tail = total % grid;
    if (split && tail > 0 && 4 * tail <= grid) {
        int P = grid / tail;
        if (P > GG_MAX_PARTS) P = GG_MAX_PARTS;
        if (P > max_units / tail) P = max_units / tail;
        while (P > 1 && (gg_part_stages(nk, P) < GG_MIN_PART_STAGES || (P - 1) * gg_part_stages(nk, P) >= nk)) --P;
        if (P > 1) { pl.P = P; pl.full = total - tail; pl.nkp = gg_part_stages(nk, P); }
    }
    pl.units = pl.full + (total - pl.full) * pl.P;
    return pl;
}

__device__ __forceinline__ int seg_of(const int* off, int n, int r) {
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (off[mid] <= r) lo = mid; else hi = mid;
    }
    return lo;
}

// One output tile of the walk: group g, n tile nt, first row row0, rv valid rows (rv <= 0: none).
struct GgTile {
    int g, nt, row0, rv;
    int ks0, nks;   // first K stage and number of K stages
};

// lin -> tile: group-major, 16-row bands, 16-column super-columns (see the XCD-aware walk above)
// DW (weight-gradient mode): every non-empty group has the same ceil(dw_rows / BM) x Nt tiles, rows [0, dw_rows) of its own
// output matrix; its K stages are its rows, 32 at a time (an even number of stages: the last ones may be partly or wholly past them).
template <int BM, bool DW = false>
__device__ __forceinline__ GgTile gg_decode(const int* g_tile_start, const int* g_row_start, int E_l, int Nt, int S_rows, int lin,
                                            int dw_rows = 0) {
    const int g = seg_of(g_tile_start, E_l + 1, lin);
    const int cnt_g = DW ? dw_rows : g_row_start[g + 1] - g_row_start[g];
    const int Mt = (cnt_g + BM - 1) / BM;
    const int idx = lin - g_tile_start[g];
    int mt, nt;
    gg_patch(idx, Mt, Nt, SUP, mt, nt);
    GgTile t;
    t.g = g;
    t.nt = nt;
    t.row0 = (DW ? 0 : g_row_start[g]) + mt * BM;
    t.rv = DW ? min(BM, cnt_g - mt * BM) : min(min(BM, cnt_g - mt * BM), S_rows - t.row0);
    return t;
}

// The tiles of a workgroup, in the order it walks them: round r of the persistent grid gives it tile r * stride + my.
// Decoding one costs a search and five integer divisions, so the workgroup decodes GG_TT of them at a time, one per
// thread, into a table in LDS; the walk itself is then one 16-byte LDS read per tile.
constexpr int GG_TT = 256;
template <int BM, bool DW>
__device__ __forceinline__ void gg_fill_table(int4* s_tiles, const int* g_tile_start, const int* g_row_start, int E_l, int Nt,
                                              int S_rows, int n, int my, int stride, int round0, int dw_rows) {
    for (int i = threadIdx.x; i < GG_TT; i += blockDim.x) {
        const int lin = (round0 + i) * stride + my;
        int4 e = make_int4(0, 0, 0, 0);  // (g, nt, row0, rv); rv <= 0: nothing there
        if ((round0 + i) < (n + stride - 1) / stride && lin < n) {
            const GgTile t = gg_decode<BM, DW>(g_tile_start, g_row_start, E_l, Nt, S_rows, lin, dw_rows);
            e = make_int4(t.g, t.nt, t.row0, t.rv);
        }
        s_tiles[i] = e;
    }
}

// The tile of round `round` if the table holds it and it has rows (rv = 0 otherwise: the caller then takes the general
// walk below).  One LDS read; nothing is advanced, refilled or skipped.
template <bool DW>
__device__ __forceinline__ GgTile gg_peek(const int4* s_tiles, const int* g_row_start, int nk, int my, int stride,
                                          int round, int round0) {
    GgTile t;
    t.g = t.nt = t.row0 = 0;
    t.rv = 0;
    t.ks0 = 0; t.nks = nk;
    if (round < round0 + GG_TT) {  // (past the end of the walk the table holds empty entries)
        const int4 e = s_tiles[round - round0];
        t.g = __builtin_amdgcn_readfirstlane(e.x); t.nt = __builtin_amdgcn_readfirstlane(e.y);
        t.row0 = __builtin_amdgcn_readfirstlane(e.z); t.rv = max(__builtin_amdgcn_readfirstlane(e.w), 0);
        if constexpr (DW) {
            t.ks0 = g_row_start[t.g];  // (the group's first row)
            t.nks = (g_row_start[t.g + 1] - t.ks0 + 63) / 64 * 2;
        }
    }
    return t;
}

// Next non-empty tile of this workgroup at or after round `round` (advanced past it); rv = 0 when there is none.
// round0 is the round the table starts at; the table is refilled (by the whole workgroup: every wave makes the same
// calls) when the walk leaves it.
template <int BM, bool DW>
__device__ __forceinline__ GgTile gg_walk(int4* s_tiles, const int* g_tile_start, const int* g_row_start, int E_l, int Nt, int S_rows,
                                          int n, int nk, int my, int stride, int& round, int& round0, int dw_rows) {
    GgTile t;
    t.g = t.nt = t.row0 = 0;
    t.rv = 0;
    t.ks0 = 0; t.nks = nk;
    const int rounds = (n + stride - 1) / stride;
    while (round < rounds) {
        if (round >= round0 + GG_TT) {
            __syncthreads();  // (every wave has read what it needed of the old table)
            round0 = round;
            gg_fill_table<BM, DW>(s_tiles, g_tile_start, g_row_start, E_l, Nt, S_rows, n, my, stride, round0, dw_rows);
            __syncthreads();
        }
        const int4 e = s_tiles[round - round0];
        ++round;
        const int rv = __builtin_amdgcn_readfirstlane(e.w);
        if (rv > 0) {
            t.g = __builtin_amdgcn_readfirstlane(e.x); t.nt = __builtin_amdgcn_readfirstlane(e.y);
            t.row0 = __builtin_amdgcn_readfirstlane(e.z); t.rv = rv;
            if constexpr (DW) {
                t.ks0 = g_row_start[t.g];
                t.nks = (g_row_start[t.g + 1] - t.ks0 + 63) / 64 * 2;
            }
            break;
        }
    }
    return t;
}


// Where the loads of a stage read: a scalar pointer, or (RANGE) a descriptor that ends where the group does.
template <bool RANGE>
__device__ __forceinline__ auto gg_stage_src(const uint8_t* base, size_t off, long long left) {
    if constexpr (RANGE) return gg_range(base + off, left - (long long)off);
    else return gg_uniform(base + off);
}

// NWM x 2 wave64s per workgroup; every wave owns a (BM/NWM) x 128 block of the tile.
//
// K moves through LDS in a ring of NRING stages of ROWB bytes per tile row.  A stage is one MFMA block
// (one 16x16x32 bf16 or 32x32x64 fp8 MFMA per pair of fragments).  Every wave takes the fragments of stage s + 1 into registers during
// block s.  Activations come in pairs of stages (2 p, 2 p + 1): the pair's slots are free after block 2 p, and block 2 p + 1 requests pair p + 2 into
// them, which block 2 p + 3 reads.  Weights come by stages: block 2 p requests stages 2 p + 3 and 2 p + 4.  The loads of a block stand one by one
// between its MFMAs, so the load pipe sees a steady stream.  (DW: block s requests stage s + 4 of both.)
// BSA: the activation operand carries block scales (fp8 down projection: GemmParams::a_bscale), applied by the MFMAs.
// TRACE: the same kernel with time stamps (GemmParams::trace); product launches never use it.
template <int BM, int NWM, int EPI, bool FP8, int BMODE = GG_B_PACKED, bool BSA = false, bool TRACE = false>
__global__ __launch_bounds__(NWM * 2 * WAVE, 1) void grouped_gemm_kernel(const GemmParams p) {
    constexpr bool DW = BMODE == GG_B_DW, BT = BMODE == GG_B_T, BN_PAIR = BMODE == GG_B_NP, BN_RAW = BMODE == GG_B_N || BN_PAIR;
    static_assert(!FP8 || BMODE == GG_B_PACKED, "raw weights are a bf16 matter");
    static_assert(BMODE != GG_B_NP || EPI == EPI_SWIGLU, "pairs are what SwiGLU multiplies with");
    constexpr int BTR = DW ? 512 : 256;   // (operands transposed out of LDS) row pitch of a stage of B
    static_assert(!TRACE || !DW, "time stamps: whole-tile forward launches only");
    [[maybe_unused]] int tr_tile = 0, tr_blk = 0;  // (TRACE) words written so far
#define GG_TRACE_TILE()                                                                                                    \
    do {                                                                                                                   \
        if constexpr (TRACE) {                                                                                             \
            if (threadIdx.x == 0 && tr_tile < GG_TRACE_TILE_WORDS) p.trace[(size_t)blockIdx.x * GG_TRACE_TILE_WORDS + tr_tile] = wall_clock64(); \
            ++tr_tile;                                                                                                     \
        }                                                                                                                  \
    } while (0)
    static_assert(!DW || (!FP8 && EPI == EPI_NONE), "the weight-gradient mode is a plain bf16 GEMM");
    static_assert(!BSA || FP8, "block scales belong to the fp8 MFMA");
    constexpr bool VARK = DW;  // the K range differs from tile to tile
    constexpr bool PEEL = !VARK && !BSA;  // the tile's first two blocks written out apart (see below)
    constexpr bool QOUT = FP8 && EPI == EPI_SWIGLU;  // the epilogue stores e4m3 codes and block scales
    constexpr int BN = GG_BN;
    constexpr int ES = FP8 ? 1 : 2;
    constexpr int NW = NWM * 2;                        // waves per workgroup
    // bf16: 16x16x32 MFMAs (4 accumulator registers each; under the power limit this shape sustains about
    // 15 % more than 32x32x16, which moves twice the accumulator bytes per flop); fp8: 32x32x64
    constexpr int MT = FP8 ? 32 : 16;                  // MFMA tile edge
    constexpr int CF = FP8 ? 2 : 1;                    // 16-byte LDS chunks per fragment and lane
    constexpr int TM = BM / (NWM * MT), TN = BN / (2 * MT);  // MFMA tiles per wave
    constexpr int NT = TM * TN;                        // MFMAs per K stage and wave
    constexpr int RPA = DW ? 2 : CF, RPB = DW || BN_RAW ? 2 : CF;  // LDS reads per fragment (transposing reads bring 8 bytes)
    constexpr int NRD = TM * RPA + TN * RPB;           // fragment reads per K stage and wave
    constexpr int LR = NW * WROWS;                     // rows fetched per load round (16 per wave)
    constexpr int RA = BM / LR, RB = BN / LR;          // load rounds per stage
    constexpr int LPS = RA + RB;                       // HBM->LDS loads per lane per stage
    // Activations come a pair of stages at a time, 128 bytes of their rows (whole cache lines) to a load: the load path takes pieces of 64
    // bytes at half the rate (see gg_swz_wide).  With a stage at a time: 33618 rows in 32 groups x 7168 x (2 x 2048) 1650 us, now 1563; x 2048 x 7168 884 -> 851;
    // 32972 x 4096 x (2 x 14336) 5519 -> 5300, x 14336 x 4096 2660 -> 2590; fp8 MLP of 81920 x 2048 x 1408 in 15 groups 858 -> 824 (same box each).
    // (DW: a stage's rows are 512 bytes as it is)
    constexpr bool WIDE = !DW;
    constexpr int LA = WIDE ? 2 * RA : RA;             // loads of A per lane: per pair (WIDE) or stage
    constexpr int LE = WIDE ? 2 * RB : LPS, LO = WIDE ? LA : LPS;  // loads behind the MFMAs of a block in an even, odd slot
    // Where the other instructions of a block sit.  bf16: a 16x16x32 MFMA covers only 16 cycles of other issue,
    // so no MFMA gets more than one: the fragment reads go behind every RSTEP-th MFMA of the first half of the
    // block (they must have landed when the block ends in the hand-over), the loads are spread evenly over the
    // whole block, behind other MFMAs where that fits (a steady stream to the load pipe: bunched at either end
    // of the block they cost 7 % more cycles).  fp8: a 32x32x64 MFMA covers 64 cycles and there are few of them;
    // two reads go behind each of the first MFMAs.
    constexpr int RPM = NRD > NT / 2 ? 2 : 1;                 // reads behind one MFMA
    constexpr int RFIRST = 0;                                 // first MFMA with a read behind it
    constexpr int RSTEP = (NT / 2) * RPM / NRD > 0 ? (NT / 2) * RPM / NRD : 1;  // MFMAs from one read group to the next
    constexpr int LFIRST = NT > LE && NT > LO ? 1 : 0;        // first MFMA with a load behind it
    // MFMAs from one load to the next.  WIDE: the pair of A is needed when the next block ends, so its loads take the first half of theirs; those of B,
    // the first of which are as urgent, three quarters (mixtral's gate / up GEMM 5238 -> 5150 us against loads over whole blocks, the others 0.3 %; all within half: 5192)
    constexpr int LSE = WIDE ? ((NT - LFIRST) / LE * 3 + 3) / 4 : (NT - LFIRST) / LE, LSO = WIDE ? ((NT - LFIRST) / LO + 1) / 2 : (NT - LFIRST) / LO;
    constexpr int ASLOT = BM * CHUNKS, BSLOT = BN * CHUNKS;  // uint4 per ring slot
    static_assert(TM * MT * NWM == BM && BM % LR == 0 && BN % LR == 0 && NT <= 64 && LSE >= 1 && LFIRST + LSE * (LE - 1) < NT && LSO >= 1 && LFIRST + LSO * (LO - 1) < NT && RFIRST + RSTEP * ((NRD - 1) / RPM) < NT, "tile shape");
    static_assert(CHUNKS == 4 && NRING == 4, "the stage schedule below is written for 64-byte stages in four slots");

    __shared__ __align__(1024) uint4 sA[NRING * ASLOT];
    __shared__ __align__(1024) uint4 sB[NRING * BSLOT];
    __shared__ int g_tile_start[GG_MAXG + 1];
    __shared__ int g_row_start[GG_MAXG + 1];
    // what the epilogue needs from global memory per tile row / tile column (fp8 scales, the output row map)
    // (two copies, used by alternate tiles: a wave may enter the next tile while another is still in this one's epilogue)
    __shared__ __align__(16) float s_row_scale[2][BM];
    __shared__ __align__(16) float s_col_scale[2][BN];
    __shared__ int s_crow[2][BM];
    __shared__ int s_amap[BM];              // the NEXT tile's input rows (a_map), fetched while this one is multiplied
    // BSA: the block-scale bytes of the tile's rows for a PAIR of K stages (4 blocks of 32 k = one dword per row), two
    // copies: pairs alternate like the ring slots they travel with
    __shared__ uint32_t s_hsc[BSA ? 2 : 1][BSA ? BM : 1];
    __shared__ __align__(16) int4 s_tiles[GG_TT];
    static_assert(BM <= NWM * 2 * WAVE && BN <= NWM * 2 * WAVE, "one thread per tile row and per tile column");

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wave_s = __builtin_amdgcn_readfirstlane(wave);  // the same, known to be wave-uniform (a scalar register)
    const int wm = wave >> 1, wn = wave & 1;
    const int Nt = p.Npad / BN;

    if (tid == 0) {
        int ts = 0, rs = 0;
        for (int g = 0; g < p.E_l; ++g) {
            g_tile_start[g] = ts;
            g_row_start[g] = rs;
            int c = max(p.cnt[g], 0);
            if constexpr (DW) {
                // tiles of the group's own dw_rows x N output
                c = min(c, max(p.dw_src_rows - rs, 0));
                ts += c > 0 ? ((p.dw_rows + BM - 1) / BM) * Nt : 0;
                rs += c;
            } else {
                // (counts that claim more rows than the buffers hold are cut at S_rows: the host's bound on the number of
                // tiles, which decides whether the whole-tile launch is left out, counts on it)
                c = min(c, max(p.S_rows - rs, 0));
                ts += ((c + BM - 1) / BM) * Nt;
                rs += c;
            }
        }
        g_tile_start[p.E_l] = ts;
        g_row_start[p.E_l] = rs;
    }
    __syncthreads();
    if constexpr (DW) {
        // the gradient of a group without rows is zero (it has no tile below)
        for (int g = 0; g < p.E_l; ++g) {
            if (g_row_start[g + 1] > g_row_start[g]) continue;
            const int nv = (p.dw_split ? p.dw_split : p.N) / 8;  // 16-byte vectors per output row (and half, where split)
            bf16_t* c = (bf16_t*)p.C + (size_t)g * p.c_group_stride;
            for (int i = blockIdx.x * NW * WAVE + threadIdx.x; i < p.dw_rows * nv; i += gridDim.x * NW * WAVE) {
                bf16_t* o = c + (size_t)(i / nv) * p.ldc + (i % nv) * 8;
                *(uint4*)o = make_uint4(0, 0, 0, 0);
                if (p.dw_split) *(uint4*)(o + p.dw_delta) = make_uint4(0, 0, 0, 0);
            }
        }
    }
    if constexpr (!DW && !FP8) gg_zero_tail(p, g_row_start[p.E_l]);
    const int nk = (p.K * ES) / ROWB;  // ring stages per tile; even (K * ES is a multiple of 2 * ROWB)
    const int n_tiles = gg_whole_tiles(g_tile_start[p.E_l], (int)gridDim.x, DW ? 0 : p.tail_max);

    // XCD-aware position inside a round of gridDim.x tiles: workgroups b, b+8, b+16, ... share an L2.
    int my = blockIdx.x;
    if (gridDim.x == 256) {
        const int xcd = blockIdx.x & 7, l = blockIdx.x >> 3;
        my = (((xcd >> 1) * 4 + (l >> 3)) * SUP) + ((xcd & 1) * 8 + (l & 7));
    }

    // lane-constant pieces of the addressing.  A tile row is 4 chunks of 16 bytes; row r keeps logical
    // chunk c at position c ^ gg_swz(r >> 2), which makes both the 16-rows-per-instruction DMA writes
    // and the 128-bit fragment reads (rows = lane % 32) bank-conflict free.
    const int lrow = wave * WROWS + (lane >> 2);         // row inside a load round
    const int lchunk = (lane & 3) ^ gg_swz(lane >> 4);   // global 16-byte chunk this lane fetches
    const int fswz = gg_swz(lane >> 2);                  // swizzle of the fragment row (tile rows start at multiples of 16)
    // first 16-byte chunk of the lane's fragment: bf16 lanes 16q .. 16q+15 take chunk q of rows 0 .. 15;
    // fp8 lanes 32h .. 32h+31 take chunks h and h + 2 of rows 0 .. 31 (both operands alike, so every k meets its partner):
    // the MFMA's first four operand registers of the two lane halves are then bytes 0-31 of the stage and the other four
    // bytes 32-63 -- the two blocks of 32 k that the scaled form of the instruction scales separately
    constexpr int FSTEP = FP8 ? 2 : 1;  // distance of a lane's second chunk
    const int fpos = (FP8 ? (lane >> 5) : (lane >> 4)) ^ fswz;
    const uint4* fa = sA + (wm * (BM / NWM) + (lane & (MT - 1))) * (WIDE ? 2 * CHUNKS : CHUNKS);
    [[maybe_unused]] const int fpos_a = (FP8 ? (lane >> 5) : (lane >> 4)) ^ gg_swz_wide(lane);
    const uint4* fb = sB + (wn * (BN / 2) + (lane & (MT - 1))) * CHUNKS;
    const uint32_t la0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)(sA + wave * WROWS * CHUNKS));
    const uint32_t lb0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)(sB + wave * WROWS * CHUNKS));

    const uint32_t ldk = DW ? (uint32_t)p.dw_rows * 2u : (uint32_t)(p.K * ES);  // row pitch of A in bytes
    // row pitch of B where it is not re-tiled: (BT) its columns are the reduction, half of it per matrix of a pair
    [[maybe_unused]] const uint32_t ldb = BT ? (uint32_t)(p.B2 ? p.K / 2 : p.K) * 2u : (uint32_t)p.N * 2u;
    [[maybe_unused]] const size_t b_group = (size_t)p.K / (BT && p.B2 ? 2 : 1) * p.N * 2;  // (BT, BN_RAW) bytes per group and matrix
    const size_t b_slab = (size_t)p.Npad * ROWB;  // packed weights are slab-major: [group][K slab][Npad rows][ROWB bytes]
    // per-round lane offsets into the weight slab (vector registers: no scalar address arithmetic per load)
    uint32_t b_off[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) {
        if constexpr (DW) b_off[r] = (uint32_t)(2 * (r * NW + wave) + (lane >> 5)) * ldb + (uint32_t)((lane & 31) ^ (4 * ((2 * wave + (lane >> 5)) & 3))) * 16u;
        else if constexpr (BT) b_off[r] = (uint32_t)gg_packed_col<false>(r * LR + lrow) * ldb + lchunk * 16;
        // (BN_RAW: a 1 KB load brings four rows of 256 bytes, half of a stage's loads per region of 128 columns)
        else if constexpr (BN_RAW) b_off[r] = (uint32_t)(4 * (r % (RB / 2) * NW + wave) + (lane >> 4)) * ldb + (uint32_t)((lane & 15) ^ (4 * (lane >> 4))) * 16u;
        else b_off[r] = (uint32_t)(r * LR + lrow) * ROWB + lchunk * 16;
    }
    static_assert(!BN_RAW || (RB % 2 == 0 && RB / 2 * NW == 8), "eight loads per region");
    // DW: an LDS stage holds 32 rows of 512 bytes per operand (a 1 KB load brings two of them); 16-byte chunk c of row k lies at
    // position c ^ f(k), which spreads the eight rows that half a wave reads together over the banks: f = 2 (k % 4 + 4 (k / 8 % 2))
    // for A, read 32 contiguous bytes a row, f = 4 (k % 4) for B, read 8 bytes of four chunks in a row (the permuted columns).
    [[maybe_unused]] uint32_t tr_a = 0, tr_b = 0;
    if constexpr (DW) {
        const int kq = (lane >> 4) * 8 + ((lane & 15) >> 2), k4 = (lane & 15) >> 2, q4 = lane & 3;  // first k, its low bits, column quad
        tr_a = (uint32_t)(uintptr_t)(lds_ptr_t)sA + kq * 512 + (((wm * 16 + (q4 >> 1)) ^ (2 * (k4 + 4 * ((lane >> 4) & 1)))) * 16) + (q4 & 1) * 8;
        tr_b = (uint32_t)(uintptr_t)(lds_ptr_t)sB + kq * 512 + (((wn * 16 + q4) ^ (4 * k4)) * 16);
    }
    // BN_RAW: a stage of B is two regions of 32 rows of 256 bytes: the two column halves of the tile, or its gate and its up columns;
    // chunk c of row k at position c ^ 4 (k % 4), as in DW's B.
    if constexpr (BN_RAW) {
        const int kq = (lane >> 4) * 8 + ((lane & 15) >> 2), k4 = (lane & 15) >> 2, q4 = lane & 3;
        tr_b = (uint32_t)(uintptr_t)(lds_ptr_t)sB + (BN_PAIR ? 0 : wn * (BSLOT * 8)) + kq * 256 + ((((BN_PAIR ? wn * 8 : 0) + q4) ^ (4 * k4)) * 16);
    }
    // LDS address of fragment i of A (16 rows of the product) / j of B (its columns 32 (j / 2) + 8 q + 4 (j % 2) ..) in ring slot sl
#define GG_TR_A(i, sl) ((tr_a ^ ((i) * 32)) + (sl) * (ASLOT * 16))
#define GG_TR_B(j, sl)                                                                                                  \
    ((tr_b ^ (BN_PAIR ? ((j) >> 2) * 64 : ((j) >> 1) * 64)) + (BN_PAIR ? (((j) >> 1) & 1) * (BSLOT * 8) : 0) + (sl) * (BSLOT * 16) + ((j) & 1) * 8)

#define GG_MAPROW_GLOBAL(t, l) p.a_map[(t).row0 + (l)]   /* the first tile: straight from memory */
#define GG_MAPROW_LDS(t, l) s_amap[(l)]                  /* later tiles: fetched into LDS one tile ahead */
#define GG_TILE_PTRS(t, Ab_, Bb_, aoff_, MAPROW_)                                                          \
    const uint8_t* Ab_ = DW ? p.A + (size_t)(t).ks0 * ldk + (size_t)(t).row0 * 2                             \
                            : (p.a_map ? p.A : p.A + (size_t)(t).row0 * p.K * ES) + (size_t)(t).ks0 * ROWB;  \
    const size_t bo0_ = DW ? (size_t)(t).ks0 * ldb + (size_t)(t).nt * BN * 2                                  \
                      : BT ? (size_t)(t).g * b_group + (size_t)(t).nt * BN * ldb + (size_t)(t).ks0 / (p.B2 ? 2 : 1) * ROWB \
                      : BN_RAW ? (size_t)(t).g * b_group + (size_t)(t).nt * (BN_PAIR ? BN : 2 * BN) + (size_t)(t).ks0 * 32 * ldb \
                               : (size_t)(t).g * p.Npad * p.K * ES + (size_t)(t).nt * BN * ROWB + (size_t)(t).ks0 * b_slab; \
    const uint8_t* Bb_ = p.B + bo0_;                                                                          \
    if constexpr (BT || BN_RAW) dw_left_b = (long long)p.E_l * b_group - (long long)bo0_;                      \
    uint32_t aoff_[LA];                                                                                     \
    const int ln_ = gg_lane_now();  /* lrow and lchunk again, derived per tile */                              \
    if constexpr (DW) {                                                                                      \
        const long long rows_ = g_row_start[(t).g + 1] - (t).ks0;                                            \
        dw_left_a = rows_ * ldk - (long long)(t).row0 * 2;                                                    \
        dw_left_b = rows_ * ldb - (long long)(t).nt * BN * 2;                                                 \
        _Pragma("unroll") for (int r = 0; r < RA; ++r)                                                        \
            aoff_[r] = (uint32_t)(2 * (r * NW + wave_s) + (ln_ >> 5)) * ldk +                                   \
                       (uint32_t)((ln_ & 31) ^ (2 * (((2 * wave_s + (ln_ >> 5)) & 3) + 4 * (r & 1)))) * 16u;      \
    } else {                                                                                                 \
        const int lrow_ = wave_s * 8 + (ln_ >> 3);                                                             \
        const uint32_t lcb_ = (uint32_t)(((ln_ & 7) ^ gg_swz_wide(lrow_)) * 16);                                \
        _Pragma("unroll") for (int r = 0; r < LA; ++r) {                                                      \
            const int lr_ = max(min(r * NW * 8 + lrow_, (t).rv - 1), 0);  /* tile row this lane fetches, clamped */ \
            aoff_[r] = (uint32_t)(p.a_map ? max(MAPROW_(t, lr_), 0) : lr_) * ldk + lcb_;                      \
        }                                                                                                     \
    }
    [[maybe_unused]] const ptrdiff_t b2_delta = p.B2 - p.B;
    [[maybe_unused]] long long dw_left_a = 0, dw_left_b = 0;  // (DW) bytes of the operands from the tile's corner to the end of the group
    // load d of a stage of B (0 .. RB - 1), of a pair of stages or a stage of A (0 .. LA - 1)
#define GG_LDB(d, bp_, slot) gg_dma16(BN_RAW && (d) >= RB / 2 ? bp_##2 : bp_, b_off[d], lb0 + (slot) * BSLOT * 16, (d) * LR * CHUNKS * 16)
#define GG_LDA(d, ap_, aoff_, slot) gg_dma16(ap_, aoff_[d], la0 + (slot) * ASLOT * 16, (d) * (WIDE ? NW * 1024 : LR * CHUNKS * 16))
    // Where stage `st` of B and the stage (WIDE: the pair that starts with it) `st` of A lie, clamped to the tile's last ones: the ring never holds data
    // of another tile, and a repeated load of the last stage lands in a slot nobody reads again
#define GG_A_PTR(Ab_, st, ap_, nks_)                                                           \
    const auto ap_ = gg_stage_src<DW>(Ab_, (size_t)min((st), (nks_) - (WIDE ? 2 : 1)) * (DW ? (size_t)32 * ldk : (size_t)ROWB), dw_left_a);
#define GG_B_PTRS(Bb_, st, bp_, nks_)                                                          \
    const int st_##bp_ = min((st), (nks_) - 1);                                                \
    const size_t so_##bp_ = BT ? (size_t)(p.B2 ? st_##bp_ >> 1 : st_##bp_) * ROWB : (size_t)st_##bp_ * (DW || BN_RAW ? (size_t)32 * ldb : b_slab); \
    const auto bp_ = gg_stage_src<BMODE != GG_B_PACKED>(BT && p.B2 && (st_##bp_ & 1) ? Bb_ + b2_delta : Bb_, so_##bp_, dw_left_b);   \
    /* (BN_RAW: the second region, in the other matrix or 256 bytes further along the rows) */                  \
    [[maybe_unused]] const auto bp_##2 = gg_stage_src<BMODE != GG_B_PACKED>(BN_RAW ? Bb_ + (BN_PAIR ? b2_delta : 256) : Bb_, so_##bp_, \
                                                                            dw_left_b - (BN_RAW && !BN_PAIR ? 256 : 0));
#define GG_ISSUE_A(Ab_, aoff_, st, slot, nks_)                                                 \
    do {                                                                                       \
        GG_A_PTR(Ab_, st, ap_i, nks_)                                                          \
        _Pragma("unroll") for (int d_ = 0; d_ < LA; ++d_) GG_LDA(d_, ap_i, aoff_, slot);        \
    } while (0)
#define GG_ISSUE_B(Bb_, st, slot, nks_)                                                        \
    do {                                                                                       \
        GG_B_PTRS(Bb_, st, bp_i, nks_)                                                         \
        _Pragma("unroll") for (int d_ = 0; d_ < RB; ++d_) GG_LDB(d_, bp_i, slot);               \
    } while (0)
    // what a tile has in flight before its first MFMA: its first four stages, one per ring slot (WIDE: the first block requests the fourth stage of B)
#define GG_PROLOGUE(Ab_, Bb_, aoff_, nks_)                    \
    do {                                                      \
        GG_SC_DMA(0, nks_, 0);                                \
        GG_ISSUE_A(Ab_, aoff_, 0, 0, nks_);                   \
        GG_ISSUE_B(Bb_, 0, 0, nks_);                          \
        if constexpr (!WIDE) GG_ISSUE_A(Ab_, aoff_, 1, 1, nks_); \
        GG_ISSUE_B(Bb_, 1, 1, nks_);                          \
        GG_SC_DMA(2, nks_, 2);                                \
        GG_ISSUE_A(Ab_, aoff_, 2, 2, nks_);                   \
        GG_ISSUE_B(Bb_, 2, 2, nks_);                          \
        if constexpr (!WIDE) {                                \
            GG_ISSUE_A(Ab_, aoff_, 3, 3, nks_);               \
            GG_ISSUE_B(Bb_, 3, 3, nks_);                      \
        }                                                     \
    } while (0)

    // BSA: the block-scale bytes travel with the stages.  One dword per tile row holds the four scale bytes of a PAIR of
    // stages (2 x 64 bytes of K = 4 blocks of 32); it is requested, one per thread, straight into LDS with the loads of the
    // pair's even stage (same block, same ring slot: copy slot / 2), and read back by the lanes one block before the pair's
    // first MFMA.  sc_row0 / sc_rv / sc_ks0 describe the tile the loads currently point at (switched with Ab / Bb).
    [[maybe_unused]] int sc_row0 = 0, sc_rv = 1, sc_ks0 = 0;
    [[maybe_unused]] int sc[TM];
#define GG_SC_DMA(st, nks_, slot)                                                                                          \
    do {                                                                                                                   \
        if constexpr (BSA) {                                                                                               \
            if (wave_s * WAVE < BM) {                                                                                      \
                const int stc_ = min((st), (nks_) - 1);                                                                    \
                const int tid_c = wave_s * WAVE + gg_lane_now();                                                           \
                const uint32_t vo_ = (uint32_t)(sc_row0 + min(tid_c, sc_rv - 1)) * (uint32_t)p.bs_pitch +                  \
                                     (uint32_t)(((sc_ks0 + stc_) >> 1) << 2);                                              \
                gg_dma4(gg_uniform(p.a_bscale), vo_,                                                                       \
                        __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)(&s_hsc[(slot) >> 1][wave_s * WAVE]))); \
            }                                                                                                              \
        }                                                                                                                  \
    } while (0)
    // lane 32 h + r of a wave takes, for each of its row tiles, the dword of row r shifted so that byte 0 is the scale of
    // block h of the pair's even stage and byte 2 that of its odd stage (the MFMA's op_sel picks 0 or 2), each raised by
    // what the weight operand's constant scale byte lacks to 2^0.  One set of registers: a pair's dwords are read behind the
    // last MFMA of the pair before.
#define GG_SC_READ(SET_)                                                                                                   \
    do {                                                                                                                   \
        if constexpr (BSA) {                                                                                               \
            const int lnr_ = gg_lane_now();                                                                                \
            _Pragma("unroll") for (int i_ = 0; i_ < TM; ++i_)                                                               \
                sc[i_] = (int)(((s_hsc[SET_][(wave_s >> 1) * (BM / NWM) + i_ * MT + (lnr_ & 31)] >> ((lnr_ >> 5) * 8)) & 0x00ff00ffu) + \
                               (uint32_t)(127 - GG_WSCALE) * 0x00010001u);                                                 \
        }                                                                                                                  \
    } while (0)

    int round = 0, round0 = 0;
    gg_fill_table<BM, DW>(s_tiles, g_tile_start, g_row_start, p.E_l, Nt, p.S_rows, n_tiles, my, (int)gridDim.x, 0, p.dw_rows);
    __syncthreads();
    GgTile cur = gg_walk<BM, DW>(s_tiles, g_tile_start, g_row_start, p.E_l, Nt, p.S_rows, n_tiles, nk, my, (int)gridDim.x, round, round0, p.dw_rows);
    uint32_t a_off[LA];
    const uint8_t *Ab = p.A, *Bb = p.B;
    if (cur.rv > 0) {
        GG_TILE_PTRS(cur, Ab0, Bb0, a_off0, GG_MAPROW_GLOBAL);
        Ab = Ab0;
        Bb = Bb0;
#pragma unroll
        for (int r = 0; r < LA; ++r) a_off[r] = a_off0[r];
        sc_row0 = cur.row0; sc_rv = cur.rv; sc_ks0 = cur.ks0;
        GG_PROLOGUE(Ab, Bb, a_off, (VARK ? cur.nks : nk));
    }
    // The ring runs on from one tile into the next: the last four blocks of a tile refill their slots with the first
    // four stages of the NEXT tile (when the table has it at hand), its last block reads that tile's first fragments,
    // and the next tile then starts with everything in place -- no burst of 32 loads per lane with the matrix pipes
    // idle, no pair of barriers.  `pre` says that the tile at hand was prepared like that; phi is the ring slot of its
    // first stage (the ring is not realigned between tiles); tpar picks the copy of the epilogue data.
    uint4 fA0[TM * CF], fB0[TN * CF], fA1[TM * CF], fB1[TN * CF];
    bool pre = false;
    int phi = 0, tpar = 0;
    while (cur.rv > 0) {
        const int g = __builtin_amdgcn_readfirstlane(cur.g), nt = __builtin_amdgcn_readfirstlane(cur.nt);
        const int row0 = __builtin_amdgcn_readfirstlane(cur.row0), rv = __builtin_amdgcn_readfirstlane(cur.rv);
        const int nks = VARK ? __builtin_amdgcn_readfirstlane(cur.nks) : nk;

        typedef typename std::conditional<FP8, floatx16, floatx4>::type acc_t;
        acc_t acc[TM][TN];  // (not cleared where the MFMAs of the tile's first block start the sums)
        if constexpr (!PEEL) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < (FP8 ? 16 : 4); ++v) acc[i][j][v] = 0.f;
        }

        // ---- One MFMA block per 64-byte stage.  Block s multiplies the fragments of stage s, reads those of
        // stage s+1 (all issued in the first half of the block, so they have landed when the block ends) and
        // requests what its predecessors have drained the slots for (above); the hand-over at its end waits for the
        // wave's own loads of stage s+2 -- what was issued after them may stay in flight: behind a block in an even slot its own loads of B, behind one in an
        // odd slot its own of A and the second half of the B loads before -- and meets the other waves.  Loads past the end of the tile are clamped
        // to its last stage (straight-line code, constant wait counts); in the last block the "next
        // fragments" are whatever the next slot holds and are never used.  Every instruction is pinned by
        // scheduling fences: each read and each load is issued in the shadow of an MFMA.
        // fragment read R of the next stage: operand R / CF (activation rows first, then weight rows), chunk R % CF
#define GG_RD(R, NA_, NB_)                                                                               \
    do {                                                                                                 \
        constexpr bool ra_ = (R) < TM * RPA;                                                             \
        constexpr int ro_ = ra_ ? (R) / RPA : TM + ((R) - TM * RPA) / RPB, rh_ = ra_ ? (R) % RPA : ((R) - TM * RPA) % RPB; \
        if constexpr (ra_ ? DW : DW || BN_RAW) {                                                         \
            const uint2 v_ = ra_ ? gg_read_tr<512>(GG_TR_A((ra_ ? ro_ : 0), nsl_), rh_) : gg_read_tr<BTR>(GG_TR_B((ra_ ? 0 : ro_ - TM), nsl_), rh_); \
            uint4& f_ = ro_ < TM ? NA_[ro_ < TM ? ro_ : 0] : NB_[ro_ < TM ? 0 : ro_ - TM];               \
            if constexpr (rh_ == 0) { f_.x = v_.x; f_.y = v_.y; } else { f_.z = v_.x; f_.w = v_.y; }      \
        }                                                                                                \
        else if constexpr (ro_ < TM) NA_[ro_ * CF + rh_] = nfa_[ro_ * MT * 2 * CHUNKS + (fpos_a ^ (nodd_ * CHUNKS + rh_ * FSTEP))];  \
        else NB_[(ro_ - TM) * CF + rh_] = nfb_[(ro_ - TM) * MT * CHUNKS + (fpos ^ (rh_ * FSTEP))];       \
    } while (0)
#define GG_ML(I, FA_, FB_, NA_, NB_, slot, Z_, EVEN_, SET_)                                                \
    do {                                                                                                 \
        if constexpr ((I) < NT) {                                                                        \
            /* boustrophedon over the wave's MFMA tiles: every instruction keeps one operand of the one before it */ \
            constexpr int pa_ = (I) / TN, pb_ = (pa_ & 1) ? TN - 1 - (I) % TN : (I) % TN;                \
            if constexpr (FP8 && BSA) mma_fp8_k64_bs<Z_, (EVEN_) ? 0 : 2, NWM == 4>(acc[pa_][pb_], FB_[2 * pb_], FB_[2 * pb_ + 1], FA_[2 * pa_], FA_[2 * pa_ + 1], sc[pa_]); \
            else if constexpr (FP8) mma_fp8_k64<Z_>(acc[pa_][pb_], FB_[2 * pb_], FB_[2 * pb_ + 1], FA_[2 * pa_], FA_[2 * pa_ + 1]); \
            else mma_bf16_k32<Z_>(acc[pa_][pb_], FB_[pb_], FA_[pa_]);                                    \
            __builtin_amdgcn_sched_barrier(0);                                                           \
            constexpr int ls_ = (EVEN_) ? LSE : LSO, ln_ = (EVEN_) ? LE : LO;                            \
            constexpr int ld_ = (I) >= LFIRST && ((I) - LFIRST) % ls_ == 0 ? ((I) - LFIRST) / ls_ : ln_;  /* load behind this MFMA */ \
            if constexpr (ld_ < ln_) {                                                                   \
                if constexpr (!WIDE) {                                                                   \
                    if constexpr (ld_ < RA) GG_LDA((ld_ < RA ? ld_ : 0), ap_, a_off, slot);              \
                    else GG_LDB((ld_ >= RA ? ld_ - RA : 0), bp_, slot);                                  \
                } else if constexpr (!(EVEN_)) GG_LDA((ld_ < LA ? ld_ : 0), ap_, a_off, ((slot) + 3) & 3);  \
                else if constexpr (ld_ < RB) GG_LDB((ld_ < RB ? ld_ : 0), bq_, ((slot) + 3) & 3);          \
                else GG_LDB((ld_ >= RB && ld_ < 2 * RB ? ld_ - RB : 0), bp_, slot);                       \
            }                                                                                            \
            constexpr int r0_ = (I) >= RFIRST && ((I) - RFIRST) % RSTEP == 0 ? (((I) - RFIRST) / RSTEP) * RPM : NRD; /* first read */ \
            if constexpr (r0_ < NRD) GG_RD((r0_ < NRD ? r0_ : 0), NA_, NB_);                             \
            if constexpr (RPM > 1 && r0_ + 1 < NRD) GG_RD((r0_ + 1 < NRD ? r0_ + 1 : 0), NA_, NB_);      \
            __builtin_amdgcn_sched_barrier(0);                                                           \
        }                                                                                                \
    } while (0)
#define GG_ML8(I, FA_, FB_, NA_, NB_, slot, Z_, E_, S_)                                                          \
    GG_ML((I) + 0, FA_, FB_, NA_, NB_, slot, Z_, E_, S_); GG_ML((I) + 1, FA_, FB_, NA_, NB_, slot, Z_, E_, S_);           \
    GG_ML((I) + 2, FA_, FB_, NA_, NB_, slot, Z_, E_, S_); GG_ML((I) + 3, FA_, FB_, NA_, NB_, slot, Z_, E_, S_);           \
    GG_ML((I) + 4, FA_, FB_, NA_, NB_, slot, Z_, E_, S_); GG_ML((I) + 5, FA_, FB_, NA_, NB_, slot, Z_, E_, S_);           \
    GG_ML((I) + 6, FA_, FB_, NA_, NB_, slot, Z_, E_, S_); GG_ML((I) + 7, FA_, FB_, NA_, NB_, slot, Z_, E_, S_)
    // SET_: which copy of the block scales (BSA) the stage's pair uses: slot / 2, as a literal (0 where the slot is a run-time value: no BSA there)
#define GG_STAGE(FA_, FB_, NA_, NB_, SL, EVEN_, s, last, Z_, SET_)                                                \
    do {                                                                                                 \
        /* WIDE: a block in an even slot requests B's stages s + 3 (into the slot whose fragments its predecessor read last) and s + 4, \
           one in an odd slot A's pair of stages s + 3 and s + 4 */                                       \
        GG_B_PTRS(Bb, (s) + 3 - kbase, bq_, nks_ld)                                                       \
        if constexpr (EVEN_) { /* (a block in an even slot) */                                           \
            /* from block nks - 4 on the loads fetch the next tile (but for the last stage of B), if it is at hand; not in a tile's first block: the  \
               row map that the tile's top requested must have landed and been handed over (one block end at least) */ \
            if ((s) == nks - 4 && (s) > 0) {                                                             \
                const GgTile pk_ = gg_peek<DW>(s_tiles, g_row_start, nk, my, (int)gridDim.x, round, round0); \
                if (pk_.rv > 0) {                                                                        \
                    GG_TILE_PTRS(pk_, Ab_s, Bb_s, a_off_s, GG_MAPROW_LDS);                               \
                    Ab = Ab_s;                                                                           \
                    Bb = Bb_s;                                                                           \
                    _Pragma("unroll") for (int r = 0; r < LA; ++r) a_off[r] = a_off_s[r];                \
                    kbase = nks;                                                                         \
                    nks_ld = VARK ? pk_.nks : nk;                                                        \
                    seam = true;                                                                         \
                    sc_row0 = pk_.row0; sc_rv = pk_.rv; sc_ks0 = pk_.ks0;                                \
                }                                                                                        \
            }                                                                                            \
        }                                                                                                \
        if constexpr (!(EVEN_)) GG_SC_DMA((s) + 3 - kbase, nks_ld, SET_ * 2);  /* (the pair's scale dwords) */ \
        GG_A_PTR(Ab, (s) + (WIDE ? 3 : 4) - kbase, ap_, nks_ld)                                          \
        GG_B_PTRS(Bb, (s) + 4 - kbase, bp_, nks_ld)                                                      \
        [[maybe_unused]] constexpr int nodd_ = (EVEN_) ? 1 : 0;  /* parity of the stage whose fragments are read */ \
        [[maybe_unused]] const int nsl_ = ((SL) + 1) & 3;                                                \
        const uint4* nfa_ = fa + (WIDE ? (((SL) + 1) & 3) >> 1 << 1 : (((SL) + 1) & 3)) * ASLOT;          \
        const uint4* nfb_ = fb + (((SL) + 1) & 3) * BSLOT;                                               \
        /* (written-out MFMAs: two wait states between the vector instructions above and an MFMA that reads their results) */ \
        if constexpr (BSA && NWM == 4) asm volatile("s_nop 1");                                          \
        __builtin_amdgcn_sched_barrier(0);                                                               \
        GG_ML8(0, FA_, FB_, NA_, NB_, SL, Z_, EVEN_, SET_); GG_ML8(8, FA_, FB_, NA_, NB_, SL, Z_, EVEN_, SET_);   \
        GG_ML8(16, FA_, FB_, NA_, NB_, SL, Z_, EVEN_, SET_); GG_ML8(24, FA_, FB_, NA_, NB_, SL, Z_, EVEN_, SET_); \
        GG_ML8(32, FA_, FB_, NA_, NB_, SL, Z_, EVEN_, SET_); GG_ML8(40, FA_, FB_, NA_, NB_, SL, Z_, EVEN_, SET_); \
        GG_ML8(48, FA_, FB_, NA_, NB_, SL, Z_, EVEN_, SET_); GG_ML8(56, FA_, FB_, NA_, NB_, SL, Z_, EVEN_, SET_); \
        /* an odd block ends a pair: the next pair's scale dwords, from the other copy, behind its last MFMA */ \
        if constexpr (!(EVEN_)) GG_SC_READ(1 - SET_);                                                    \
        if (!(last) || seam) { /* (the last block hands over too when the next tile's stages are behind it) */ \
            gg_wait<WIDE ? ((EVEN_) ? 2 * RB : RB + LA) : 2 * LPS, 0>();                                 \
            __builtin_amdgcn_s_barrier();                                                                \
        }                                                                                                \
        if constexpr (TRACE) {                                                                           \
            if (blockIdx.x == 0 && threadIdx.x == 0 && tr_blk < GG_TRACE_BLOCK_WORDS)                    \
                p.trace[(size_t)gridDim.x * GG_TRACE_TILE_WORDS + tr_blk] = wall_clock64();              \
            ++tr_blk;                                                                                    \
        }                                                                                                \
    } while (0)
        GG_TRACE_TILE();
        int kbase = 0, nks_ld = nks;  // the loads of block s fetch stage s + 4 - kbase of the tile (Ab, Bb, a_off) point to
        bool seam = false;            // ... which is the next tile from block nks - 4 on
        {
            if (!pre) {
                // the four stages of this tile were requested before the previous tile's epilogue (or above, for
                // the first tile); the epilogue's stores sit behind them in the same counter, so wait for
                // everything
                gg_wait<0, 15>();
                __syncthreads();
            }
            if (p.a_map) {
                // the input rows of the NEXT tile, one per thread, straight into LDS: the switch to the next tile inside
                // this tile's K loop then reads them from there instead of waiting for memory
                const GgTile pk = gg_peek<DW>(s_tiles, g_row_start, nk, my, (int)gridDim.x, round, round0);
                if (pk.rv > 0 && wave_s * WAVE < BM) {
                    const int tid_a = wave_s * WAVE + gg_lane_now();
                    gg_dma4(gg_uniform((const uint8_t*)(p.a_map + pk.row0)), (uint32_t)min(tid_a, pk.rv - 1) * 4u,
                            __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)(s_amap + wave_s * WAVE)));
                }
            }
            {
                // What the epilogue needs from global memory per tile row / column (fp8 scales, the output row map) is
                // requested here, straight into LDS, one value per thread (into the copy the previous tile does not
                // use): the loads land during the first K stages (they are older than every load the K loop waits
                // for), and no epilogue waits for a memory round trip.  No register holds anything across the K loop.
                const int lane_t = gg_lane_now(), tid_t = wave_s * WAVE + lane_t;  // (a fresh lane id: nothing kept live for this)
                const uint32_t t4 = (uint32_t)min(tid_t, rv - 1) * 4u;
                if (wave_s * WAVE < BM) {
                    if ((FP8 || EPI == EPI_GATE) && (!BSA || p.row_scale))  // (BSA: the rows carry no scale of their own; a gate, if any)
                        gg_dma4(gg_uniform((const uint8_t*)(p.row_scale + row0)), t4,
                                __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)(s_row_scale[tpar] + wave_s * WAVE)));
                    if (p.c_map)
                        gg_dma4(gg_uniform((const uint8_t*)(p.c_map + row0)), t4,
                                __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)(s_crow[tpar] + wave_s * WAVE)));
                }
                if (FP8 && wave_s * WAVE < BN) {
                    const int pc = gg_packed_col<true>(nt * BN + tid_t);  // packed column of the launch behind this row of the weight tile; the lanes 32..63 of a wave hold up columns
                    int col = EPI == EPI_SWIGLU ? (pc / 64) * 32 + pc % 32 : pc;
                    col = col < p.N ? col : 0;  // (columns past N are never stored: any valid scale will do)
                    const uint32_t lds_cs = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)(s_col_scale[tpar] + wave_s * WAVE));
                    const uint32_t c4 = (uint32_t)col * 4u;
                    if (EPI == EPI_SWIGLU && lane_t >= 32) gg_dma4(gg_uniform((const uint8_t*)(p.col_scale2 + (size_t)g * p.ncs)), c4, lds_cs);
                    else gg_dma4(gg_uniform((const uint8_t*)(p.col_scale + (size_t)g * p.ncs)), c4, lds_cs);
                }
            }
            if (!pre) {
                const uint4* fa0 = fa + phi * ASLOT;
                const uint4* fb0 = fb + phi * BSLOT;
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    if constexpr (DW) {
                        const uint2 lo = gg_read_tr<512>(GG_TR_A(i, phi), 0), hi = gg_read_tr<512>(GG_TR_A(i, phi), 1);
                        fA0[i] = make_uint4(lo.x, lo.y, hi.x, hi.y);
                    } else {
#pragma unroll
                        for (int h = 0; h < CF; ++h) fA0[i * CF + h] = fa0[i * MT * 2 * CHUNKS + (fpos_a ^ (h * FSTEP))];
                    }
                }
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    if constexpr (DW || BN_RAW) {
                        const uint2 lo = gg_read_tr<BTR>(GG_TR_B(j, phi), 0), hi = gg_read_tr<BTR>(GG_TR_B(j, phi), 1);
                        fB0[j] = make_uint4(lo.x, lo.y, hi.x, hi.y);
                    } else {
#pragma unroll
                        for (int h = 0; h < CF; ++h) fB0[j * CF + h] = fb0[j * MT * CHUNKS + (fpos ^ (h * FSTEP))];
                    }
                }
                GG_SC_READ(0);  // (a tile that starts here starts in slot 0)
                // the first slot is refilled from the first block on: every wave must hold its stage-0 fragments first
                gg_wait<63, 0>();
                __syncthreads();
            }
            // The blocks are written out for the slots 0 .. 3; a tile whose first stage lies in slot 2 (phi = 2: the
            // tiles before it left the ring there) enters at the third.  nk >= 2 and even.
            if constexpr (PEEL) {
                // The tile's first two blocks are written out apart, with the slot as a run-time value: the MFMAs of the
                // very first start the sums (constant zero as their C operand), so that no accumulator has to be cleared
                // between two tiles.  (Not where the stage count varies from tile to tile: the register allocation of
                // those instantiations does not survive it.)
                const int phi_s = __builtin_amdgcn_readfirstlane(phi);
                GG_STAGE(fA0, fB0, fA1, fB1, phi_s, true, 0, false, true, 0);
                GG_STAGE(fA1, fB1, fA0, fB0, phi_s + 1, false, 1, 2 >= nks, false, 0);
                int ks = phi_s ? 2 : 0;             // phi = 0: on with the slots 2, 3 (the first half of the loop body is
                const int kmin = phi_s ? 2 : 4;     // skipped once); phi = 2: with the slots 0, 1
                while (ks < nks) {
                    if (ks >= kmin) {
                        GG_STAGE(fA0, fB0, fA1, fB1, 0, true, ks, false, false, 0);
                        GG_STAGE(fA1, fB1, fA0, fB0, 1, false, ks + 1, ks + 2 >= nks, false, 0);
                    }
                    if (ks + 2 < nks) {
                        GG_STAGE(fA0, fB0, fA1, fB1, 2, true, ks + 2, false, false, 1);
                        GG_STAGE(fA1, fB1, fA0, fB0, 3, false, ks + 3, ks + 4 >= nks, false, 1);
                    }
                    ks += 4;
                }
            } else {
                int ks = -phi;
                do {
                    if (ks >= 0) {
                        GG_STAGE(fA0, fB0, fA1, fB1, 0, true, ks, false, false, 0);
                        GG_STAGE(fA1, fB1, fA0, fB0, 1, false, ks + 1, ks + 2 >= nks, false, 0);
                    }
                    if (ks + 2 < nks) {
                        GG_STAGE(fA0, fB0, fA1, fB1, 2, true, ks + 2, false, false, 1);
                        GG_STAGE(fA1, fB1, fA0, fB0, 3, false, ks + 3, ks + 4 >= nks, false, 1);
                    }
                    ks += 4;
                } while (ks < nks);
            }
        }
#undef GG_STAGE
#undef GG_ML8
#undef GG_ML
#undef GG_RD

        if constexpr (BSA && NWM == 4) {
            // the last MFMAs of the tile were written out as asm (see mma_fp8_k64_bs): the wait states the compiler would put
            // between an MFMA and the first read of its result by another kind of instruction (18 for this shape)
            asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
        }
        // ---- next tile: decode it and request its first stages now (every slot is free once all waves
        // have passed the barrier: the last fragments of this tile are already in registers)
        // (when the K loop has switched over, the walk only confirms what the look-ahead saw)
        GG_TRACE_TILE();
        const GgTile nxt = gg_walk<BM, DW>(s_tiles, g_tile_start, g_row_start, p.E_l, Nt, p.S_rows, n_tiles, nk, my, (int)gridDim.x, round, round0, p.dw_rows);
        if (!seam && nxt.rv > 0) {
            GG_TILE_PTRS(nxt, Ab_n, Bb_n, a_off_n, GG_MAPROW_GLOBAL);
            Ab = Ab_n;
            Bb = Bb_n;
#pragma unroll
            for (int r = 0; r < LA; ++r) a_off[r] = a_off_n[r];
            sc_row0 = nxt.row0; sc_rv = nxt.rv; sc_ks0 = nxt.ks0;
            __syncthreads();
            GG_PROLOGUE(Ab, Bb, a_off, (VARK ? nxt.nks : nk));
        }
        const int phi_n = seam ? ((phi + nks) & 3) : 0;

        // ---- epilogue: acc -> (scales) -> activation -> bf16 -> C
        // acc(i,j) holds the TRANSPOSED MT x MT product (weights as the MFMA A operand, activations as B):
        // a lane owns one token row of the tile and runs of four consecutive rows of the weight tile
        //   bf16 (16x16): token row l % 16, weight rows 4 * (l / 16) + v, v = 0..3
        //   fp8  (32x32): token row l % 32, weight rows 8 * q + 4 * (l / 32) + v for the four register quads q
        // and the rows of a group of 32 packed columns are ordered (gg_col_to_row32) so that two of those runs are
        // eight consecutive output columns -> 16-byte stores.
        // SwiGLU: packed columns alternate gate / up in groups of 32, so a gate group and its up group lie
        // 32 packed columns apart and land on output column (packed column of the gate group) / 2 + ... .
        bf16_t* C = (bf16_t*)p.C;
        constexpr int GT = 32 / MT;                  // MFMA tiles per group of 32 packed columns
        constexpr int NG = TN / GT;                  // groups per wave (its 128 packed columns)
        constexpr int NU = FP8 ? 2 : 1;              // 16-byte stores per lane and group
        // (the lane-derived constants of the epilogue are derived here, once per tile, from a fresh read of the lane id)
        const int lane_e = gg_lane_now(), rbase_e = (wave_s >> 1) * (BM / NWM), cbase_e = (wave_s & 1) * (BN / 2);
        const int lsub = FP8 ? (lane_e >> 5) : (lane_e >> 4);  // which of the lanes that share a tile row this one is
        // What the tile's top requested into LDS (scales, row map) is behind two block ends of the K loop at least -- the
        // second one has waited for it in every wave -- unless the tile has only two stages:
        if (nks < 4 && (FP8 || EPI == EPI_GATE || p.c_map)) {
            gg_wait<0, 15>();
            __syncthreads();
        }
        // fp8 with bf16 output: a lane stores to TWO rows of a row tile (its accumulators change lanes first, below);
        // bf16, and fp8 with quantised output: to its own
        constexpr int NR = (FP8 && !QOUT) ? 2 : 1;
        bool ok[TM][NR];
        bf16_t* crow[TM][NR];
        float rs[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            rs[i] = 1.f;
            if constexpr (FP8 || EPI == EPI_GATE) {
                if (!BSA || p.row_scale) rs[i] = s_row_scale[tpar][rbase_e + i * MT + (lane_e & (MT - 1))];  // (of the row it computed)
            }
#pragma unroll
            for (int h = 0; h < NR; ++h) {
                const int r = rbase_e + i * MT + ((FP8 && !QOUT) ? (lane_e & 15) + 16 * h : (lane_e & (MT - 1)));
                ok[i][h] = r < rv && !(TRACE && (p.trace_flags & 1));
                const size_t grow = (size_t)(row0 + (ok[i][h] ? r : 0));
                const int crow_i = p.c_map ? s_crow[tpar][r] : 0;
                ok[i][h] = ok[i][h] && crow_i >= 0;  // a negative map entry: the row has no place in the output
                // (quantised output: C holds one-byte codes, addressed below from the same row index)
                crow[i][h] = C + (p.c_map ? (size_t)max(crow_i, 0) : grow) * (QOUT ? (size_t)1 : (size_t)p.ldc) + (DW ? (size_t)g * p.c_group_stride : (size_t)0);
            }
        }
#pragma unroll
        for (int o = 0; o < TM * NG; ++o) {
            // fp8: column groups outermost; bf16: row tiles outermost, so that the stores of one row tile fill whole
            // cache lines back to back (the other order wrote 50 % more bytes to memory: lines left the L2
            // half written)
            const int i = FP8 ? o % TM : o / NG, jg = FP8 ? o / TM : o % NG;
            if constexpr (EPI == EPI_SWIGLU) {
                if (jg % 2 == 1) continue;  // an up group: consumed together with its gate group
            }
            const int pcol = nt * BN + cbase_e + jg * 32;  // first packed column of the group
            const bool pair = EPI == EPI_SWIGLU || (DW && p.dw_split);
            const int colg = pair ? (pcol / 64) * 32 : pcol;  // its first output column
            [[maybe_unused]] const long long cshift = DW && p.dw_split && (pcol & 32) ? p.dw_delta : 0;
            [[maybe_unused]] uint4 pk[2];  // fp8: the lane's two 16-byte units of the group, stored after they changed lanes
            [[maybe_unused]] float xq[2][8];  // quantised output: the lane's sixteen values of the group's block of 32 columns
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                // the lane's eight consecutive columns: two runs of four accumulators (bf16: the group's two tiles;
                // fp8: the register quads 2u and 2u + 1 of the group's one tile)
                const int col = colg + (FP8 ? 16 * u : 0) + 8 * lsub;
                float x[8];
                [[maybe_unused]] float pre_g[8], pre_u[8];  // bf16 kernels asked to keep them: the values before the activation
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int j = FP8 ? jg : jg * GT + t;       // MFMA tile of the run
                    const int qd = FP8 ? 2 * u + t : 0;         // its register quad
                    const int ju = j + GT;                      // SwiGLU: the up tile (32 packed columns further)
                    float cg[4] = {1.f, 1.f, 1.f, 1.f}, cu[4] = {1.f, 1.f, 1.f, 1.f};
                    if constexpr (FP8) {
                        // channel scales by row of the weight tile (an LDS read: cheap enough to repeat for every row tile)
                        const int tc = cbase_e + j * MT + 8 * qd + 4 * lsub;
                        const float4 s0 = *(const float4*)(s_col_scale[tpar] + tc);
                        cg[0] = s0.x; cg[1] = s0.y; cg[2] = s0.z; cg[3] = s0.w;
                        if constexpr (EPI == EPI_SWIGLU) {
                            const float4 s1 = *(const float4*)(s_col_scale[tpar] + tc + 32);
                            cu[0] = s1.x; cu[1] = s1.y; cu[2] = s1.z; cu[3] = s1.w;
                        }
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float v = acc[i][j][4 * qd + e];
                        if constexpr (FP8) v *= cg[e] * rs[i];
                        if constexpr (!FP8 && EPI == EPI_GATE) v *= rs[i];
                        if constexpr (!FP8 && EPI != EPI_NONE && EPI != EPI_GATE) pre_g[4 * t + e] = v;
                        if constexpr (EPI == EPI_SWIGLU) {
                            float uv = acc[i][ju % TN][4 * qd + e];
                            if constexpr (FP8) uv *= cu[e] * rs[i];
                            if constexpr (!FP8) pre_u[4 * t + e] = uv;
                            v = act_silu_fast(v) * uv;
                        }
                        if constexpr (EPI == EPI_GELU) v = act_gelu(v);
                        if constexpr (EPI == EPI_SILU) v = act_silu_fast(v);
                        x[4 * t + e] = v;
                    }
                }
                if constexpr (QOUT) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) xq[u][e] = x[e];
                    continue;
                }
                uint4 o4;
                o4.x = gg_pack_bf16(x[0], x[1]);
                o4.y = gg_pack_bf16(x[2], x[3]);
                o4.z = gg_pack_bf16(x[4], x[5]);
                o4.w = gg_pack_bf16(x[6], x[7]);
                if constexpr (FP8) {
                    pk[u] = o4;
                } else if (ok[i][0] && col + (pair && DW ? pcol - colg : 0) < p.N) {
                    *(uint4*)(crow[i][0] + col + (DW ? cshift : 0)) = o4;
                    if constexpr (EPI != EPI_NONE && EPI != EPI_GATE) {
                        if (p.C2) {
                            // same row, in a matrix whose rows are as long (SwiGLU: twice as long, packed column order)
                            constexpr int W2 = EPI == EPI_SWIGLU ? 2 : 1;
                            bf16_t* r2 = (bf16_t*)p.C2 + (size_t)(crow[i][0] - C) * W2 + (EPI == EPI_SWIGLU ? pcol + 8 * lsub : col);
                            uint4 g4;
                            g4.x = gg_pack_bf16(pre_g[0], pre_g[1]); g4.y = gg_pack_bf16(pre_g[2], pre_g[3]);
                            g4.z = gg_pack_bf16(pre_g[4], pre_g[5]); g4.w = gg_pack_bf16(pre_g[6], pre_g[7]);
                            *(uint4*)r2 = g4;
                            if constexpr (EPI == EPI_SWIGLU) {
                                uint4 u4;
                                u4.x = gg_pack_bf16(pre_u[0], pre_u[1]); u4.y = gg_pack_bf16(pre_u[2], pre_u[3]);
                                u4.z = gg_pack_bf16(pre_u[4], pre_u[5]); u4.w = gg_pack_bf16(pre_u[6], pre_u[7]);
                                *(uint4*)(r2 + 32) = u4;
                            }
                        }
                    }
                }
            }
            if constexpr (QOUT) {
                // The group is one block of 32 output columns of the hidden activation: the lane holds 16 of its values
                // (columns 8 lsub .. + 7 and 16 + 8 lsub .. + 7), the lane 32 further the other 16.  Block scale = the
                // smallest power of two under which the block's largest magnitude fits e4m3; codes = the values divided by
                // it (exact), rounded to e4m3; the two lanes trade a run of 8 codes each, so that each stores 16 contiguous
                // bytes of its row; one lane of the pair stores the scale byte.
                float am = 0.f;
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int e = 0; e < 8; ++e) am = fmaxf(am, fabsf(xq[u][e]));
                {
                    const auto sw_ = __builtin_amdgcn_permlane32_swap(__float_as_uint(am), __float_as_uint(am), false, false);
                    am = fmaxf(__uint_as_float(sw_[0]), __uint_as_float(sw_[1]));
                }
                const int sbyte = gg_block_scale_byte(__float_as_uint(am));
                const float inv = __uint_as_float(gg_block_inv_bits(sbyte));
                uint32_t cd[2][2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    int lo = 0, hi = 0;
                    lo = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(xq[u][0], inv), __fmul_rn(xq[u][1], inv), lo, false);
                    lo = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(xq[u][2], inv), __fmul_rn(xq[u][3], inv), lo, true);
                    hi = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(xq[u][4], inv), __fmul_rn(xq[u][5], inv), hi, false);
                    hi = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(xq[u][6], inv), __fmul_rn(xq[u][7], inv), hi, true);
                    cd[u][0] = (uint32_t)lo;
                    cd[u][1] = (uint32_t)hi;
                }
                // lanes 0-31 keep their first run and take the partner's first run (columns 0-15 of the block), lanes 32-63
                // take the partner's second run and keep their own (columns 16-31)
                const auto s0_ = __builtin_amdgcn_permlane32_swap(cd[0][0], cd[1][0], false, false);
                const auto s1_ = __builtin_amdgcn_permlane32_swap(cd[0][1], cd[1][1], false, false);
                const uint4 codes = make_uint4(s0_[0], s1_[0], s0_[1], s1_[1]);
                const int col = colg + 16 * lsub;
                if (ok[i][0] && col < p.N) {
                    uint8_t* qrow = (uint8_t*)p.C + (size_t)(crow[i][0] - C) * p.ldc;
                    *(uint4*)(qrow + col) = codes;
                    if (lsub == 0) p.c_bscale[(size_t)(crow[i][0] - C) * p.bs_pitch + colg / 32] = (uint8_t)sbyte;
                }
            } else if constexpr (FP8) {
                // A lane holds 16 bytes of each half of its row's 64 (columns 8 lsub .. and 16 + 8 lsub ..) and the lane 16
                // further the same of the row 16 further.  They trade one half each (v_permlane16_swap: lanes 16-31 and
                // 48-63 of the first operand against lanes 0-15 and 32-47 of the second), after which the first operand
                // holds whole 64-byte segments of rows 0-15 of the row tile and the second those of rows 16-31: a store
                // instruction then covers 16 rows instead of 32 -- the store path's cost follows the number of row
                // segments per instruction, not the bytes.
#define GG_SWAP16(a_, b_)                                                          \
    do {                                                                           \
        const auto sw_ = __builtin_amdgcn_permlane16_swap((a_), (b_), false, false); \
        (a_) = sw_[0];                                                             \
        (b_) = sw_[1];                                                             \
    } while (0)
                GG_SWAP16(pk[0].x, pk[1].x);
                GG_SWAP16(pk[0].y, pk[1].y);
                GG_SWAP16(pk[0].z, pk[1].z);
                GG_SWAP16(pk[0].w, pk[1].w);
#undef GG_SWAP16
                const int col = colg + 16 * ((lane_e >> 4) & 1) + 8 * lsub;
                if (col < p.N) {
                    if (ok[i][0]) *(uint4*)(crow[i][0] + col) = pk[0];
                    if (ok[i][NR - 1]) *(uint4*)(crow[i][NR - 1] + col) = pk[1];
                }
            }
            // keep the accumulator read-out of one group from being hoisted over the previous group's stores
            // (that would need every accumulator in a VGPR at once)
            __builtin_amdgcn_sched_barrier(0);
        }
        GG_TRACE_TILE();
        cur = nxt;
        pre = seam;
        phi = phi_n;
        tpar ^= 1;
    }
#undef GG_TRACE_TILE
#undef GG_TILE_PTRS
#undef GG_MAPROW_GLOBAL
#undef GG_MAPROW_LDS
#undef GG_LDA
#undef GG_LDB
#undef GG_A_PTR
#undef GG_B_PTRS
#undef GG_ISSUE_A
#undef GG_ISSUE_B
#undef GG_PROLOGUE
#undef GG_SC_DMA
#undef GG_SC_READ
#undef GG_TR_A
#undef GG_TR_B
}

// ---- one-time weight re-tiling: w [E_l,K,N] (N contiguous) -> out [E_l][K/SK][Npad][SK], SK = one LDS
// stage of K (ROWB bytes): the B tile of a stage is one contiguous 32 KB block -----------------------
// With w_up, gate and up columns are interleaved in groups of 32: packed col = (n/32)*64 + {0,32} + n%32.
template <typename T>
__global__ __launch_bounds__(256) void prepack_kernel(const T* __restrict__ w, const T* __restrict__ w_up, T* __restrict__ out,
                                                       int K, int N, int Npad) {
    __shared__ T tile[64][64 + 2];
    const int e = blockIdx.z;
    const int k0 = blockIdx.y * 64, n0 = blockIdx.x * 64;  // n0 in source columns
    const T* src = w + (size_t)e * K * N;
    const T* src2 = w_up ? w_up + (size_t)e * K * N : nullptr;
    T* dst = out + (size_t)e * Npad * K;
    constexpr int SK = ROWB / (int)sizeof(T);  // K elements per slab
    for (int pass = 0; pass < (src2 ? 2 : 1); ++pass) {
        const T* s = pass ? src2 : src;
        for (int i = threadIdx.x; i < 64 * 64; i += 256) {
            const int kk = i / 64, nn = i % 64;
            tile[kk][nn] = (k0 + kk < K && n0 + nn < N) ? s[(size_t)(k0 + kk) * N + n0 + nn] : (T)0;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < 64 * 64; i += 256) {
            const int nn = i / 64, kk = i % 64;
            const int n = n0 + nn;
            // (columns [N, next multiple of 64) leave as the zeros they were loaded as: the rows of a group of 32 are
            // permuted, so a partly filled group cannot be zeroed as a range of rows)
            const int np = src2 ? ((n >> 5) * 64 + pass * 32 + (n & 31)) : n;
            if ((n < N || (!src2 && np < Npad)) && k0 + kk < K) {
                const int k = k0 + kk;
                dst[((size_t)(k / SK) * Npad + gg_packed_row<sizeof(T) == 1>(np)) * SK + (k % SK)] = tile[kk][nn];
            }
        }
        __syncthreads();
    }
}

// The same for 16-bit weights with K a multiple of 64 and N of 8 (what the GEMMs take) at multiples of 16 bytes: 64 k x 128 n through LDS, 16 bytes per load
// and store.  Columns [N, Npad) leave as zeros.
__global__ __launch_bounds__(256) void prepack16_kernel(const uint16_t* __restrict__ w, const uint16_t* __restrict__ w_up,
                                                         uint16_t* __restrict__ out, int K, int N, int Npad) {
    constexpr int TN = 128, LD = TN + 8;
    __shared__ __align__(16) uint16_t tile[64][LD];
    const int passes = w_up ? 2 : 1, e = blockIdx.z / passes, pass = blockIdx.z % passes;
    const int k0 = blockIdx.y * 64, n0 = blockIdx.x * TN;
    const uint16_t* s = (pass ? w_up : w) + (size_t)e * K * N;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int v = threadIdx.x + i * 256, kk = v / 16, nn = (v % 16) * 8;
        uint4 x = make_uint4(0, 0, 0, 0);
        if (n0 + nn < N) x = *(const uint4*)(s + (size_t)(k0 + kk) * N + n0 + nn);
        *(uint4*)&tile[kk][nn] = x;
    }
    __syncthreads();
    constexpr int SK = 32;
    uint16_t* dst = out + (size_t)e * Npad * K;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int v = threadIdx.x + i * 256, k8 = (v % 4) * 8, row = v / 4;  // row: (slab of the tile, row of the packed columns)
        const int slab = row / TN, rr = row % TN;
        const int nn = gg_packed_col<false>(rr);  // (consecutive threads write consecutive packed rows)
        const int pr = w_up ? ((n0 + rr) >> 5) * 64 + pass * 32 + (rr & 31) : n0 + rr;
        if (pr >= Npad) continue;
        uint32_t o[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = (uint32_t)tile[slab * SK + k8 + 2 * q][nn] | ((uint32_t)tile[slab * SK + k8 + 2 * q + 1][nn] << 16);
        *(uint4*)(dst + ((size_t)(k0 / SK + slab) * Npad + pr) * SK + k8) = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

template <typename T>
__global__ void zero_pad_rows_kernel(T* __restrict__ out, int K, int Nreal, int Npad) {
    // rows [Nreal, Npad) of every K slab of every expert's packed matrix (Nreal a multiple of 32: whole groups)
    constexpr int SK = ROWB / (int)sizeof(T);
    const int e = blockIdx.y;
    const size_t per_slab = (size_t)(Npad - Nreal) * SK;
    const size_t n = per_slab * (size_t)(K / SK);
    T* dst = out + (size_t)e * Npad * K;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const size_t slab = i / per_slab, r = i % per_slab;
        dst[(slab * Npad + Nreal) * SK + r] = (T)0;
    }
}

// fp32 grouped GEMM (the plumbing workload's experts, and the fp32 gradients to rows): tiles of 32R x 32R rows and columns, four waves
// of 16R x 16R each, on the fp32 matrix instruction (16x16x4; products and sums of one k after the other).  Weights in the reference layout [E_l][K][N].
// A sum is one chain over ascending k, the order of a scalar fmaf chain, with KG = 1; with KG = 2 two such chains, over the even and the odd pieces of
// 128 of K, added once.  Which of the two a launch takes depends on its rows, groups and columns (f32_plan): the same row may differ
// by rounding between launches of different sizes.
// Bound at the plumbing sizes (487 rows, K 256 / 512) by the length of its chain: load, LDS, matrix instructions, slab by slab, with few
// workgroups in flight; hence the long slabs (R = 1: 128 of K, twice the loads under way) and small tiles (256 workgroups of
// 32 x 32 where 64 x 64 gives 64).  KG = 2, where the tiles are one round: eight waves to a tile, slabs twice as long, every set of four with half of
// a slab's steps and the second half's sums added at the end: the two GEMMs of the plumbing step 8.0 and 12.4 us with one set, 7.4 and 8.7 with two
// (fastest launches; on the vector units with 64 x 64 tiles they took 32 and 56).  What of the chain need not wait does not: the weights' first slab is asked for
// before the rows' places are known, the second slab (R = 1) with the first, and the sources' counts beside the counts per expert.  A plumbing step
// 33.6 -> 31.1 us; rows x K x N of a group: 256 x 1024 x 256 13.0 -> 11.9, 1000 x 516 x 500 of four 15.9 -> 14.2, 4096 x 256 x 512 of eight 24.8 -> 19.6, 4096 x 512 x 1024
// (R = 2, whose loads no longer jump either) 55 -> 50.
// R = 2 for launches of many tiles: every operand value out of LDS feeds two matrix instructions.
// A in LDS as [row][k % 4][k / 4]: the four values a lane needs in four consecutive steps are one 16-byte read; B as
// [k][column], rows padded so that the four k of a step lie in different banks.
// SIDE: the copy of the rows beside the GEMM.  F32_RETURN: result rows go to their slots of the returned [W,M,N] buffer as well, and the
// workgroups from side.tiles_y on zero its padding rows.  F32_UNPACK: the rows come from their slots of the received [W,M,K] buffer, and the workgroups
// of the first columns leave them in expert-major order in side.rows (zeros for rows past the pair capacity, and past the total), and the counts
// per expert in side.cnt.  As launches of their own the two copies took 2.5 and 3 us of the 43 of the plumbing step.  A tile's rows belong to one
// expert, whose slots start at the sums of the received counts before it.
enum { F32_ROWS = 0, F32_RETURN = 1, F32_UNPACK = 2 };
struct F32Side {
    const int32_t* rc;  // received counts [W,E_l]
    int W, M;
    float* buf;         // [W,M,...]: written (F32_RETURN) or read
    int tiles_y;
    float* rows;
    int32_t* cnt;
};
template <int EPI, int R, int KG, int SIDE, bool VEC /* K, N and the bases allow 16-byte loads */>
__global__ __launch_bounds__(256 * KG) void grouped_gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ Wt,
                                                                const float* __restrict__ Wup, float* __restrict__ C,
                                                                const int32_t* __restrict__ cnt, int E_l, int K, int N,
                                                                int S_rows, const F32Side side) {
    // PT: 16-byte units of each operand per thread and slab
    constexpr int TM = 32 * R, KC = 128 / R * KG, NTH = 256 * KG, PT = TM * KC / 4 / NTH, STEPS = KC / 16 / KG;
    constexpr int PA = KC + 4, PB = TM + 16;
    constexpr bool UP = EPI == EPI_SWIGLU;
    constexpr int D = R == 1 && VEC ? 2 : 1;  // slabs under way (many tiles cover each other's loads)
    extern __shared__ __align__(16) float slab[];
    float *const As = slab, *const Bs = As + TM * PA, *const Us = Bs + KC * PB;
    __shared__ int s_g, s_row0, s_rv, s_first;
    constexpr bool RET = SIDE == F32_RETURN, SRC = SIDE == F32_UNPACK;
    __shared__ int32_t s_from[SIDE ? MOE_MAX_EXPERTS : 1], s_slot[SIDE ? MOE_MAX_EXPERTS : 1], s_at[SIDE ? TM : 1];
    __shared__ int32_t s_rc[SIDE ? MOE_MAX_EXPERTS : 1], s_cnt[SRC ? MOE_MAX_EXPERTS : 1];
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    if constexpr (RET) {
        if ((int)blockIdx.y >= side.tiles_y) {  // padding rows: a wave's share of all slots, slot by slot
            const int waves = (gridDim.y - side.tiles_y) * gridDim.x * (NTH / WAVE);
            const int w0 = ((blockIdx.y - side.tiles_y) * gridDim.x + blockIdx.x) * (NTH / WAVE) + wave;
            for (int sr = 0; sr < side.W; ++sr) {
                int rows = 0;
                for (int e = lane; e < E_l; e += WAVE) rows += side.rc[sr * E_l + e];
                rows = max(wave_sum(rows), 0);
                for (int m = rows + w0; m < side.M; m += waves)
                    for (int c = lane; c < N; c += WAVE) side.buf[((size_t)sr * side.M + m) * N + c] = 0.f;
            }
            return;
        }
        if (wave > 0)  // (while the first wave reads the counts)
            for (int i = threadIdx.x - WAVE; i < side.W * E_l; i += NTH - WAVE) s_rc[i] = side.rc[i];
    }
    if constexpr (SRC) {
        for (int i = threadIdx.x; i < side.W * E_l; i += NTH) s_rc[i] = side.rc[i];
        __syncthreads();
        for (int e = threadIdx.x; e < E_l; e += NTH) {
            int c = 0;
            for (int sr = 0; sr < side.W; ++sr) c += s_rc[sr * E_l + e];
            s_cnt[e] = c;
            if (blockIdx.x + blockIdx.y == 0) side.cnt[e] = c;
        }
        __syncthreads();
    }
    const int32_t* const counts = SRC ? s_cnt : cnt;
    if (wave == 0) {  // which expert's rows: 64 experts at a time, tiles and rows before them by a scan
        int mt = blockIdx.y, rs = 0;
        bool found = false;
        if (lane == 0) s_g = -1;
        for (int base = 0; base < E_l; base += WAVE) {
            const GgRows r = gg_rows<true>(counts, base + lane, E_l, rs, S_rows);
            const int t = (r.n + TM - 1) / TM;
            const int tiles = wave_incl_scan(t);
            const bool mine = mt < tiles && mt >= tiles - t;
            if (mine) {
                const int first = (mt - (tiles - t)) * TM;
                s_g = base + lane; s_row0 = r.start + first; s_rv = min(TM, r.n - first); s_first = first;
            }
            if (__ballot(mine)) { found = true; break; }
            mt -= wave_lane(tiles, WAVE - 1);
            rs = r.end;
        }
        // (the workgroups behind the tiles are as many as the rows behind the total, and more)
        if (SRC && lane == 0 && !found) { s_row0 = rs + mt * TM; s_rv = min(TM, S_rows - s_row0); }
    }
    __syncthreads();
    const int g = s_g;
    if (SRC && g < 0 && blockIdx.x == 0)
        for (int i = threadIdx.x; i < s_rv * K; i += NTH) side.rows[(size_t)s_row0 * K + i] = 0.f;
    if (g < 0 || s_rv <= 0) return;
    const int row0 = s_row0, rv = s_rv, n0 = blockIdx.x * TM;
    const float* W = Wt + (size_t)g * K * N;
    const float* U = UP ? Wup + (size_t)g * K * N : nullptr;
    auto handover = [] {  // what went to LDS is there; loads stay under way
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto place = [&](int i) {  // row i of the tile: its slot
        const int r = s_first + i;  // of the expert's rows
        int lo = 0, hi = side.W;    // (the last of a run of equal starts owns the row)
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (s_from[mid] <= r) lo = mid; else hi = mid;
        }
        const int m = s_slot[lo] + r - s_from[lo];
        s_at[i] = (unsigned)m < (unsigned)side.M ? lo * side.M + m : -1;  // (past the pair capacity: the row has no slot)
    };
    // where the rows of every source start among the expert's, and among the slots (the first wave)
    auto sources = [&] {
        int run = 0;
        for (int base = 0; base < side.W; base += WAVE) {
            const int sr = base + lane;
            int mine = 0, before = 0;
            if (sr < side.W) {
                mine = s_rc[sr * E_l + g];
#pragma unroll 8
                for (int e = 0; e < g; ++e) before += s_rc[sr * E_l + e];
            }
            const int incl = wave_incl_scan(mine);
            if (sr < side.W) { s_from[sr] = run + incl - mine; s_slot[sr] = before; }
            run += wave_lane(incl, WAVE - 1);
        }
    };
    // Nothing jumps over a 16-byte load: addresses are clamped into the operand, and what lies outside it becomes zero on the way to LDS -- so that the wait
    // for one slab's loads can leave the next one's under way (D sets of registers).
    static_assert(NTH % (KC / 4) == 0 && NTH % (TM / 4) == 0, "a thread's units lie below one another");
    const int ka = threadIdx.x % (KC / 4) * 4, ra0 = threadIdx.x / (KC / 4);            // A: consecutive threads walk K; units NTH / (KC / 4) rows apart
    const int nb = n0 + threadIdx.x % (TM / 4) * 4, kb0 = threadIdx.x / (TM / 4);       // W: consecutive threads walk N; units NTH / (TM / 4) of K apart
    float4 ra[D][PT], rb[D][PT], ru[D][UP ? PT : 1];
    const float* arow[PT];
    bool aok[PT];
    auto load = [&](const float* p, int at, int end, [[maybe_unused]] bool ok) {  // (ok: the row exists)
        if constexpr (VEC) return *reinterpret_cast<const float4*>(p + (at < end ? at : 0));  // (a unit lies wholly inside or outside)
        else {  // (value by value, and jumped over: the clamped addresses are more work than the jumps, 2000 x 130 x 131 10.0 us against 9.3)
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            end = ok ? end : 0;
            if (at < end) v.x = p[at];
            if (at + 1 < end) v.y = p[at + 1];
            if (at + 2 < end) v.z = p[at + 2];
            if (at + 3 < end) v.w = p[at + 3];
            return v;
        }
    };
    auto inside = [](const float4& v, bool ok) { return VEC && !ok ? make_float4(0.f, 0.f, 0.f, 0.f) : v; };
    auto fetch_w = [&](auto d_c, int k0) {
        constexpr int d = decltype(d_c)::value;
#pragma unroll
        for (int q = 0; q < PT; ++q) {
            const int kb = k0 + kb0 + q * (NTH / (TM / 4));
            const size_t row = (size_t)min(kb, K - 1) * N;
            rb[d][q] = load(W + row, nb, N, kb < K);
            if constexpr (UP) ru[d][q] = load(U + row, nb, N, kb < K);
        }
    };
    auto fetch_a = [&](auto d_c, int k0) {
        constexpr int d = decltype(d_c)::value;
#pragma unroll
        for (int q = 0; q < PT; ++q) ra[d][q] = load(arow[q], k0 + ka, K, aok[q]);
    };
    typedef std::integral_constant<int, 0> set0;
    typedef std::integral_constant<int, D - 1> set1;
    fetch_w(set0{}, 0);
    if constexpr (SRC) {
        if (wave == 0) sources();
        handover();
        if ((int)threadIdx.x < rv) place(threadIdx.x);
        handover();
    }
#pragma unroll
    for (int q = 0; q < PT; ++q) {
        const int r = ra0 + q * (NTH / (KC / 4)), at = SRC ? s_at[min(r, rv - 1)] : row0 + min(r, rv - 1);
        aok[q] = r < rv && at >= 0;
        arow[q] = (SRC ? side.buf : A) + (size_t)max(at, 0) * K;
    }
    fetch_a(set0{}, 0);
    if constexpr (D == 2) {
        fetch_w(set1{}, KC);
        fetch_a(set1{}, KC);
    }
    if constexpr (RET)
        if (wave == 0) sources();
    const int half = wave / 4;  // which steps of a slab are this wave's
    const int wm = (wave / 2 % 2) * 16 * R, wn = (wave % 2) * 16 * R, l16 = lane % 16, kg = lane / 16;
    floatx4 acc[R][R] = {}, acu[UP ? R : 1][R] = {};
    typedef std::integral_constant<bool, true> more;
    typedef std::integral_constant<bool, false> last;
    auto slab_pass = [&](auto d_c, auto more_c, int k0) {
        constexpr int d = decltype(d_c)::value;
#pragma unroll
        for (int q = 0; q < PT; ++q) {
            const int r = ra0 + q * (NTH / (KC / 4)), kb = kb0 + q * (NTH / (TM / 4));
            const float4 va = inside(ra[d][q], aok[q] && k0 + ka < K);
            if constexpr (SRC) {  // (rows are multiples of 16 bytes)
                if (blockIdx.x == 0 && r < rv && k0 + ka < K) *reinterpret_cast<float4*>(side.rows + (size_t)(row0 + r) * K + k0 + ka) = va;
            }
            float* a = As + r * PA + ka / 4;
            a[0] = va.x; a[KC / 4] = va.y; a[2 * (KC / 4)] = va.z; a[3 * (KC / 4)] = va.w;
            const int b = kb * PB + nb - n0;
            const bool wok = k0 + kb < K && nb < N;
            *reinterpret_cast<float4*>(Bs + b) = inside(rb[d][q], wok);
            if constexpr (UP) *reinterpret_cast<float4*>(Us + b) = inside(ru[d][q], wok);
        }
        handover();
        if (D == 1 ? k0 + KC < K : decltype(more_c)::value) {
            fetch_w(d_c, k0 + D * KC);
            fetch_a(d_c, k0 + D * KC);
        }
        if constexpr (RET)
            if (k0 == 0 && (int)threadIdx.x < rv) place(threadIdx.x);  // (read behind the barrier below)
        // slab positions past K hold zeros: adding +0 products leaves every sum as it is
        const int steps = min(KC, K - k0 + 15) / 16 - half * STEPS;
        auto step = [&](int s4) {
            floatx4 a[R];
#pragma unroll
            for (int i = 0; i < R; ++i) a[i] = *reinterpret_cast<const floatx4*>(As + (wm + 16 * i + l16) * PA + kg * (KC / 4) + 4 * s4);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int j = 0; j < R; ++j) {
                    const int b = (16 * s4 + 4 * u + kg) * PB + wn + 16 * j + l16;
                    const float bv = Bs[b], uv = UP ? Us[UP ? b : 0] : 0.f;
#pragma unroll
                    for (int i = 0; i < R; ++i) {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][u], bv, acc[i][j], 0, 0, 0);
                        if constexpr (UP) acu[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][u], uv, acu[i][j], 0, 0, 0);
                    }
                }
        };
        if (steps >= STEPS) {  // (all of them in one piece: the reads of the next steps go under the products of this one)
#pragma unroll
            for (int s4 = 0; s4 < STEPS; ++s4) step(half * STEPS + s4);
        } else {
            for (int s4 = 0; s4 < steps; ++s4) step(half * STEPS + s4);
        }
        handover();
    };
    if constexpr (D == 2) {
        int k0 = 0;
        for (; k0 + KC < K; k0 += 2 * KC) {
            slab_pass(set0{}, more{}, k0);
            slab_pass(set1{}, more{}, k0 + KC);
        }
        if (k0 < K) slab_pass(set0{}, last{}, k0);
    } else {
        for (int k0 = 0; k0 < K; k0 += KC) slab_pass(set0{}, more{}, k0);
    }
    if constexpr (KG == 2) {  // the second half's sums, through LDS
        float* const o = slab + (threadIdx.x & 255) * (R * R * 4 * (UP ? 2 : 1));
        if (half) {
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int j = 0; j < R; ++j) {
                    *reinterpret_cast<floatx4*>(o + (i * R + j) * 4) = acc[i][j];
                    if constexpr (UP) *reinterpret_cast<floatx4*>(o + (R * R + i * R + j) * 4) = acu[i][j];
                }
        }
        __syncthreads();
        if (half) return;
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int j = 0; j < R; ++j) {
                acc[i][j] += *reinterpret_cast<const floatx4*>(o + (i * R + j) * 4);
                if constexpr (UP) acu[i][j] += *reinterpret_cast<const floatx4*>(o + (R * R + i * R + j) * 4);
            }
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < R; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = wm + 16 * i + 4 * kg + q, c = n0 + wn + 16 * j + l16;
                if (r >= rv || c >= N) continue;
                float x = acc[i][j][q];
                if constexpr (EPI == EPI_GELU) x = act_gelu(x);
                if constexpr (EPI == EPI_SILU) x = act_silu(x);
                if constexpr (UP) x = act_silu(x) * acu[i][j][q];
                C[(size_t)(row0 + r) * N + c] = x;
                if constexpr (RET)
                    if (s_at[r] >= 0) side.buf[(size_t)s_at[r] * N + c] = x;
            }
}

// ---- per-row fp8 quantisation of bf16 rows (one wave per row) -------------------------------------
// Rows of up to 64 * NV * 8 columns are held in registers between the amax pass and the conversion, so
// they are read from memory once; longer rows are read twice.
template <int NV>  // 16-byte vectors per lane kept in registers (0: stream the row twice)
__global__ __launch_bounds__(256) void quantize_rows_fp8_kernel(const bf16_t* __restrict__ x, int rows, int cols,
                                                                 uint8_t* __restrict__ q, float* __restrict__ scale,
                                                                 const int32_t* __restrict__ n_rows_dev,
                                                                 const int32_t* __restrict__ src_map) {
    const int wave = threadIdx.x / WAVE, lane = lane_id();
    const int limit = n_rows_dev ? min(rows, *n_rows_dev) : rows;
    const int nv = cols / 8;
    for (int r = blockIdx.x * 4 + wave; r < limit; r += gridDim.x * 4) {
        const uint4* src = (const uint4*)(x + (size_t)(src_map ? max(src_map[r], 0) : r) * cols);
        uint4 held[NV > 0 ? NV : 1];
        float amax = 0.f;
        if constexpr (NV > 0) {
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int c = lane + i * WAVE;
                held[i] = c < nv ? src[c] : make_uint4(0, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < NV; ++i) amax = fp8_row_amax(held[i], amax);
        } else {
            for (int c = lane; c < nv; c += WAVE) amax = fp8_row_amax(src[c], amax);
        }
        amax = __int_as_float(wave_max0(__float_as_int(amax)));  // (never NaN, never below 0: the bits are ordered alike)
        const bool zero = amax == 0.f;
        const float inv = zero ? 1.f : __fdiv_rn(448.f, amax);
        if (lane == 0) scale[r] = zero ? 1.f : __fdiv_rn(amax, 448.f);
        uint2* dst = (uint2*)(q + (size_t)r * cols);
        if constexpr (NV > 0) {
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int c = lane + i * WAVE;
                if (c < nv) dst[c] = fp8_row_convert(held[i], inv);
            }
        } else {
            for (int c = lane; c < nv; c += WAVE) dst[c] = fp8_row_convert(src[c], inv);
        }
    }
}

// out[r] = scale[map[r]] (map NULL: scale[r]; a negative entry takes row 0, like the GEMM's row gather)
__global__ __launch_bounds__(256) void gather_scale_kernel(const float* __restrict__ scale, const int32_t* __restrict__ map, int n,
                                                            float* __restrict__ out) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < n) out[r] = scale[map ? max(map[r], 0) : r];
}

// ---- backward pass helpers -----------------------------------------------------------------------------------------
// Re-tiling of w [E_l,K,N] as the weights of the TRANSPOSED product (d tokens = d out @ w^T: reduction over N, K output
// columns): out[e][n / SK][k][n % SK] = w[e][k][n], rows k in [K, Kpad) zero.  No transposition is involved: the 64-byte
// runs of n are contiguous on both sides.  With w_up the slabs alternate (32 n of w, 32 n of w_up, ...), which is the
// column order of the fused gate/up product, so the same call serves d tokens = [d gate | d up] @ [w_gate | w_up]^T.
template <typename T>
__global__ __launch_bounds__(256) void prepack_t_kernel(const T* __restrict__ w, const T* __restrict__ w_up, T* __restrict__ out,
                                                         int K, int N, int Kpad, bool vec) {
    constexpr int SK = ROWB / (int)sizeof(T);
    constexpr int VPS = ROWB / 16;  // 16-byte vectors per 64-byte run
    const int e = blockIdx.y;
    const int nsl = N / SK, passes = w_up ? 2 : 1;
    const size_t total = (size_t)nsl * passes * Kpad * VPS;
    const uint4 z = make_uint4(0, 0, 0, 0);
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const int v = (int)(i % VPS);
        const int k = (int)((i / VPS) % Kpad);
        const int slab = (int)(i / ((size_t)VPS * Kpad));  // output slab: (n / SK) * passes + pass
        const int ns = slab / passes, pass = slab % passes;
        const T* src = (pass ? w_up : w) + (size_t)e * K * N;
        uint4 val = z;
        const int kc = gg_packed_col<sizeof(T) == 1>(k);  // the output column of the transposed product this row stands for
        const T* from = src + (size_t)kc * N + (size_t)ns * SK + v * (16 / (int)sizeof(T));
        if (kc < K) {
            if (vec) val = *reinterpret_cast<const uint4*>(from);
            else __builtin_memcpy(&val, from, 16);  // (w or w_up not at a multiple of 16 bytes)
        }
        *reinterpret_cast<uint4*>(out + (((size_t)e * nsl * passes + slab) * Kpad + k) * SK + v * (16 / (int)sizeof(T))) = val;
    }
}

// Gradient through the activation of the expert MLP.  a1: the pre-activations as the first GEMM produces them without an
// epilogue ([rows, F] for GELU / SiLU; [rows, 2F] in the fused gate/up column order -- 32 gate columns, their 32 up
// columns, ... -- for SwiGLU); dh: gradient of the hidden activation [rows, F]; out: gradient of a1, same layout as a1.
//   GELU (erf):  dx = dh * (Phi(x) + x phi(x));   SiLU: dx = dh * s (1 + x (1 - s)), s = sigmoid(x);
//   SwiGLU h = silu(g) u:  dg = dh * u * silu'(g),  du = dh * silu(g).
template <typename T>
__device__ __forceinline__ void store_f32(T* p, float v);
template <>
__device__ __forceinline__ void store_f32<float>(float* p, float v) { *p = v; }
template <>
__device__ __forceinline__ void store_f32<bf16_t>(bf16_t* p, float v) { *p = f32_to_bf16(v); }

template <int EPI, typename T>
__global__ __launch_bounds__(256) void act_backward_kernel(const T* __restrict__ a1, const T* __restrict__ dh,
                                                            T* __restrict__ out, size_t rows, int F) {
    const size_t total = rows * (size_t)F;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const size_t r = i / F;
        const int n = (int)(i % F);
        const float d = load_f32<T>(dh + i);
        if constexpr (EPI == EPI_SWIGLU) {
            const size_t base = r * (size_t)(2 * F) + (size_t)(n / 32) * 64 + n % 32;
            const float gv = load_f32<T>(a1 + base), uv = load_f32<T>(a1 + base + 32);
            const float s = 1.0f / (1.0f + __expf(-gv));
            store_f32<T>(out + base, d * uv * (s * (1.0f + gv * (1.0f - s))));
            store_f32<T>(out + base + 32, d * (gv * s));
        } else {
            const float x = load_f32<T>(a1 + i);
            float dv = d;
            if constexpr (EPI == EPI_GELU)
                dv = d * (0.5f * (1.0f + erff(x * 0.70710678118654752440f)) + x * 0.39894228040143267794f * __expf(-0.5f * x * x));
            if constexpr (EPI == EPI_SILU) {
                const float s = 1.0f / (1.0f + __expf(-x));
                dv = d * (s * (1.0f + x * (1.0f - s)));
            }
            store_f32<T>(out + i, dv);
        }
    }
}

// The bf16 form: eight consecutive columns per thread, 16 bytes per load and store (F a multiple of 8, aligned buffers; the gate and the up column of
// a SwiGLU unit lie 32 columns apart).  Memory-bound: 10 bytes per hidden value for SwiGLU.
template <int EPI>
__global__ __launch_bounds__(256) void act_backward_vec_kernel(const uint4* __restrict__ a1, const uint4* __restrict__ dh, uint4* __restrict__ out,
                                                                unsigned total, unsigned F8) {
    auto unpack = [](const uint4& v, float* f) {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) { f[2 * i] = __uint_as_float(w[i] << 16); f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u); }
    };
    auto pack = [](const float* f) {
        return make_uint4(gg_pack_bf16(f[0], f[1]), gg_pack_bf16(f[2], f[3]), gg_pack_bf16(f[4], f[5]), gg_pack_bf16(f[6], f[7]));
    };
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        float d[8], x[8], o[8];
        unpack(dh[i], d);
        if constexpr (EPI == EPI_SWIGLU) {
            const unsigned r = i / F8, n8 = i % F8;  // (four vectors per group of 32 columns)
            const size_t base = (size_t)r * 2 * F8 + (n8 / 4) * 8 + n8 % 4;
            float u[8], ou[8];
            unpack(a1[base], x);
            unpack(a1[base + 4], u);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float s = 1.0f / (1.0f + __expf(-x[e]));
                o[e] = d[e] * u[e] * (s * (1.0f + x[e] * (1.0f - s)));
                ou[e] = d[e] * (x[e] * s);
            }
            out[base] = pack(o);
            out[base + 4] = pack(ou);
        } else {
            unpack(a1[i], x);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if constexpr (EPI == EPI_GELU)
                    o[e] = d[e] * (0.5f * (1.0f + erff(x[e] * 0.70710678118654752440f)) + x[e] * 0.39894228040143267794f * __expf(-0.5f * x[e] * x[e]));
                else {
                    const float s = 1.0f / (1.0f + __expf(-x[e]));
                    o[e] = d[e] * (s * (1.0f + x[e] * (1.0f - s)));
                }
            }
            out[i] = pack(o);
        }
    }
}

// fp32 path of the backward pass (plumbing-size workloads), and bf16 operands that 16-byte loads cannot start at: d w[g] = x_g^T @
// dy_g, 64 x 64 output tiles, the group's rows in slabs of 32 through LDS, element by element; split, ldc and delta as in launch_dw.
// And the plain transposition w [E,K,N] -> [E,N,K] that d tokens = dy @ w^T needs.
template <typename T>
__global__ __launch_bounds__(256) void grouped_dw_kernel(const T* __restrict__ x, const T* __restrict__ dy, const int32_t* __restrict__ cnt,
                                                          int E_l, int K, int N, int S_rows, T* __restrict__ dw, int ldc, bool split,
                                                          long long delta) {
    constexpr int SC = 32;
    __shared__ float xs[SC][64 + 1];
    __shared__ float ys[SC][64 + 1];
    const int g = blockIdx.z, k0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    int row0 = 0;
    for (int e = 0; e < g; ++e) row0 += min(max(cnt[e], 0), S_rows - row0);  // (counts that claim too much are cut, not added)
    const int c = min(max(cnt[g], 0), S_rows - row0);
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    float acc[4][4] = {};
    for (int s0 = 0; s0 < c; s0 += SC) {
        for (int i = threadIdx.x; i < SC * 64; i += 256) {
            const int r = i / 64, cc = i % 64;
            const bool live = s0 + r < c;
            xs[r][cc] = (live && k0 + cc < K) ? load_f32<T>(x + (size_t)(row0 + s0 + r) * K + k0 + cc) : 0.f;
            ys[r][cc] = (live && n0 + cc < N) ? load_f32<T>(dy + (size_t)(row0 + s0 + r) * N + n0 + cc) : 0.f;
        }
        __syncthreads();
#pragma unroll 4
        for (int r = 0; r < SC; ++r) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = xs[r][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = ys[r][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = k0 + ty * 4 + i, n = n0 + tx * 4 + j;
            if (k >= K || n >= N) continue;
            T* row = dw + ((size_t)g * K + k) * ldc;
            store_f32<T>(split ? row + (n / 64) * 32 + n % 32 + (n % 64 >= 32 ? delta : 0) : row + n, acc[i][j]);
        }
}

__global__ __launch_bounds__(256) void transpose_f32_kernel(const float* __restrict__ w, float* __restrict__ out, int K, int N) {
    __shared__ float tile[32][33];
    const float* src = w + (size_t)blockIdx.z * K * N;
    float* dst = out + (size_t)blockIdx.z * K * N;
    const int k0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
    for (int i = threadIdx.x; i < 1024; i += 256) {
        const int k = i / 32, n = i % 32;
        tile[k][n] = (k0 + k < K && n0 + n < N) ? src[(size_t)(k0 + k) * N + n0 + n] : 0.f;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 1024; i += 256) {
        const int n = i / 32, k = i % 32;
        if (k0 + k < K && n0 + n < N) dst[(size_t)(n0 + n) * K + k0 + k] = tile[k][n];
    }
}

int num_cus() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess) cus = prop.multiProcessorCount;
        if (cus <= 0) cus = 256;
    }
    return cus;
}

int round_up(int a, int b) { return (a + b - 1) / b * b; }

// moe_diag_gemm_trace: where the next forward GEMM launches of this process leave time stamps (not thread-safe: a diagnostic)
struct { unsigned long long* buf; int flags; } g_trace = {nullptr, 0};

// What a launch of S_rows rows in E_l groups takes: the height of its tiles (32, 64: gemm_small.hip; 128: gemm_duo.hip; 256: above) and, for large ones,
// GemmParams::tail_max.  The one place where that is decided (moe_gemm_launch_plan shows it).
// The host knows the row total, not its split over the groups: every group adds about half a tile of ragged tail.  Of four estimates the smallest decides.
// Their coefficients (us) are those whose choices were best over 2300 drawn launches, each timed on all four kernels (64 .. 40000 rows, 1 .. 32 groups, K and
// columns 512 .. 14336, bf16 and fp8, even and skewed): bf16 1.3 % (geometric mean), fp8 0.7 % over the best of the four each time, where the rule before, without
// the kernel of gemm_duo.hip but with a 128-row form of the one above, was at 6.4 and 3.6 %.  They are no launch's time: what two estimates share is left
// out.  Tiles of 128 rows: 0.36 us per 64 bytes of K while a compute unit has one, 0.69 for every two; of 256 rows: 0.34 to 0.37, but they start 42 behind (few rounds
// of few tiles fill the chip badly, and a tile's store and the next one's first stages stand alone on their unit).  So 128-row tiles serve short K at any number
// of rows and long K up to some two rounds: 16384 rows of 8 groups x 2048 x 2048 139 us on 256-row tiles, 118 on these; 33618 rows of 32 x 7168 x 4096 1543 and 1638.
struct GgChoice {
    int bm, tail_max;
};
constexpr int gg_round(int bm, int cus) { return bm == 128 ? 2 * cus : cus; }  // tiles that run at a time
static GgChoice gg_choose(int S_rows, int E_l, int K, int nt, int ncols, bool fp8, int cus, const void* part_ws, size_t part_ws_bytes, bool whole) {
    if (S_rows > GG_SCAN_ROWS) return {256, 0};
    if (whole) {  // (time stamps: only the kernel above writes them, and only launches whose tiles it fills about as well as half-height ones would)
        const double t256 = ((double)S_rows / 256 + 0.5 * E_l) * nt, t128 = ((double)S_rows / 128 + 0.5 * E_l) * nt;
        return {0.62 * ceil(t128 / cus) < ceil(t256 / cus) ? 128 : 256, 0};
    }
    const int nk = K * (fp8 ? 1 : 2) / ROWB, nts = ceil_div(ncols, 128);
    const double E = std::min(E_l, S_rows), stream = E * K * ncols * (fp8 ? 1 : 2) / 5.5e6;  // (us that the weights alone take)
    GgChoice best = {32, 0};
    // (where the weights are the time, in part out of the infinity cache, the smallest tiles)
    double least = std::max(gs_estimate(32, (S_rows / 32.0 + 0.5 * E) * nts, nk, fp8, cus, part_ws, part_ws_bytes), 0.4 * stream);
    auto consider = [&](int bm, double us) {
        us = std::max(us, 0.4 * stream);
        if (us < least) { least = us; best.bm = bm; }
    };
    consider(64, gs_estimate(64, (S_rows / 64.0 + 0.5 * E) * nts, nk, fp8, cus, part_ws, part_ws_bytes));
    {
        const double x = (S_rows / 128.0 + 0.5 * E) * nt / cus, two = std::min(1.0, std::max(0.0, (x - 0.9) / 0.27));
        consider(128, 1.25 + (1 - two) * 0.36 * nk + two * std::max(1.0, x / 2 + 0.04) * 0.69 * nk + 0.09 * stream);
    }
    const GgTail t256 = gg_tail(nk, 256, fp8, cus), t128 = gg_tail(nk, 128, fp8, cus);
    {
        double us;
        if (E == 1) {  // (no group but this one: the host knows the last round)
            const int total = ceil_div(S_rows, 256) * nt, full = total / cus, rem = total % cus;
            double last = rem ? 0.37 * nk : 0;
            if (full && rem && rem <= t256.most) last = std::min(last, 4 + 0.15 * nk * (fp8 ? 1.4 : 1.225) * std::max(1.0, rem * 8.0 / cus));
            us = 43 + full * 0.34 * nk + last;
        } else {
            const double x = (S_rows / 256.0 + 0.5 * E) * nt / cus;
            us = x <= 1.2 ? 42.5 + 0.37 * nk : 43 + (x + 1) * 0.34 * nk;
        }
        consider(256, us + 0.045 * stream);
    }
    if (best.bm < 128) return best;
    const GgTail t = best.bm == 128 ? t128 : t256;
    if (E_l == 1) {
        const int total = ceil_div(S_rows, best.bm) * nt;
        best.tail_max = gg_whole_tiles(total, gg_round(best.bm, cus), t.most) == total ? 0 : t.most;
    } else best.tail_max = t.worth ? t.most : 0;
    return best;
}

template <bool FP8>
int launch_gemm(const GemmParams& p_in, int epi, hipStream_t s, void* part_ws = nullptr, size_t part_ws_bytes = 0) {
    const int grid = num_cus();
    GemmParams p = p_in;
    const bool traced = g_trace.buf && (!(g_trace.flags & 0x300) || (g_trace.flags & (epi == EPI_NONE ? 0x100 : 0x200)));
    if (traced) {  // (see moe_diag_gemm_trace: whole tiles only, so that every tile leaves its stamps)
        p.trace = g_trace.buf;
        p.trace_flags = g_trace.flags;
        part_ws = nullptr;
    }
    const GgChoice ch = gg_choose(p.S_rows, p.E_l, p.K, p.Npad / GG_BN, epi == EPI_SWIGLU ? 2 * p.N : p.N, FP8, grid, part_ws, part_ws_bytes, traced);
    if (ch.bm < 128) return launch_gemm_small(p, FP8, ch.bm, epi, part_ws, part_ws_bytes, grid, s);
    p.tail_max = ch.tail_max;
    if (FP8 && epi == EPI_NONE && !p.a_bscale) return moe_fail(MOE_ERR_INVALID, "grouped_gemm: the fp8 down projection needs block scales");
    auto tail = [&]() -> int {
        if (!p.tail_max) return moe_check_launch("grouped_gemm");
        GemmParams q = p;
        q.zero_tail = 0;
        return launch_gemm_tail(q, FP8, ch.bm, epi, part_ws, part_ws_bytes, grid, s);
    };
    if (ch.bm == 128) {
        if (traced) return moe_fail(MOE_ERR_UNSUPPORTED, "grouped_gemm: no time-stamping instantiation for this launch (256-row tiles, no activation or SwiGLU)");
        const int rc = launch_gemm_duo(p, FP8, epi, grid, s);
        return rc ? rc : tail();
    }
    // fp8 without activation is the down projection of the expert MLP: its activation operand is block-scaled
#define GG_LAUNCH(BMv, NWMv, EPIv, MODEv)                                                                      \
    do {                                                                                                  \
        constexpr bool BSAv = FP8 && EPIv == EPI_NONE;                                                    \
        if (traced) {                                                                                     \
            if constexpr (BMv == 256 && (EPIv == EPI_NONE || EPIv == EPI_SWIGLU))                         \
                grouped_gemm_kernel<BMv, NWMv, EPIv, FP8, GG_B_PACKED, BSAv, true><<<grid, NWMv * 2 * WAVE, 0, s>>>(p); \
            else return moe_fail(MOE_ERR_UNSUPPORTED, "grouped_gemm: no time-stamping instantiation for this launch (256-row tiles, no activation or SwiGLU)"); \
            break;                                                                                        \
        }                                                                                                 \
        grouped_gemm_kernel<BMv, NWMv, EPIv, FP8, MODEv, BSAv><<<grid, NWMv * 2 * WAVE, 0, s>>>(p); \
    } while (0)
#define GG_EPI_MODE(EPIv, MODEv) GG_LAUNCH(256, (FP8 ? (EPIv == EPI_NONE ? GG_FP8_BSA_NWM : GG_FP8_NWM) : GG_BIG_NWM), EPIv, MODEv)
#define GG_EPI(EPIv) GG_EPI_MODE(EPIv, GG_B_PACKED)
    if constexpr (!FP8) {  // weights in the reference layout
        if (p.b_mode != GG_B_PACKED) {
            if (traced) return moe_fail(MOE_ERR_UNSUPPORTED, "grouped_gemm: no time-stamping instantiation for weights in the reference layout");
            if (p.b_mode == GG_B_T && epi == EPI_NONE) GG_EPI_MODE(EPI_NONE, GG_B_T);
            else if (p.b_mode == GG_B_N && epi == EPI_NONE) GG_EPI_MODE(EPI_NONE, GG_B_N);
            else if (p.b_mode == GG_B_N && epi == EPI_GELU) GG_EPI_MODE(EPI_GELU, GG_B_N);
            else if (p.b_mode == GG_B_N && epi == EPI_SILU) GG_EPI_MODE(EPI_SILU, GG_B_N);
            else if (p.b_mode == GG_B_NP && epi == EPI_SWIGLU) GG_EPI_MODE(EPI_SWIGLU, GG_B_NP);
            else return moe_fail(MOE_ERR_INVALID, "grouped_gemm: weight mode %d with activation %d", p.b_mode, epi);
            return tail();
        }
    }
    switch (epi) {
        case EPI_NONE:
            GG_EPI(EPI_NONE);
            break;
        // (no fp8 entry point asks for these two: not instantiated)
        case EPI_GELU: if constexpr (FP8) return moe_fail(MOE_ERR_UNSUPPORTED, "grouped_gemm: fp8 with activation %d", epi); else GG_EPI(EPI_GELU); break;
        case EPI_SILU: if constexpr (FP8) return moe_fail(MOE_ERR_UNSUPPORTED, "grouped_gemm: fp8 with activation %d", epi); else GG_EPI(EPI_SILU); break;
        case EPI_SWIGLU: GG_EPI(EPI_SWIGLU); break;
        case EPI_GATE: if constexpr (FP8) return moe_fail(MOE_ERR_UNSUPPORTED, "grouped_gemm: fp8 folds a gate into its row scale"); else GG_EPI(EPI_GATE); break;
        default: return moe_fail(MOE_ERR_INVALID, "grouped_gemm: activation %d", epi);
    }
#undef GG_EPI
#undef GG_EPI_MODE
#undef GG_LAUNCH
    return tail();
}

constexpr int gg_f32_lds(int R, int KG, bool up) {
    const int KC = 128 / R * KG;
    return (32 * R * (KC + 4) + (up ? 2 : 1) * KC * (32 * R + 16)) * 4;
}
// How an fp32 launch goes (the one place where that is decided; moe_gemm_f32_plan shows it).
struct F32Plan {
    int tile, sets;
    int cols, rows;  // workgroups of the tiles
};
// 64 x 64 tiles once they give every compute unit two workgroups, 32 x 32 below
bool gg_f32_big(int S_rows, int N, int cus) { return (long long)ceil_div(N, 64) * ceil_div(S_rows, 64) >= 2 * cus; }
static int f32_plan(int S_rows, int E_l, int K, int N, int epi, int side, int cus, F32Plan* p) {
    const bool big = gg_f32_big(S_rows, N, cus);
    // (a side that a launch does not have would be left out without a word: rows or padding unwritten)
    MOE_REQUIRE(side == F32_ROWS || !big, MOE_ERR_UNSUPPORTED, "grouped_gemm: 64 x 64 tiles do not move rows (%d rows, %d columns)", S_rows, N);
    MOE_REQUIRE(side != F32_RETURN || epi == EPI_NONE, MOE_ERR_UNSUPPORTED, "grouped_gemm: results go to their slots without an activation (%d)", epi);
    // Two sets of waves to a tile where the chip takes all tiles at once: one such workgroup fits a compute unit (82 KB of LDS), three of the others
    // do.  One set / two, us at K 132, 400 and 1024: 256 tiles ratio 0.95, 0.85 and 0.71, 192 0.90, 0.82, 0.74; but 264 to 420 tiles 1.14, 1.11 and 1.06, 640
    // 1.35, 1.33 and 1.33.  Counted are the tiles that rows spread at random make: one per group that has any while groups are small, then about half a
    // tile per group more than the rows fill; near the line either choice is right for about half the spreads.
    const double per = (double)S_rows / E_l;
    const double tiles = ceil_div(N, 32) * (E_l == 1 ? (double)ceil_div(S_rows, 32) : per < 16 ? E_l * (1 - exp(-per)) : S_rows / 32.0 + 0.484 * E_l);
    const bool split = !big && K > 128 && tiles <= (E_l == 1 ? 1.0 : 1.03) * cus;
    p->tile = big ? 64 : 32;
    p->sets = split ? 2 : 1;
    p->cols = ceil_div(N, p->tile);
    p->rows = ceil_div(S_rows, p->tile) + E_l;
    return MOE_OK;
}
int launch_f32(const float* A, const float* W, const float* U, float* C, const int32_t* cnt, int E_l, int K, int N, int S_rows,
               int epi, hipStream_t s, int side = F32_ROWS, F32Side sd = {}) {
    if (S_rows == 0) return MOE_OK;
    const bool vec = K % 4 == 0 && N % 4 == 0 && (((uintptr_t)(side == F32_UNPACK ? sd.buf : A) | (uintptr_t)W | (uintptr_t)U) & 15) == 0;
    F32Plan plan;
    const int rc = f32_plan(S_rows, E_l, K, N, epi, side, num_cus(), &plan);
    if (rc) return rc;
    const bool big = plan.tile == 64, split = plan.sets == 2;
    dim3 grid(plan.cols, plan.rows);
    // (a workgroup for every 16 rows of the returned buffer that S_rows cannot fill, up to a round of the chip)
    sd.tiles_y = grid.y;
    if (side == F32_RETURN) grid.y += std::min(ceil_div(std::max(sd.W * sd.M - S_rows, 1), 16 * (int)grid.x), ceil_div(num_cus(), (int)grid.x));
#define GG_F32_L(EPI, R, KG, SIDE)                                                                                                   \
    (vec ? grouped_gemm_f32_kernel<EPI, R, KG, SIDE, true> : grouped_gemm_f32_kernel<EPI, R, KG, SIDE, false>)<<<grid, 256 * KG, gg_f32_lds(R, KG, EPI == EPI_SWIGLU), s>>>(A, W, U, C, cnt, E_l, K, N, S_rows, sd)
#define GG_F32_K(EPI, R, KG)                                                                                                         \
    do {                                                                                                                             \
        if (side == F32_UNPACK) GG_F32_L(EPI, R, KG, F32_UNPACK);                                                                    \
        else if (EPI == EPI_NONE && side == F32_RETURN) GG_F32_L(EPI_NONE, R, KG, F32_RETURN);                                       \
        else GG_F32_L(EPI, R, KG, F32_ROWS);                                                                                         \
    } while (0)
#define GG_F32(EPI)                                                                                                                  \
    case EPI:                                                                                                                        \
        if (big) GG_F32_L(EPI, 2, 1, F32_ROWS);                                                                                      \
        else if (split) GG_F32_K(EPI, 1, 2);                                                                                         \
        else GG_F32_K(EPI, 1, 1);                                                                                                    \
        break
    switch (epi) {
        GG_F32(EPI_NONE);
        GG_F32(EPI_GELU);
        GG_F32(EPI_SILU);
        GG_F32(EPI_SWIGLU);
        default: return moe_fail(MOE_ERR_INVALID, "grouped_gemm: activation %d", epi);
    }
#undef GG_F32
#undef GG_F32_K
#undef GG_F32_L
    return moe_check_launch("grouped_gemm_f32");
}

template <typename T>
int launch_prepack(const T* w, const T* w_up, int E_l, int K, int N, T* out, hipStream_t s) {
    const int n_eff = N * (w_up ? 2 : 1);
    const int Npad = round_up(n_eff, GG_BN);
    if constexpr (sizeof(T) == 2) {
        if (K % 64 == 0 && N % 8 == 0 && aligned16(w) && aligned16(w_up) && aligned16(out)) {
            prepack16_kernel<<<dim3(ceil_div(w_up ? Npad / 2 : Npad, 128), K / 64, E_l * (w_up ? 2 : 1)), 256, 0, s>>>(w, w_up, out, K, N, Npad);
            return moe_check_launch("prepack_weights");
        }
    }
    const int n_zero = w_up ? n_eff : std::min(round_up(N, 64), Npad);  // (the re-tiling kernel writes the zeros up to there)
    if (Npad > n_zero) zero_pad_rows_kernel<T><<<dim3(64, E_l), 256, 0, s>>>(out, K, n_zero, Npad);
    prepack_kernel<T><<<dim3(ceil_div(N, 64), ceil_div(K, 64), E_l), 256, 0, s>>>(w, w_up, out, K, N, Npad);
    return moe_check_launch("prepack_weights");
}

}  // namespace moe_gg
using namespace moe_gg;

extern "C" size_t moe_diag_gemm_trace_words(void) { return (size_t)num_cus() * GG_TRACE_TILE_WORDS + GG_TRACE_BLOCK_WORDS; }

extern "C" int moe_diag_gemm_trace(unsigned long long* trace, size_t words, int flags) {
    MOE_REQUIRE(!trace || words >= moe_diag_gemm_trace_words(), MOE_ERR_WORKSPACE, "diag_gemm_trace: %zu words, %zu needed", words,
                moe_diag_gemm_trace_words());
    g_trace.buf = trace;
    g_trace.flags = trace ? flags : 0;
    return MOE_OK;
}

extern "C" size_t moe_prepack_bytes(int dtype, int E_l, int K, int N) {
    if (dtype == MOE_F32) return 0;
    const size_t es = dtype == MOE_BF16 ? 2 : 1;
    return (size_t)E_l * (size_t)round_up(N, GG_BN) * (size_t)K * es;
}

extern "C" int moe_prepack_weights(const void* w, const void* w_up, int dtype, int E_l, int K, int N, void* packed,
                                   moe_stream_t stream) {
    MOE_REQUIRE(dtype == MOE_BF16, MOE_ERR_INVALID, "prepack_weights: bf16 only (dtype %d)", dtype);
    MOE_REQUIRE(E_l > 0 && K > 0 && N > 0 && w && packed, MOE_ERR_INVALID, "prepack_weights: bad arguments");
    MOE_REQUIRE(!w_up || N % 32 == 0, MOE_ERR_UNSUPPORTED, "prepack_weights: gate/up interleave needs N %% 32 == 0 (N=%d)", N);
    return launch_prepack<uint16_t>((const uint16_t*)w, (const uint16_t*)w_up, E_l, K, N, (uint16_t*)packed, (hipStream_t)stream);
}

extern "C" int moe_prepack_weights_fp8(const uint8_t* w, const uint8_t* w_up, int E_l, int K, int N, uint8_t* packed,
                                       moe_stream_t stream) {
    MOE_REQUIRE(E_l > 0 && K > 0 && N > 0 && w && packed, MOE_ERR_INVALID, "prepack_weights_fp8: bad arguments");
    MOE_REQUIRE(!w_up || N % 32 == 0, MOE_ERR_UNSUPPORTED, "prepack_weights_fp8: gate/up interleave needs N %% 32 == 0");
    return launch_prepack<uint8_t>(w, w_up, E_l, K, N, packed, (hipStream_t)stream);
}

extern "C" int moe_grouped_gemm(const void* tokens, const void* weights, const int32_t* expert_cnt, int dtype, int S_rows,
                                int K, int N, int E_l, void* out, void* ws, size_t ws_bytes, moe_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    MOE_REQUIRE(S_rows >= 0 && K > 0 && N > 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "grouped_gemm: bad shape");
    if (S_rows == 0) return MOE_OK;
    MOE_REQUIRE(tokens && weights && expert_cnt && out, MOE_ERR_INVALID, "grouped_gemm: null pointer");
    if (dtype == MOE_F32)
        return launch_f32((const float*)tokens, (const float*)weights, nullptr, (float*)out, expert_cnt, E_l, K, N, S_rows,
                          EPI_NONE, s);
    MOE_REQUIRE(dtype == MOE_BF16, MOE_ERR_INVALID, "grouped_gemm: dtype %d", dtype);
    MOE_REQUIRE(K % 64 == 0 && N % 8 == 0, MOE_ERR_UNSUPPORTED, "grouped_gemm: bf16 needs K %% 64 == 0 and N %% 8 == 0 (K=%d N=%d)", K, N);
    // (the weights are taken as they are: a re-tiled copy per call would read and write them once more.  Those that the kernels' 16-byte
    // loads cannot start at are re-tiled into ws.)
    GemmParams p{};
    p.A = (const uint8_t*)tokens; p.B = (const uint8_t*)weights; p.b_mode = GG_B_N; p.C = out; p.cnt = expert_cnt;
    p.E_l = E_l; p.K = K; p.N = N; p.Npad = round_up(N, GG_BN); p.ldc = N; p.S_rows = S_rows;
    if (!aligned16(weights)) {
        MOE_REQUIRE(ws && ws_bytes >= moe_prepack_bytes(dtype, E_l, K, N), MOE_ERR_WORKSPACE,
                    "grouped_gemm: weights that are not 16-byte aligned need a workspace of %zu bytes (%zu given)",
                    moe_prepack_bytes(dtype, E_l, K, N), ws ? ws_bytes : (size_t)0);
        const int rc = moe_prepack_weights(weights, nullptr, dtype, E_l, K, N, ws, stream);
        if (rc) return rc;
        p.B = (const uint8_t*)ws; p.b_mode = GG_B_PACKED;
    }
    return launch_gemm<false>(p, EPI_NONE, s);
}

extern "C" int moe_grouped_gemm_packed(const void* tokens, const void* packed, const int32_t* expert_cnt, int S_rows, int K,
                                       int N, int E_l, int act, void* out, moe_stream_t stream) {
    MOE_REQUIRE(S_rows >= 0 && K > 0 && N > 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "grouped_gemm_packed: bad shape");
    MOE_REQUIRE(act >= EPI_NONE && act <= EPI_SWIGLU, MOE_ERR_INVALID, "grouped_gemm_packed: activation %d", act);
    MOE_REQUIRE(K % 64 == 0 && N % 8 == 0, MOE_ERR_UNSUPPORTED, "grouped_gemm_packed: needs K %% 64 == 0 and N %% 8 == 0 (K=%d N=%d)", K, N);
    if (S_rows == 0) return MOE_OK;
    MOE_REQUIRE(tokens && packed && expert_cnt && out, MOE_ERR_INVALID, "grouped_gemm_packed: null pointer");
    GemmParams p{};
    p.A = (const uint8_t*)tokens; p.B = (const uint8_t*)packed; p.C = out; p.cnt = expert_cnt;
    p.E_l = E_l; p.K = K; p.N = N; p.ldc = N; p.S_rows = S_rows;
    p.Npad = round_up(act == EPI_SWIGLU ? 2 * N : N, GG_BN);
    return launch_gemm<false>(p, act, (hipStream_t)stream);
}

// (an earlier plan for part-filled last rounds, kept for its callers: no launch follows it any more)
extern "C" int moe_gemm_split_plan(int total_tiles, int grid, int k_stages, int max_units, int32_t* out) {
    MOE_REQUIRE(total_tiles >= 0 && grid > 0 && k_stages >= 2 && k_stages % 2 == 0 && max_units >= 0 && out, MOE_ERR_INVALID,
                "gemm_split_plan: bad arguments");
    const GgPlan pl = gg_plan(total_tiles, grid, k_stages, max_units >= 2, max_units);
    out[0] = pl.full; out[1] = pl.P; out[2] = pl.nkp; out[3] = pl.units;
    return MOE_OK;
}

extern "C" int moe_gemm_launch_plan(int S_rows, int E_l, int K, int N, int act, int fp8, int cus, size_t part_ws_bytes, int tiles, int32_t* out) {
    MOE_REQUIRE(S_rows > 0 && E_l > 0 && K > 0 && N > 0 && act >= EPI_NONE && act <= EPI_SWIGLU && cus > 0 && tiles >= 0 && out, MOE_ERR_INVALID,
                "gemm_launch_plan: bad arguments");
    const int ncols = act == EPI_SWIGLU ? 2 * N : N, nk = K * (fp8 ? 1 : 2) / ROWB;
    const void* ws = part_ws_bytes ? out : nullptr;  // (any address: only whether there is one counts)
    const GgChoice ch = gg_choose(S_rows, E_l, K, ceil_div(ncols, GG_BN), ncols, fp8 != 0, cus, ws, part_ws_bytes, false);
    const bool large = ch.bm >= 128;
    const int whole = large ? gg_whole_tiles(tiles, gg_round(ch.bm, cus), ch.tail_max) : 0;
    const int small = large ? (tiles - whole) * (ch.bm / 64) * (GG_BN / 128) : tiles;  // small tiles of the launch, or of its last round
    out[0] = ch.bm;
    out[1] = whole;
    out[2] = gs_plan_parts(small, large ? 64 : ch.bm, nk, cus, ws, part_ws_bytes);
    out[3] = out[2] > 1 ? gg_part_stages(nk, out[2]) : nk;
    return MOE_OK;
}

extern "C" int moe_gemm_f32_plan(int S_rows, int E_l, int K, int N, int act, int side, int cus, int32_t* out) {
    MOE_REQUIRE(S_rows > 0 && E_l > 0 && K > 0 && N > 0 && act >= EPI_NONE && act <= EPI_SWIGLU && side >= F32_ROWS && side <= F32_UNPACK &&
                cus > 0 && out, MOE_ERR_INVALID, "gemm_f32_plan: bad arguments");
    F32Plan p;
    const int rc = f32_plan(S_rows, E_l, K, N, act, side, cus, &p);
    if (rc) return rc;
    out[0] = p.tile; out[1] = p.sets; out[2] = p.cols; out[3] = p.rows;
    return MOE_OK;
}

extern "C" size_t moe_gemm_part_workspace_bytes(void) { return gs_workspace_bytes(num_cus()); }

extern "C" int moe_grouped_gemm_mapped(const void* a_base, int a_rows, const int32_t* a_row_map, const void* packed,
                                       const int32_t* expert_cnt, int S_rows, int K, int N, int E_l, int act, void* out,
                                       int out_rows, const int32_t* c_row_map, void* part_ws, size_t part_ws_bytes,
                                       moe_stream_t stream) {
    MOE_REQUIRE(S_rows >= 0 && K > 0 && N > 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "grouped_gemm_mapped: bad shape");
    MOE_REQUIRE(act >= EPI_NONE && act <= EPI_SWIGLU, MOE_ERR_INVALID, "grouped_gemm_mapped: activation %d", act);
    MOE_REQUIRE(K % 64 == 0 && N % 8 == 0, MOE_ERR_UNSUPPORTED, "grouped_gemm_mapped: needs K %% 64 == 0 and N %% 8 == 0 (K=%d N=%d)", K, N);
    MOE_REQUIRE(a_rows >= 0 && out_rows >= 0, MOE_ERR_INVALID, "grouped_gemm_mapped: negative buffer rows");
    // gathered rows are addressed with 32-bit byte offsets from a_base
    MOE_REQUIRE(!a_row_map || (unsigned long long)a_rows * (unsigned long long)K * 2ull < (1ull << 32), MOE_ERR_UNSUPPORTED,
                "grouped_gemm_mapped: the gathered buffer must be smaller than 4 GiB (%d rows of %d)", a_rows, K);
    if (S_rows == 0) return MOE_OK;
    MOE_REQUIRE(a_base && packed && expert_cnt && out, MOE_ERR_INVALID, "grouped_gemm_mapped: null pointer");
    GemmParams p{};
    p.A = (const uint8_t*)a_base; p.B = (const uint8_t*)packed; p.C = out; p.cnt = expert_cnt;
    p.a_map = a_row_map; p.c_map = c_row_map;
    p.E_l = E_l; p.K = K; p.N = N; p.ldc = N; p.S_rows = S_rows;
    p.Npad = round_up(act == EPI_SWIGLU ? 2 * N : N, GG_BN);
    return launch_gemm<false>(p, act, (hipStream_t)stream, part_ws, part_ws_bytes);
}

extern "C" int moe_expert_forward(const void* tokens, const void* weights, int layout, const int32_t* expert_cnt, int S_rows, int K, int N,
                                  int E_l, void* out, void* part_ws, size_t part_ws_bytes, moe_stream_t stream) {
    MOE_REQUIRE(layout >= MOE_W_TILED && layout <= MOE_W_RAW_T, MOE_ERR_INVALID, "expert_forward: weight layout %d", layout);
    MOE_REQUIRE(S_rows >= 0 && K > 0 && N > 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "expert_forward: bad shape");
    MOE_REQUIRE(K % 64 == 0 && N % 8 == 0, MOE_ERR_UNSUPPORTED, "expert_forward: needs K %% 64 == 0 and N %% 8 == 0 (K=%d N=%d)", K, N);
    if (S_rows == 0) return MOE_OK;
    MOE_REQUIRE(tokens && weights && expert_cnt && out, MOE_ERR_INVALID, "expert_forward: null pointer");
    MOE_REQUIRE(aligned16(weights), MOE_ERR_INVALID, "expert_forward: weights must be 16-byte aligned");
    GemmParams p{};
    p.A = (const uint8_t*)tokens; p.B = (const uint8_t*)weights; p.C = out; p.cnt = expert_cnt; p.zero_tail = 1;
    p.b_mode = layout == MOE_W_TILED ? GG_B_PACKED : layout == MOE_W_RAW ? GG_B_N : GG_B_T;
    p.E_l = E_l; p.K = K; p.N = N; p.ldc = N; p.S_rows = S_rows; p.Npad = round_up(N, GG_BN);
    return launch_gemm<false>(p, EPI_NONE, (hipStream_t)stream, part_ws, part_ws_bytes);
}

extern "C" int moe_grouped_gemm_mapped_gated(const void* a_base, int a_rows, const int32_t* a_row_map, const void* packed,
                                             const int32_t* expert_cnt, int S_rows, int K, int N, int E_l, const float* row_gate,
                                             void* out, int out_rows, const int32_t* c_row_map, void* part_ws, size_t part_ws_bytes,
                                             moe_stream_t stream) {
    MOE_REQUIRE(S_rows >= 0 && K > 0 && N > 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "grouped_gemm_mapped_gated: bad shape");
    MOE_REQUIRE(K % 64 == 0 && N % 8 == 0, MOE_ERR_UNSUPPORTED, "grouped_gemm_mapped_gated: needs K %% 64 == 0 and N %% 8 == 0 (K=%d N=%d)", K, N);
    MOE_REQUIRE(a_rows >= 0 && out_rows >= 0, MOE_ERR_INVALID, "grouped_gemm_mapped_gated: negative buffer rows");
    MOE_REQUIRE(!a_row_map || (unsigned long long)a_rows * (unsigned long long)K * 2ull < (1ull << 32), MOE_ERR_UNSUPPORTED,
                "grouped_gemm_mapped_gated: the gathered buffer must be smaller than 4 GiB (%d rows of %d)", a_rows, K);
    if (S_rows == 0) return MOE_OK;
    MOE_REQUIRE(a_base && packed && expert_cnt && out && row_gate, MOE_ERR_INVALID, "grouped_gemm_mapped_gated: null pointer");
    GemmParams p{};
    p.A = (const uint8_t*)a_base; p.B = (const uint8_t*)packed; p.C = out; p.cnt = expert_cnt;
    p.a_map = a_row_map; p.c_map = c_row_map; p.row_scale = row_gate;
    p.E_l = E_l; p.K = K; p.N = N; p.ldc = N; p.S_rows = S_rows;
    p.Npad = round_up(N, GG_BN);
    return launch_gemm<false>(p, EPI_GATE, (hipStream_t)stream, part_ws, part_ws_bytes);
}

extern "C" int moe_grouped_gemm_act_keep(const void* a_base, int a_rows, const int32_t* a_row_map, const void* packed,
                                         const int32_t* expert_cnt, int S_rows, int K, int N, int E_l, int act, void* out,
                                         void* pre_act, void* part_ws, size_t part_ws_bytes, moe_stream_t stream) {
    MOE_REQUIRE(S_rows >= 0 && K > 0 && N > 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "grouped_gemm_act_keep: bad shape");
    MOE_REQUIRE(act > EPI_NONE && act <= EPI_SWIGLU, MOE_ERR_INVALID, "grouped_gemm_act_keep: activation %d", act);
    MOE_REQUIRE(K % 64 == 0 && N % 8 == 0, MOE_ERR_UNSUPPORTED, "grouped_gemm_act_keep: needs K %% 64 == 0 and N %% 8 == 0 (K=%d N=%d)", K, N);
    MOE_REQUIRE(a_rows >= 0, MOE_ERR_INVALID, "grouped_gemm_act_keep: negative buffer rows");
    MOE_REQUIRE(!a_row_map || (unsigned long long)a_rows * (unsigned long long)K * 2ull < (1ull << 32), MOE_ERR_UNSUPPORTED,
                "grouped_gemm_act_keep: the gathered buffer must be smaller than 4 GiB (%d rows of %d)", a_rows, K);
    if (S_rows == 0) return MOE_OK;
    MOE_REQUIRE(a_base && packed && expert_cnt && out && pre_act, MOE_ERR_INVALID, "grouped_gemm_act_keep: null pointer");
    GemmParams p{};
    p.A = (const uint8_t*)a_base; p.B = (const uint8_t*)packed; p.C = out; p.C2 = pre_act; p.cnt = expert_cnt;
    p.a_map = a_row_map;
    p.E_l = E_l; p.K = K; p.N = N; p.ldc = N; p.S_rows = S_rows;
    p.Npad = round_up(act == EPI_SWIGLU ? 2 * N : N, GG_BN);
    return launch_gemm<false>(p, act, (hipStream_t)stream, part_ws, part_ws_bytes);
}

extern "C" int moe_grouped_mlp(const void* tokens, const int32_t* expert_cnt, int dtype, int S_rows, int H, int F, int E_l,
                               int act, const void* w1, const void* w_up, const void* w2, void* hidden_ws, void* out,
                               moe_stream_t stream) {
    return moe_grouped_mlp_split(tokens, expert_cnt, dtype, S_rows, H, F, E_l, act, w1, w_up, w2, hidden_ws, out, nullptr, 0, stream);
}

int moe_mlp_f32_slots(const float* recv, const int32_t* recv_counts, int W, int M, int S_rows, int H, int F, int E_l, int act, const float* w1,
                      const float* w_up, const float* w2, float* rows, int32_t* expert_cnt, float* hidden_ws, float* y, float* ret,
                      hipStream_t s) {
    MOE_REQUIRE(S_rows > 0 && H > 0 && H % 4 == 0 && F > 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "grouped_mlp: bad shape");
    MOE_REQUIRE(act == EPI_GELU || act == EPI_SILU || act == EPI_SWIGLU || act == EPI_NONE, MOE_ERR_INVALID,
                "grouped_mlp: activation %d", act);
    MOE_REQUIRE(recv && rows && expert_cnt && w1 && w2 && hidden_ws && y && (act != EPI_SWIGLU || w_up), MOE_ERR_INVALID, "grouped_mlp: null pointer");
    MOE_REQUIRE(W > 0 && W * E_l <= MOE_MAX_EXPERTS && M >= 1 && recv_counts && ret, MOE_ERR_INVALID, "return_pack: bad arguments");
    MOE_REQUIRE((long long)W * M < (1ll << 31), MOE_ERR_UNSUPPORTED, "return_pack: W*M too large");
    // (with large tiles the rows' places, looked up slab by slab, cost more than the copies: H 512, F 1024, 54 940 rows 1443 -> 1635 us a step, 14 613 456 -> 480)
    const bool up = !gg_f32_big(S_rows, F, num_cus()), down = !gg_f32_big(S_rows, H, num_cus());
    int rc = up ? MOE_OK : moe_unpack_expert_major(recv, MOE_F32, W, M, H, recv_counts, E_l, rows, S_rows, expert_cnt, nullptr, s);
    if (rc) return rc;
    rc = launch_f32(rows, w1, w_up, hidden_ws, expert_cnt, E_l, H, F, S_rows, act, s, up ? F32_UNPACK : F32_ROWS,
                    {recv_counts, W, M, const_cast<float*>(recv), 0, rows, expert_cnt});
    if (rc) return rc;
    rc = launch_f32(hidden_ws, w2, nullptr, y, expert_cnt, E_l, F, H, S_rows, EPI_NONE, s, down ? F32_RETURN : F32_ROWS,
                    {recv_counts, W, M, ret, 0, nullptr, nullptr});
    if (rc || down) return rc;
    return moe_return_pack(y, MOE_F32, S_rows, H, recv_counts, W, E_l, M, ret, nullptr, s);
}

extern "C" int moe_grouped_mlp_split(const void* tokens, const int32_t* expert_cnt, int dtype, int S_rows, int H, int F, int E_l,
                                     int act, const void* w1, const void* w_up, const void* w2, void* hidden_ws, void* out,
                                     void* part_ws, size_t part_ws_bytes, moe_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    MOE_REQUIRE(S_rows >= 0 && H > 0 && F > 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "grouped_mlp: bad shape");
    MOE_REQUIRE(act == EPI_GELU || act == EPI_SILU || act == EPI_SWIGLU || act == EPI_NONE, MOE_ERR_INVALID,
                "grouped_mlp: activation %d", act);
    if (S_rows == 0) return MOE_OK;
    MOE_REQUIRE(tokens && expert_cnt && w1 && w2 && hidden_ws && out, MOE_ERR_INVALID, "grouped_mlp: null pointer");
    if (dtype == MOE_F32) {
        MOE_REQUIRE(act != EPI_SWIGLU || w_up, MOE_ERR_INVALID, "grouped_mlp: swiglu needs w_up");
        int rc = launch_f32((const float*)tokens, (const float*)w1, (const float*)w_up, (float*)hidden_ws, expert_cnt, E_l, H,
                            F, S_rows, act, s);
        if (rc) return rc;
        return launch_f32((const float*)hidden_ws, (const float*)w2, nullptr, (float*)out, expert_cnt, E_l, F, H, S_rows,
                          EPI_NONE, s);
    }
    MOE_REQUIRE(dtype == MOE_BF16, MOE_ERR_INVALID, "grouped_mlp: dtype %d", dtype);
    MOE_REQUIRE(w_up == nullptr, MOE_ERR_INVALID, "grouped_mlp: bf16 takes gate/up interleaved in w1 (w_up must be NULL)");
    MOE_REQUIRE(H % 64 == 0 && F % 64 == 0, MOE_ERR_UNSUPPORTED, "grouped_mlp: bf16 needs H, F multiples of 64 (H=%d F=%d)", H, F);
    GemmParams p{};
    p.A = (const uint8_t*)tokens; p.B = (const uint8_t*)w1; p.C = hidden_ws; p.cnt = expert_cnt;
    p.E_l = E_l; p.K = H; p.N = F; p.ldc = F; p.S_rows = S_rows;
    p.Npad = round_up(act == EPI_SWIGLU ? 2 * F : F, GG_BN);
    int rc = launch_gemm<false>(p, act, s, part_ws, part_ws_bytes);
    if (rc) return rc;
    GemmParams q{};
    q.A = (const uint8_t*)hidden_ws; q.B = (const uint8_t*)w2; q.C = out; q.cnt = expert_cnt;
    q.E_l = E_l; q.K = F; q.N = H; q.Npad = round_up(H, GG_BN); q.ldc = H; q.S_rows = S_rows;
    return launch_gemm<false>(q, EPI_NONE, s, part_ws, part_ws_bytes);
}

static int launch_quantize(const void* x_bf16, const int32_t* src_map, int rows, int cols, uint8_t* q, float* scale,
                           const int32_t* n_rows_dev, hipStream_t s) {
    const int blocks = min(ceil_div(rows, 4), 65535 * 8);
    const int nv = ceil_div(cols / 8, WAVE);  // 16-byte vectors per lane
#define GG_Q(NVv) quantize_rows_fp8_kernel<NVv><<<blocks, 256, 0, s>>>((const bf16_t*)x_bf16, rows, cols, q, scale, n_rows_dev, src_map)
    if (nv <= 2) GG_Q(2);
    else if (nv <= 4) GG_Q(4);
    else if (nv <= 8) GG_Q(8);
    else if (nv <= 16) GG_Q(16);
    else GG_Q(0);
#undef GG_Q
    return moe_check_launch("quantize_rows_fp8");
}

extern "C" int moe_quantize_rows_fp8(const void* x_bf16, int rows, int cols, uint8_t* q, float* scale,
                                     const int32_t* n_rows_dev, moe_stream_t stream) {
    MOE_REQUIRE(rows >= 0 && cols > 0 && cols % 8 == 0, MOE_ERR_INVALID, "quantize_rows_fp8: cols must be a multiple of 8");
    if (rows == 0) return MOE_OK;
    MOE_REQUIRE(x_bf16 && q && scale, MOE_ERR_INVALID, "quantize_rows_fp8: null pointer");
    return launch_quantize(x_bf16, nullptr, rows, cols, q, scale, n_rows_dev, (hipStream_t)stream);
}

// The two GEMMs of the fp8 SwiGLU expert on quantised rows (xq codes gathered through a_map, xs their scales in GEMM row
// order): gate/up + SwiGLU with the hidden activation quantised in the epilogue (codes hq, one E8M0 scale byte per row and
// 32 columns in hscale), then the down projection, which takes those bytes as the scale operand of its MFMAs; row_gate
// (nullable) multiplies the result rows.
static int fp8_mlp_gemms(const uint8_t* xq, const int32_t* a_map, const float* xs, const int32_t* expert_cnt, int S_rows, int H, int F,
                         int E_l, const uint8_t* wgu_packed, const float* sg, const float* su, const uint8_t* wd_packed,
                         const float* sd, uint8_t* hq_ws, uint8_t* hscale_ws, const float* row_gate, void* out,
                         const int32_t* c_row_map, void* part_ws, size_t part_ws_bytes, hipStream_t s) {
    GemmParams p{};
    p.A = xq; p.B = wgu_packed; p.C = hq_ws; p.cnt = expert_cnt; p.row_scale = xs; p.col_scale = sg; p.col_scale2 = su;
    p.a_map = a_map; p.c_bscale = hscale_ws; p.bs_pitch = F / 32;
    p.E_l = E_l; p.K = H; p.N = F; p.Npad = round_up(2 * F, GG_BN); p.ldc = F; p.S_rows = S_rows; p.ncs = F;
    int rc = launch_gemm<true>(p, EPI_SWIGLU, s, part_ws, part_ws_bytes);
    if (rc) return rc;
    GemmParams q{};
    q.A = hq_ws; q.B = wd_packed; q.C = out; q.cnt = expert_cnt; q.row_scale = row_gate; q.col_scale = sd;
    q.c_map = c_row_map; q.a_bscale = hscale_ws; q.bs_pitch = F / 32;
    q.E_l = E_l; q.K = F; q.N = H; q.Npad = round_up(H, GG_BN); q.ldc = H; q.S_rows = S_rows; q.ncs = H;
    return launch_gemm<true>(q, EPI_NONE, s, part_ws, part_ws_bytes);
}

extern "C" int moe_grouped_mlp_fp8_mapped(const void* a_base_bf16, int a_rows, const int32_t* a_row_map,
                                          const int32_t* expert_cnt, int S_rows, int H, int F, int E_l,
                                          const uint8_t* wgu_packed, const float* sg, const float* su,
                                          const uint8_t* wd_packed, const float* sd, uint8_t* xq_ws, float* xs_ws,
                                          uint8_t* hq_ws, uint8_t* hscale_ws, const float* row_gate, void* out, int out_rows,
                                          const int32_t* c_row_map, void* part_ws, size_t part_ws_bytes, moe_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    MOE_REQUIRE(S_rows >= 0 && H > 0 && F > 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "grouped_mlp_fp8: bad shape");
    MOE_REQUIRE(H % 128 == 0 && F % 128 == 0, MOE_ERR_UNSUPPORTED, "grouped_mlp_fp8: needs H, F multiples of 128 (H=%d F=%d)", H, F);
    MOE_REQUIRE(a_rows >= 0 && out_rows >= 0, MOE_ERR_INVALID, "grouped_mlp_fp8: negative buffer rows");
    MOE_REQUIRE((unsigned long long)S_rows * (unsigned long long)(F / 32) < (1ull << 32), MOE_ERR_UNSUPPORTED,
                "grouped_mlp_fp8: the block scales must stay under 4 GiB");
    if (S_rows == 0) return MOE_OK;
    MOE_REQUIRE(a_base_bf16 && expert_cnt && wgu_packed && sg && su && wd_packed && sd && xq_ws && xs_ws && hq_ws && hscale_ws && out,
                MOE_ERR_INVALID, "grouped_mlp_fp8: null pointer");
    // the row quantisation reads every input row once anyway: with a map it reads it where the transfer left it
    int rc = launch_quantize(a_base_bf16, a_row_map, S_rows, H, xq_ws, xs_ws, nullptr, s);
    if (rc) return rc;
    return fp8_mlp_gemms(xq_ws, nullptr, xs_ws, expert_cnt, S_rows, H, F, E_l, wgu_packed, sg, su, wd_packed, sd, hq_ws, hscale_ws,
                         row_gate, out, c_row_map, part_ws, part_ws_bytes, s);
}

extern "C" int moe_grouped_mlp_fp8(const void* tokens_bf16, const int32_t* expert_cnt, int S_rows, int H, int F, int E_l,
                                   const uint8_t* wgu_packed, const float* sg, const float* su, const uint8_t* wd_packed,
                                   const float* sd, uint8_t* xq_ws, float* xs_ws, uint8_t* hq_ws, uint8_t* hscale_ws, void* out,
                                   moe_stream_t stream) {
    return moe_grouped_mlp_fp8_mapped(tokens_bf16, S_rows, nullptr, expert_cnt, S_rows, H, F, E_l, wgu_packed, sg, su, wd_packed,
                                      sd, xq_ws, xs_ws, hq_ws, hscale_ws, nullptr, out, S_rows, nullptr, nullptr, 0, stream);
}

extern "C" int moe_grouped_mlp_fp8_q_mapped(const uint8_t* a_q, const float* a_scale, int a_rows, const int32_t* a_row_map,
                                            const int32_t* expert_cnt, int S_rows, int H, int F, int E_l,
                                            const uint8_t* wgu_packed, const float* sg, const float* su,
                                            const uint8_t* wd_packed, const float* sd, float* xs_ws, uint8_t* hq_ws,
                                            uint8_t* hscale_ws, const float* row_gate, void* out, int out_rows,
                                            const int32_t* c_row_map, void* part_ws, size_t part_ws_bytes, moe_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    MOE_REQUIRE(S_rows >= 0 && H > 0 && F > 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "grouped_mlp_fp8_q: bad shape");
    MOE_REQUIRE(H % 128 == 0 && F % 128 == 0, MOE_ERR_UNSUPPORTED, "grouped_mlp_fp8_q: needs H, F multiples of 128 (H=%d F=%d)", H, F);
    MOE_REQUIRE(a_rows >= 0 && out_rows >= 0, MOE_ERR_INVALID, "grouped_mlp_fp8_q: negative buffer rows");
    MOE_REQUIRE(!a_row_map || (unsigned long long)a_rows * (unsigned long long)H < (1ull << 32), MOE_ERR_UNSUPPORTED,
                "grouped_mlp_fp8_q: the gathered buffer must be smaller than 4 GiB (%d rows of %d)", a_rows, H);
    MOE_REQUIRE((unsigned long long)S_rows * (unsigned long long)(F / 32) < (1ull << 32), MOE_ERR_UNSUPPORTED,
                "grouped_mlp_fp8_q: the block scales must stay under 4 GiB");
    if (S_rows == 0) return MOE_OK;
    MOE_REQUIRE(a_q && expert_cnt && wgu_packed && sg && su && wd_packed && sd && xs_ws && hq_ws && hscale_ws && out,
                MOE_ERR_INVALID, "grouped_mlp_fp8_q: null pointer");
    // the row scales in the order of the GEMM's rows (the codes themselves are gathered by the GEMM as it loads them)
    if (a_scale) gather_scale_kernel<<<ceil_div(S_rows, 256), 256, 0, s>>>(a_scale, a_row_map, S_rows, xs_ws);
    return fp8_mlp_gemms(a_q, a_row_map, xs_ws, expert_cnt, S_rows, H, F, E_l, wgu_packed, sg, su, wd_packed, sd, hq_ws, hscale_ws,
                         row_gate, out, c_row_map, part_ws, part_ws_bytes, s);
}

// ---- backward pass entry points --------------------------------------------------------------------------------------
extern "C" int moe_prepack_weights_transposed(const void* w, const void* w_up, int dtype, int E_l, int K, int N, void* packed,
                                              moe_stream_t stream) {
    MOE_REQUIRE(dtype == MOE_BF16, MOE_ERR_INVALID, "prepack_weights_transposed: bf16 only (dtype %d)", dtype);
    MOE_REQUIRE(E_l > 0 && K > 0 && N > 0 && w && packed, MOE_ERR_INVALID, "prepack_weights_transposed: bad arguments");
    MOE_REQUIRE(N % 64 == 0 && K % 8 == 0, MOE_ERR_UNSUPPORTED,
                "prepack_weights_transposed: needs N %% 64 == 0 and K %% 8 == 0 (K=%d N=%d)", K, N);
    const int Kpad = round_up(K, GG_BN);
    prepack_t_kernel<uint16_t><<<dim3(1024, E_l), 256, 0, (hipStream_t)stream>>>((const uint16_t*)w, (const uint16_t*)w_up,
                                                                               (uint16_t*)packed, K, N, Kpad, aligned16(w) && aligned16(w_up));
    return moe_check_launch("prepack_weights_transposed");
}

// (the operands were rewritten with the row index fastest here once; the kernel reads them as they are now)
extern "C" size_t moe_dw_workspace_bytes(int, int, int, int) { return 0; }

// split_F > 0: dy's columns in the fused gate / up order; gate columns go to dw (row pitch ldc), up columns dw_delta elements further
static int launch_dw(const void* x, const void* dy, const int32_t* expert_cnt, int S_rows, int K, int N, int E_l, int split_F, void* dw,
                     int ldc, long long dw_delta, hipStream_t s) {
    MOE_REQUIRE(N % 8 == 0 && K % 8 == 0, MOE_ERR_UNSUPPORTED, "grouped_gemm_dw: bf16 needs K, N multiples of 8 (K=%d N=%d)", K, N);
    if (!(aligned16(x) && aligned16(dy) && aligned16(dw) && dw_delta % 8 == 0)) {
        grouped_dw_kernel<bf16_t><<<dim3(ceil_div(N, 64), ceil_div(K, 64), E_l), 256, 0, s>>>(
            (const bf16_t*)x, (const bf16_t*)dy, expert_cnt, E_l, K, N, S_rows, (bf16_t*)dw, ldc, split_F > 0, dw_delta);
        return moe_check_launch("grouped_gemm_dw");
    }
    GemmParams p{};
    p.A = (const uint8_t*)x; p.B = (const uint8_t*)dy; p.C = dw; p.cnt = expert_cnt;
    p.E_l = E_l; p.K = 64; p.N = N; p.Npad = round_up(N, GG_BN); p.ldc = ldc; p.S_rows = K;
    p.dw_rows = K; p.dw_src_rows = S_rows; p.dw_split = split_F; p.dw_delta = dw_delta; p.c_group_stride = (size_t)K * ldc;
    // 128-row tiles (gemm_duo.hip) while 256-row ones do not fill the chip, and for short reductions over some rounds of them, where storing tiles is most of
    // the work.  160 drawn launches: 0.53 to 0.85 of the time at up to half a round (817 rows of 2 groups x 576 x 640 18.2 us -> 10.6) and, up to 300 rows a
    // group, to five rounds; from 10 rounds or some 2000 rows times rounds on 0.9 to 1.1 (33618 rows of 32 groups x 7168 x 4096: 1780 us, 1900 on these).
    const int cus = num_cus();
    const double rounds = (double)E_l * ceil_div(K, 256) * (p.Npad / GG_BN) / cus;
    if (S_rows <= GG_SCAN_ROWS && (rounds <= 0.9 || (rounds <= 10 && rounds * S_rows / E_l <= 2000))) return launch_gemm_duo(p, false, EPI_NONE, cus, s);
    grouped_gemm_kernel<256, GG_BIG_NWM, EPI_NONE, false, GG_B_DW><<<cus, GG_BIG_NWM * 2 * WAVE, 0, s>>>(p);
    return moe_check_launch("grouped_gemm_dw");
}

extern "C" int moe_grouped_gemm_dw(const void* x, const void* dy, const int32_t* expert_cnt, int dtype, int S_rows, int K, int N,
                                   int E_l, int split_F, void* dw, void* ws, size_t ws_bytes, moe_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    (void)ws; (void)ws_bytes;
    MOE_REQUIRE(S_rows >= 0 && K > 0 && N > 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "grouped_gemm_dw: bad shape");
    MOE_REQUIRE(expert_cnt && dw && (S_rows == 0 || (x && dy)), MOE_ERR_INVALID, "grouped_gemm_dw: null pointer");
    MOE_REQUIRE(split_F == 0 || (dtype == MOE_BF16 && split_F % 32 == 0 && N == 2 * split_F), MOE_ERR_INVALID,
                "grouped_gemm_dw: split_F=%d needs bf16, split_F %% 32 == 0 and N == 2 split_F", split_F);
    if (dtype == MOE_F32) {
        grouped_dw_kernel<float><<<dim3(ceil_div(N, 64), ceil_div(K, 64), E_l), 256, 0, s>>>((const float*)x, (const float*)dy, expert_cnt, E_l, K,
                                                                                              N, S_rows, (float*)dw, N, false, 0);
        return moe_check_launch("grouped_gemm_dw_f32");
    }
    MOE_REQUIRE(dtype == MOE_BF16, MOE_ERR_INVALID, "grouped_gemm_dw: dtype %d", dtype);
    return launch_dw(x, dy, expert_cnt, S_rows, K, N, E_l, split_F, dw, N, split_F, s);
}

extern "C" int moe_grouped_gemm_dw_pair(const void* x, const void* dy, const int32_t* expert_cnt, int S_rows, int K, int F, int E_l,
                                        void* dw_gate, void* dw_up, moe_stream_t stream) {
    MOE_REQUIRE(S_rows >= 0 && K > 0 && F > 0 && F % 32 == 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "grouped_gemm_dw_pair: bad shape");
    MOE_REQUIRE(expert_cnt && dw_gate && dw_up && (S_rows == 0 || (x && dy)), MOE_ERR_INVALID, "grouped_gemm_dw_pair: null pointer");
    return launch_dw(x, dy, expert_cnt, S_rows, K, 2 * F, E_l, F, dw_gate, F, (bf16_t*)dw_up - (bf16_t*)dw_gate, (hipStream_t)stream);
}

// ---- the expert MLP of a training step, one call per direction (bf16); pre_act as moe_grouped_gemm_act_keep leaves it.
extern "C" int moe_mlp_train_forward(const void* x, const int32_t* expert_cnt, int S_rows, int H, int F, int E_l, int act, int layout,
                                     const void* w1, const void* w_up, const void* w2, void* hidden, void* pre_act, void* out, void* part_ws,
                                     size_t part_ws_bytes, moe_stream_t stream) {
    MOE_REQUIRE(S_rows > 0 && H > 0 && F > 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "mlp_train_forward: bad shape");
    MOE_REQUIRE(act > EPI_NONE && act <= EPI_SWIGLU, MOE_ERR_INVALID, "mlp_train_forward: activation %d", act);
    MOE_REQUIRE(H % 64 == 0 && F % 64 == 0, MOE_ERR_UNSUPPORTED, "mlp_train_forward: needs H, F multiples of 64 (H=%d F=%d)", H, F);
    MOE_REQUIRE(layout == MOE_W_TILED || layout == MOE_W_RAW, MOE_ERR_INVALID, "mlp_train_forward: weight layout %d", layout);
    const bool raw = layout == MOE_W_RAW, pair = raw && act == EPI_SWIGLU;
    MOE_REQUIRE(x && expert_cnt && w1 && w2 && hidden && pre_act && out && (!pair || w_up), MOE_ERR_INVALID, "mlp_train_forward: null pointer");
    MOE_REQUIRE(aligned16(w1) && aligned16(w_up) && aligned16(w2), MOE_ERR_INVALID, "mlp_train_forward: weights must be 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    GemmParams p{};
    p.A = (const uint8_t*)x; p.B = (const uint8_t*)w1; p.C = hidden; p.C2 = pre_act; p.cnt = expert_cnt;
    p.B2 = pair ? (const uint8_t*)w_up : nullptr;
    p.b_mode = pair ? GG_B_NP : raw ? GG_B_N : GG_B_PACKED;
    p.E_l = E_l; p.K = H; p.N = F; p.ldc = F; p.S_rows = S_rows; p.Npad = round_up(act == EPI_SWIGLU ? 2 * F : F, GG_BN);
    const int rc = launch_gemm<false>(p, act, s, part_ws, part_ws_bytes);
    if (rc) return rc;
    GemmParams q{};
    q.A = (const uint8_t*)hidden; q.B = (const uint8_t*)w2; q.C = out; q.cnt = expert_cnt; q.zero_tail = 1;
    q.b_mode = raw ? GG_B_N : GG_B_PACKED;
    q.E_l = E_l; q.K = F; q.N = H; q.ldc = H; q.S_rows = S_rows; q.Npad = round_up(H, GG_BN);
    return launch_gemm<false>(q, EPI_NONE, s, part_ws, part_ws_bytes);
}

extern "C" int moe_mlp_train_backward(const void* x, const void* hidden, const void* pre_act, const void* dy, const int32_t* expert_cnt,
                                      int S_rows, int H, int F, int E_l, int act, int layout, const void* w1, const void* w_up,
                                      const void* w2, void* dh, void* d_pre, void* dx, void* dw1, void* dw_up, void* dw2, void* part_ws, size_t part_ws_bytes, moe_stream_t stream) {
    MOE_REQUIRE(S_rows > 0 && H > 0 && F > 0 && E_l > 0 && E_l <= GG_MAXG, MOE_ERR_INVALID, "mlp_train_backward: bad shape");
    MOE_REQUIRE(act > EPI_NONE && act <= EPI_SWIGLU, MOE_ERR_INVALID, "mlp_train_backward: activation %d", act);
    MOE_REQUIRE(H % 64 == 0 && F % 64 == 0, MOE_ERR_UNSUPPORTED, "mlp_train_backward: needs H, F multiples of 64 (H=%d F=%d)", H, F);
    MOE_REQUIRE(layout == MOE_W_TILED || layout == MOE_W_RAW_T, MOE_ERR_INVALID, "mlp_train_backward: weight layout %d", layout);
    const bool raw = layout == MOE_W_RAW_T;
    MOE_REQUIRE(x && hidden && pre_act && dy && expert_cnt && w1 && w2 && dh && d_pre && dx && dw1 && dw2 && (act != EPI_SWIGLU || (dw_up && (w_up || !raw))),
                MOE_ERR_INVALID, "mlp_train_backward: null pointer");
    MOE_REQUIRE(aligned16(w1) && aligned16(w_up) && aligned16(w2), MOE_ERR_INVALID, "mlp_train_backward: weights must be 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    const int NP = act == EPI_SWIGLU ? 2 * F : F;
    GemmParams p{};
    p.A = (const uint8_t*)dy; p.B = (const uint8_t*)w2; p.b_mode = raw ? GG_B_T : GG_B_PACKED; p.C = dh; p.cnt = expert_cnt;
    p.E_l = E_l; p.K = H; p.N = F; p.ldc = F; p.S_rows = S_rows; p.Npad = round_up(F, GG_BN);
    int rc = launch_gemm<false>(p, EPI_NONE, s, part_ws, part_ws_bytes);
    if (!rc) rc = launch_dw(hidden, dy, expert_cnt, S_rows, F, H, E_l, 0, dw2, H, 0, s);
    if (!rc) rc = moe_mlp_act_backward(pre_act, dh, MOE_BF16, S_rows, F, act, d_pre, stream);
    if (rc) return rc;
    GemmParams q{};
    q.A = (const uint8_t*)d_pre; q.B = (const uint8_t*)w1; q.b_mode = raw ? GG_B_T : GG_B_PACKED; q.C = dx; q.cnt = expert_cnt; q.zero_tail = 1;
    q.B2 = raw && act == EPI_SWIGLU ? (const uint8_t*)w_up : nullptr;
    q.E_l = E_l; q.K = NP; q.N = H; q.ldc = H; q.S_rows = S_rows; q.Npad = round_up(H, GG_BN);
    rc = launch_gemm<false>(q, EPI_NONE, s, part_ws, part_ws_bytes);
    if (rc) return rc;
    if (act == EPI_SWIGLU) return launch_dw(x, d_pre, expert_cnt, S_rows, H, NP, E_l, F, dw1, F, (bf16_t*)dw_up - (bf16_t*)dw1, s);
    return launch_dw(x, d_pre, expert_cnt, S_rows, H, NP, E_l, 0, dw1, F, 0, s);
}

extern "C" int moe_transpose_weights_f32(const float* w, int E_l, int K, int N, float* out, moe_stream_t stream) {
    MOE_REQUIRE(E_l > 0 && K > 0 && N > 0 && w && out, MOE_ERR_INVALID, "transpose_weights_f32: bad arguments");
    transpose_f32_kernel<<<dim3(ceil_div(N, 32), ceil_div(K, 32), E_l), 256, 0, (hipStream_t)stream>>>(w, out, K, N);
    return moe_check_launch("transpose_weights_f32");
}

extern "C" int moe_mlp_act_backward(const void* a1, const void* dh, int dtype, int rows, int F, int act, void* d_a1,
                                    moe_stream_t stream) {
    MOE_REQUIRE(rows >= 0 && F > 0, MOE_ERR_INVALID, "mlp_act_backward: bad shape");
    MOE_REQUIRE(dtype == MOE_BF16 || (dtype == MOE_F32 && act != EPI_SWIGLU), MOE_ERR_UNSUPPORTED,
                "mlp_act_backward: dtype %d with activation %d", dtype, act);
    MOE_REQUIRE(act == EPI_GELU || act == EPI_SILU || act == EPI_SWIGLU, MOE_ERR_INVALID, "mlp_act_backward: activation %d", act);
    MOE_REQUIRE(act != EPI_SWIGLU || F % 32 == 0, MOE_ERR_UNSUPPORTED, "mlp_act_backward: swiglu needs F %% 32 == 0");
    if (rows == 0) return MOE_OK;
    MOE_REQUIRE(a1 && dh && d_a1, MOE_ERR_INVALID, "mlp_act_backward: null pointer");
    hipStream_t s = (hipStream_t)stream;
    if (dtype == MOE_BF16 && F % 8 == 0 && aligned16(a1) && aligned16(dh) && aligned16(d_a1)) {
        const int F8 = F / 8, chunk = (int)std::min<long long>(rows, (1ll << 31) / F8);  // rows per launch: 32-bit indices
        for (int r0 = 0; r0 < rows; r0 += chunk) {
            const unsigned total = (unsigned)std::min(chunk, rows - r0) * (unsigned)F8;
            const int blocks = (int)std::min<unsigned>((total + 255) / 256, (unsigned)num_cus() * 32);
            const size_t off = (size_t)r0 * F8, off1 = off * (act == EPI_SWIGLU ? 2 : 1);
#define GG_ACTV(EPIv) act_backward_vec_kernel<EPIv><<<blocks, 256, 0, s>>>((const uint4*)a1 + off1, (const uint4*)dh + off, (uint4*)d_a1 + off1, total, F8)
            if (act == EPI_GELU) GG_ACTV(EPI_GELU);
            else if (act == EPI_SILU) GG_ACTV(EPI_SILU);
            else GG_ACTV(EPI_SWIGLU);
#undef GG_ACTV
        }
        return moe_check_launch("mlp_act_backward");
    }
    const int blocks = (int)std::min<size_t>(((size_t)rows * F + 255) / 256, (size_t)num_cus() * 32);
#define GG_ACTB(EPIv, Tv) act_backward_kernel<EPIv, Tv><<<blocks, 256, 0, s>>>((const Tv*)a1, (const Tv*)dh, (Tv*)d_a1, (size_t)rows, F)
    if (dtype == MOE_F32) {
        if (act == EPI_GELU) GG_ACTB(EPI_GELU, float);
        else GG_ACTB(EPI_SILU, float);
    } else if (act == EPI_GELU) GG_ACTB(EPI_GELU, bf16_t);
    else if (act == EPI_SILU) GG_ACTB(EPI_SILU, bf16_t);
    else GG_ACTB(EPI_SWIGLU, bf16_t);
#undef GG_ACTB
    return moe_check_launch("mlp_act_backward");
}
