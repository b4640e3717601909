// Grouped GEMM for launches that do not fill the chip with large tiles: small batches, generation, short training batches.
//
// Same operands, packed weights and epilogues as grouped_gemm.hip (bf16 and OCP fp8, row maps on either side, activations,
// kept pre-activations, block-quantised hidden activations).  What differs is the shape of the work: one tile of BM x 128
// outputs per workgroup of four waves, several workgroups per compute unit (the barriers and epilogues of one run under the
// MFMAs of the others), a plain ring of LDS stages, and the K range of every tile cut into P parts when there are fewer tiles
// than workgroups the chip can hold.  The parts of a tile leave their fp32 sums in the workspace; the workgroup that finishes
// last adds them in part order (so the result does not depend on who that is) and applies the epilogue: one launch, where
// the large-tile path needs a launch for whole tiles, one for the parts and one for their reduction.  Where every tile has a compute unit
// to itself, two sets of four waves share one (KG = 2): pairs of stages in turn, each set through its own ring, the sums added at the end.
#include "gg_common.h"
#include <algorithm>
#include <atomic>
#include <math.h>
#include <time.h>
#include <type_traits>

namespace moe_gg {

constexpr int GS_BN = 128;
constexpr int GS_THREADS = 256;
constexpr int GS_CTR_BYTES = 16384;  // arrival counters at the start of the workspace: one 64-bit word per tile
constexpr int GS_MIN_PART_STAGES = 32;  // K stages per part at least: what the hand-over of a split tile costs is worth about as many
static_assert((2 * GS_MIN_PART_STAGES - 2) * ROWB == MOE_SPLIT_MIN_K_BYTES, "(two parts, the second a pair of stages shorter: what the header tells callers)");
constexpr int GS_PART_BYTES = 8 << 20;  // room for parts that a launch uses at most: splits beyond that cost more than they give
constexpr int GS_LDO = GS_BN + 4;    // pitch of the epilogue's fp32 tile in LDS

template <int BM>
struct GsShape {
    static constexpr int WM = BM == 32 ? 1 : 2, WN = 4 / WM;  // waves along rows and columns
    static constexpr int WR = BM / WM, WC = GS_BN / WN;       // rows and columns of a wave
    static constexpr int NST = 3;                             // ring slots, a pair of 64-byte stages each (two workgroups fit a compute unit)
    static constexpr int RA = BM / 32;                        // activation loads per wave and pair of stages (1 KB each)
    static constexpr int RB = GS_BN / 64;                     // weight loads per wave and stage
};
template <int BM, bool BSA, int KG>
constexpr int gs_lds_bytes() {
    using S = GsShape<BM>;
    const int ring = KG * (S::NST * (BM + GS_BN) * 2 * ROWB + (BSA ? 4 * S::NST * 256 : 0));
    const int epi = BM * GS_LDO * 4;
    return ring > epi ? ring : epi;
}

struct GsParams {
    GemmParams g;
    int ncols;                 // packed columns that exist (N, or 2 N for SwiGLU)
    int slots;                 // units up to which tiles are split: one workgroup per compute unit
    unsigned long long nonce;  // what this launch's arrival counters carry in their upper bits
    int big_bm, big_grid;      // the tail of a launch of large tiles of big_bm rows (g.tail_max); 0: all rows
};

// How many parts every tile's K range is cut into.
__host__ __device__ inline int gs_parts(long long tiles, int slots, int nk, int max_units) {
    const int most = slots < max_units ? slots : max_units;
    if (tiles <= 0 || 2 * tiles > most) return 1;  // (nothing to divide: a launch of small tiles is short enough to see the division)
    int P = most / (int)tiles < GG_MAX_PARTS ? most / (int)tiles : GG_MAX_PARTS;
    while (P > 1 && (gg_part_stages(nk, P) < GS_MIN_PART_STAGES || (P - 1) * gg_part_stages(nk, P) >= nk)) --P;
    return P;
}

template <int BM, bool FP8, int EPI, bool BSA, int BMODE, bool TAIL, int KG>
__global__ __launch_bounds__(GS_THREADS * KG, 2) void gemm_small_kernel(const GsParams q) {
    constexpr bool BT = BMODE == GG_B_T, BN_PAIR = BMODE == GG_B_NP, BN_RAW = BMODE == GG_B_N || BN_PAIR;  // (see GG_B_*)
    static_assert(!FP8 || BMODE == GG_B_PACKED, "raw weights are a bf16 matter");
    using S = GsShape<BM>;
    constexpr int ES = FP8 ? 1 : 2;
    constexpr int MT = FP8 ? 32 : 16, CF = FP8 ? 2 : 1;
    constexpr int TM = S::WR / MT, TN = S::WC / MT;
    constexpr int NST = S::NST, RA = S::RA, RB = S::RB;
    constexpr int LPS = RA + 2 * RB + (BSA ? 1 : 0);  // loads per wave and pair
    constexpr int ASZ = BM * ROWB, BSZ = GS_BN * ROWB;  // bytes of a stage (a ring slot holds two)
    constexpr bool QOUT = FP8 && EPI == EPI_SWIGLU;
    static_assert(TM >= 1 && TN >= 1, "wave tile");
    extern __shared__ __align__(1024) uint8_t lds[];
    __shared__ int s_last;
    const GemmParams& p = q.g;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3, kg = KG > 1 ? __builtin_amdgcn_readfirstlane(tid >> 8) : 0;  // (of the set; the set)
    constexpr int NTH = GS_THREADS * KG;
    const int wm = wave / S::WN, wn = wave % S::WN;

    // ---- this workgroup's unit: group, column tile, row tile, part.  Every wave scans the row counts by itself (64 groups at
    // a time); counts that claim more rows than the buffers hold are cut at S_rows.
    // TAIL: the tiles are those of a launch of large tiles that fill no round of its grid, each cut into tiles of this kernel.
    const int nt_all = TAIL ? p.Npad / GG_BN : (q.ncols + GS_BN - 1) / GS_BN;  // (TAIL: large tiles)
    const int tm = TAIL ? q.big_bm : BM, subs = TAIL ? tm / BM * (GG_BN / GS_BN) : 1;
    int mt_all = 0;
    GgRows gr;
    int mt, ti;  // row tiles of the lane's group, and of the groups up to it
    {
        int rows = 0;
        for (int g0 = 0; g0 < p.E_l; g0 += WAVE) {
            gr = gg_rows<false>(p.cnt, g0 + lane, p.E_l, rows, p.S_rows);
            mt = (gr.n + tm - 1) / tm;
            ti = wave_incl_scan(mt);
            mt_all += wave_lane(ti, WAVE - 1);
            rows = gr.end;
        }
        if constexpr (!FP8) gg_zero_tail(p, rows);
    }
    const int nk = (p.K * ES) / ROWB;
    // the launch's tiles [first, first + tiles / subs) of mt_all * nt_all
    const int first = TAIL ? gg_whole_tiles(mt_all * nt_all, q.big_grid, p.tail_max) : 0;
    const int tiles = __builtin_amdgcn_readfirstlane((mt_all * nt_all - first) * subs);
    const int P = __builtin_amdgcn_readfirstlane(p.part_ws ? gs_parts(tiles, q.slots, nk, p.max_units) : 1);
    const int units = tiles * P;
    // consecutive units share an XCD (workgroups b, b + 8, ... do): parts of a tile, then the row tiles of a weight panel
    const int per = (units + 7) / 8;
    const int unit = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (((int)blockIdx.x >> 3) >= per || unit >= units) return;
    int tile = unit, part = 0;
    if (P > 1) { tile = unit / P; part = unit - tile * P; }
    const int whole = first + tile / subs;
    int g = 0, row0 = 0, rv = 0, nt = 0;
    {
        int rows = 0, before = 0;
        for (int g0 = 0; g0 < p.E_l; g0 += WAVE) {
            if (p.E_l > WAVE) {  // (else the lanes hold their groups as they are)
                gr = gg_rows<false>(p.cnt, g0 + lane, p.E_l, rows, p.S_rows);
                mt = (gr.n + tm - 1) / tm;
                ti = wave_incl_scan(mt);
            }
            const int t0 = (before + ti - mt) * nt_all;
            const unsigned long long hit = __ballot(mt > 0 && whole >= t0 && whole < t0 + mt * nt_all);
            if (hit) {
                const int l = __builtin_ctzll(hit);
                const int mt_g = wave_lane(mt, l), in = whole - wave_lane(t0, l);
                g = g0 + l;
                int m = 0;
                nt = in;
                if (mt_g > 1) { nt = in / mt_g; m = in - nt * mt_g; }
                if constexpr (TAIL) {
                    gg_patch(in, mt_g, nt_all, tm == 128 ? SUP_DUO : SUP, m, nt);
                    nt = nt * (GG_BN / GS_BN) + tile % (GG_BN / GS_BN);
                }
                const int r = m * tm + (TAIL ? tile % subs / (GG_BN / GS_BN) * BM : 0);
                row0 = wave_lane(gr.start, l) + r;
                rv = min(BM, wave_lane(gr.n, l) - r);
                break;
            }
            rows = gr.end;
            before += wave_lane(ti, WAVE - 1);
        }
    }
    if (TAIL && (rv <= 0 || nt * GS_BN >= q.ncols)) return;  // (past the rows or columns; all parts of the tile alike)
    g = __builtin_amdgcn_readfirstlane(g); nt = __builtin_amdgcn_readfirstlane(nt);
    row0 = __builtin_amdgcn_readfirstlane(row0); rv = __builtin_amdgcn_readfirstlane(rv);
    const int nkp = P > 1 ? gg_part_stages(nk, P) : nk;
    const int ks0 = part * nkp, nks = min(nkp, nk - ks0);

    // ---- addresses.  LDS tiles: weights as in the large kernel, 64-byte rows, chunk c of row r at position c ^ gg_swz(r >> 2);
    // activations a pair of stages at a time, 128-byte rows, chunk c of row r at position c ^ gg_swz_wide(r) (in 64-byte pieces, a stage at a
    // time: 1724 rows x 4096 x 1024 in two groups 24.9 us, now 24.0; 1003 x 4096 x 2048 36 -> 34; 200 x 1024 x 1024 7.2 -> 6.9).
    const int lchunk = (lane & 3) ^ gg_swz(lane >> 4);
    const uint32_t ldk = (uint32_t)(p.K * ES);
    const uint8_t* Ab = (p.a_map ? p.A : p.A + (size_t)row0 * ldk) + (size_t)ks0 * ROWB;
    // weights: bytes from one stage to the next, from the start of the tensor to the tile's first stage, and (not re-tiled) of a tensor
    [[maybe_unused]] const bool pair = p.B2 != nullptr;
    [[maybe_unused]] const uint32_t ldb = BT ? (uint32_t)(pair ? p.K / 2 : p.K) * 2u : (uint32_t)p.N * 2u;
    [[maybe_unused]] const size_t b_group = (size_t)p.K / (BT && pair ? 2 : 1) * p.N * 2;
    [[maybe_unused]] const ptrdiff_t b2_delta = p.B2 - p.B;
    const size_t b_slab = BT ? (size_t)ROWB : BN_RAW ? (size_t)32 * ldb : (size_t)p.Npad * ROWB;
    const size_t b_at = BT ? (size_t)g * b_group + (size_t)nt * GS_BN * ldb + (size_t)ks0 / (pair ? 2 : 1) * ROWB
                      : BN_RAW ? (size_t)g * b_group + (size_t)nt * (BN_PAIR ? GS_BN : 2 * GS_BN) + (size_t)ks0 * b_slab
                               : (size_t)g * p.Npad * ldk + (size_t)nt * GS_BN * ROWB + (size_t)ks0 * b_slab;
    const uint8_t* Bb = p.B + b_at;
    [[maybe_unused]] const long long b_left = (long long)p.E_l * b_group - (long long)b_at;
    uint32_t aoff[RA], boff[RB];
    int arow[RA];  // (of the lane's rows: all under way together)
#pragma unroll
    for (int r = 0; r < RA; ++r) arow[r] = min((r * 4 + wave) * 8 + (lane >> 3), rv - 1);
    if (p.a_map) {
#pragma unroll
        for (int r = 0; r < RA; ++r) arow[r] = p.a_map[row0 + arow[r]];
    }
#pragma unroll
    for (int r = 0; r < RA; ++r) aoff[r] = (uint32_t)max(arow[r], 0) * ldk + ((lane & 7) ^ gg_swz_wide((r * 4 + wave) * 8 + (lane >> 3))) * 16;
#pragma unroll
    for (int r = 0; r < RB; ++r) {
        if constexpr (BT) boff[r] = (uint32_t)gg_packed_col<false>(r * 64 + wave * WROWS + (lane >> 2)) * ldb + lchunk * 16;
        // BN_RAW: a stage is 32 rows of 256 bytes, four to a 1 KB load, chunk c of row k at position c ^ 4 (k % 4); a pair: 32 rows of
        // 128 bytes of either matrix, eight to a load, chunk c at position c ^ 4 (k / 2 % 2)
        else if constexpr (BN_PAIR) boff[r] = (uint32_t)(8 * wave + (lane >> 3)) * ldb + (uint32_t)((lane & 7) ^ (4 * ((lane >> 4) & 1))) * 16u;
        else if constexpr (BN_RAW) boff[r] = (uint32_t)(4 * (r * 4 + wave) + (lane >> 4)) * ldb + (uint32_t)((lane & 15) ^ (4 * (lane >> 4))) * 16u;
        else boff[r] = (uint32_t)(r * 64 + wave * WROWS + (lane >> 2)) * ROWB + lchunk * 16;
    }
    static_assert(!BN_RAW || RB == 2, "two loads per wave and stage");
    uint8_t* const sA = lds + kg * (gs_lds_bytes<BM, BSA, KG>() / KG);
    uint8_t* const sB = sA + NST * 2 * ASZ;
    uint32_t* const sS = (uint32_t*)(sA + NST * 2 * (ASZ + BSZ)) + wave * NST * 64;  // (BSA) the wave's scale dwords, one per row
    const uint32_t la0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)sA) + wave * 1024;
    const uint32_t lb0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)sB) + wave * WROWS * ROWB;
    [[maybe_unused]] const uint32_t ls0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)sS);
    [[maybe_unused]] const uint32_t soff = BSA ? (uint32_t)(row0 + min(wm * S::WR + (lane & (S::WR - 1)), rv - 1)) * (uint32_t)p.bs_pitch : 0u;

    const int npair = nks / 2, mine = (npair + KG - 1 - kg) / KG, steps = (npair + KG - 1) / KG;  // pairs of the set (kg, kg + KG, ...), steps of all
    // load d (0 .. LPS - 1) of the pair whose first stage lies at ap / bp: activations, weights, (BSA) scale dwords
    // (bp[stage][matrix of a pair])
    typedef typename std::conditional<BMODE == GG_B_PACKED, const uint8_t*, gg_i32x4>::type bsrc_t;
    auto load = [&](int d, const uint8_t* ap, const bsrc_t (&bp)[2][2], const uint8_t* sp, int slot) {
        if (d < RA) gg_dma16(ap, aoff[d], la0 + slot * 2 * ASZ + d * 4096);
        else if (d < RA + 2 * RB) {
            const int e = d - RA;
            gg_dma16(bp[e / RB][BN_PAIR ? e % RB : 0], boff[e % RB], lb0 + slot * 2 * BSZ + (e / RB) * BSZ + (e % RB) * 64 * ROWB);
        } else if constexpr (BSA) gg_dma4(sp, soff, ls0 + slot * 256);
    };
#define GS_PAIR_PTRS(pr)                                                    \
    const int st_ = 2 * min((pr) * KG + kg, npair - 1);                     \
    const uint8_t* ap_ = gg_uniform(Ab + (size_t)st_ * ROWB);               \
    bsrc_t bp_[2][2];                                                       \
    _Pragma("unroll") for (int u_ = 0; u_ < 2; ++u_)                         \
        _Pragma("unroll") for (int m_ = 0; m_ < (BN_PAIR ? 2 : 1); ++m_) {   \
            const size_t so_ = BT && pair ? (size_t)(st_ >> 1) * ROWB : (size_t)(st_ + u_) * b_slab; \
            if constexpr (BMODE == GG_B_PACKED) bp_[u_][m_] = gg_uniform(Bb + so_);                  \
            else bp_[u_][m_] = gg_range((BN_PAIR ? m_ : BT && pair && u_) ? Bb + b2_delta + so_ : Bb + so_, b_left - (long long)so_); \
        }                                                                   \
    const uint8_t* sp_ = BSA ? gg_uniform(p.a_bscale + (((ks0 + st_) >> 1) << 2)) : nullptr;

    typedef typename std::conditional<FP8, floatx16, floatx4>::type acc_t;
    acc_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < (FP8 ? 16 : 4); ++v) acc[i][j][v] = 0.f;

    // ---- K loop.  While a pair of stages is multiplied, the fragments of the next one are read into the other set of registers
    // and the pair NST behind it is requested into the slot that has just been read out; one barrier per pair (it says that the
    // next pair's loads of every wave have landed and that nobody reads the slot the new loads go to any more).
    const int fpos = (FP8 ? (lane >> 5) : (lane >> 4)) ^ gg_swz(lane >> 2);
    const uint4* fa = (const uint4*)sA + (wm * S::WR + (lane & (MT - 1))) * 2 * CHUNKS;
    const int fpos_a = (FP8 ? (lane >> 5) : (lane >> 4)) ^ gg_swz_wide(lane);  // (rows of a fragment start at multiples of 16)
    const uint4* fb = (const uint4*)sB + (wn * S::WC + (lane & (MT - 1))) * CHUNKS;
    // (BN_RAW) LDS address of the lane's part of the first of the two fragments of each group of 32 columns (see gg_read_tr)
    constexpr int BTR = BN_PAIR ? 128 : 256;
    [[maybe_unused]] uint32_t trb[TN > 1 ? TN / 2 : 1];
    if constexpr (BN_RAW) {
        const int kq = (lane >> 4) * 8 + ((lane & 15) >> 2), k4 = (lane & 15) >> 2, q4 = lane & 3;
#pragma unroll
        for (int h = 0; h < TN / 2; ++h) {
            const int grp = wn * (S::WC / 32) + h;
            trb[h] = (uint32_t)(uintptr_t)(lds_ptr_t)sB + kq * BTR +
                     (BN_PAIR ? (grp & 1) * (BSZ / 2) + ((((grp >> 1) * 4 + q4) ^ (4 * (k4 >> 1))) * 16) : (((grp * 4 + q4) ^ (4 * k4)) * 16));
        }
    }
    struct Frag {
        uint4 a[2][TM][CF], b[2][TN][CF];
        uint32_t sc[TM];
    } f0, f1;
    auto read = [&](Frag& f, int slot) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint4* as = fa + slot * (2 * ASZ / 16);
            const uint4* bs = fb + (slot * 2 + u) * (BSZ / 16);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if constexpr (BN_RAW) {
                    const uint32_t at = trb[j >> 1] + (slot * 2 + u) * BSZ + (j & 1) * 8;
                    const uint2 lo = gg_read_tr<BTR>(at, 0), hi = gg_read_tr<BTR>(at, 1);
                    f.b[u][j][0] = make_uint4(lo.x, lo.y, hi.x, hi.y);
                } else {
#pragma unroll
                    for (int h = 0; h < CF; ++h) f.b[u][j][h] = bs[j * MT * CHUNKS + (fpos ^ (2 * h))];
                }
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int h = 0; h < CF; ++h) f.a[u][i][h] = as[i * MT * 2 * CHUNKS + (fpos_a ^ (CHUNKS * u + 2 * h))];
        }
        if constexpr (BSA) {
            // lane 32 h + r: the scale bytes of row r, block h of either stage (see mma_fp8_k64_bs), in bytes 0 and 2
#pragma unroll
            for (int i = 0; i < TM; ++i)
                f.sc[i] = ((sS[slot * 64 + i * MT + (lane & 31)] >> ((lane >> 5) * 8)) & 0x00ff00ffu) + (uint32_t)(127 - GG_WSCALE) * 0x00010001u;
        }
    };
#pragma unroll
    for (int d = 0; d < NST; ++d) {
        GS_PAIR_PTRS(d)
#pragma unroll
        for (int l = 0; l < LPS; ++l) load(l, ap_, bp_, sp_, d);
    }
    gg_wait<(NST - 1) * LPS, 0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(f0, 0);
    int slot = 0;
    // The loads go between the MFMAs: issued in one go they keep the wave from its MFMAs for as long as the load path needs
    // to take them (64 bytes a cycle and compute unit).
    auto step = [&](const Frag& f, Frag& nxt, int s) {
        asm volatile("" ::: "memory");
        gg_wait<(NST - 2) * LPS, 0>();
        __builtin_amdgcn_s_barrier();
        GS_PAIR_PTRS(s + NST)
        const int fill = slot;
        slot = slot == NST - 1 ? 0 : slot + 1;
        asm volatile("" ::: "memory");
        read(nxt, slot);
        __builtin_amdgcn_sched_barrier(0);
        if (KG > 1 && s >= mine) return;  // (an odd number of pairs: this set has none left)
        constexpr int NM = 2 * TM * TN, STEP = NM / LPS > 0 ? NM / LPS : 1, PER = (LPS + NM - 1) / NM;  // MFMAs per load, loads per MFMA
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const int u = m / (TM * TN), i = (m % (TM * TN)) / TN, jj = m % TN, j = (i & 1) ? TN - 1 - jj : jj;
            if constexpr (FP8 && BSA) {
                if (u == 0) mma_fp8_k64_bs<false, 0>(acc[i][j], f.b[u][j][0], f.b[u][j][CF - 1], f.a[u][i][0], f.a[u][i][CF - 1], (int)f.sc[i]);
                else mma_fp8_k64_bs<false, 2>(acc[i][j], f.b[u][j][0], f.b[u][j][CF - 1], f.a[u][i][0], f.a[u][i][CF - 1], (int)f.sc[i]);
            } else if constexpr (FP8) mma_fp8_k64(acc[i][j], f.b[u][j][0], f.b[u][j][CF - 1], f.a[u][i][0], f.a[u][i][CF - 1]);
            else mma_bf16_k32(acc[i][j], f.b[u][j][0], f.a[u][i][0]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < PER; ++e) {
                const int d = PER > 1 ? m * PER + e : m % STEP == 0 ? m / STEP : LPS;
                if (d < LPS) load(d, ap_, bp_, sp_, fill);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int s = 0; s < steps; s += 2) {
        step(f0, f1, s);
        if (s + 1 < steps) step(f1, f0, s + 1);
    }
    asm volatile("" ::: "memory");
    gg_wait<0, 0>();
    __syncthreads();

    // ---- epilogue, row by row: the accumulators change into row-major order in LDS, then a thread takes eight consecutive output
    // columns of a row.  Parts write their sums to the workspace instead; the last one of a tile goes through the same code
    // with the sums read back from there.
    float* const so = (float*)lds;
    constexpr int OCW = EPI == EPI_SWIGLU ? GS_BN / 2 : GS_BN;  // output columns of the tile
    constexpr int TPR = OCW / 8, RPP = NTH / TPR;         // threads per row, rows per pass
    const int oc = (tid % TPR) * 8;                              // the thread's first output column inside the tile
    const int pc = EPI == EPI_SWIGLU ? (oc / 32) * 64 + oc % 32 : oc;  // its packed column inside the tile
    const int gp = nt * GS_BN + pc;
    const int col = EPI == EPI_SWIGLU ? (gp / 64) * 32 + gp % 32 : gp;
    float cg[8], cu[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) cg[e] = cu[e] = 1.f;
    if constexpr (FP8) {
        if (col < p.N) {
            const float4* c0 = (const float4*)(p.col_scale + (size_t)g * p.ncs + col);
            const float4 u0 = c0[0], u1 = c0[1];
            cg[0] = u0.x; cg[1] = u0.y; cg[2] = u0.z; cg[3] = u0.w; cg[4] = u1.x; cg[5] = u1.y; cg[6] = u1.z; cg[7] = u1.w;
            if constexpr (EPI == EPI_SWIGLU) {
                const float4* c1 = (const float4*)(p.col_scale2 + (size_t)g * p.ncs + col);
                const float4 v0 = c1[0], v1 = c1[1];
                cu[0] = v0.x; cu[1] = v0.y; cu[2] = v0.z; cu[3] = v0.w; cu[4] = v1.x; cu[5] = v1.y; cu[6] = v1.z; cu[7] = v1.w;
            }
        }
    }
    auto finish = [&](int r, const float* x0, const float* x1) {  // row r of the tile; x0: the eight (gate) sums, x1: the up sums
        const int grow = row0 + min(r, rv - 1);
        const int crow = p.c_map ? p.c_map[grow] : grow;
        float rs = 1.f;
        if constexpr (FP8 || EPI == EPI_GATE) rs = p.row_scale ? p.row_scale[grow] : 1.f;
        float y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float v = x0[e];
            if constexpr (FP8) v *= cg[e] * rs;
            if constexpr (!FP8 && EPI == EPI_GATE) v *= rs;
            if constexpr (EPI == EPI_SWIGLU) {
                float u = x1[e];
                if constexpr (FP8) u *= cu[e] * rs;
                v = act_silu_fast(v) * u;
            }
            if constexpr (EPI == EPI_GELU) v = act_gelu(v);
            if constexpr (EPI == EPI_SILU) v = act_silu_fast(v);
            y[e] = v;
        }
        if constexpr (QOUT) {  // four threads hold a block of 32 columns: one scale byte, 32 codes
            float am = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) am = fmaxf(am, fabsf(y[e]));
            if (col >= p.N) am = 0.f;
            am = fmaxf(am, __shfl_xor(am, 1, WAVE));
            am = fmaxf(am, __shfl_xor(am, 2, WAVE));
            const int sbyte = gg_block_scale_byte(__float_as_uint(am));
            const float inv = __uint_as_float(gg_block_inv_bits(sbyte));
            int lo = 0, hi = 0;
            lo = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(y[0], inv), __fmul_rn(y[1], inv), lo, false);
            lo = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(y[2], inv), __fmul_rn(y[3], inv), lo, true);
            hi = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(y[4], inv), __fmul_rn(y[5], inv), hi, false);
            hi = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(y[6], inv), __fmul_rn(y[7], inv), hi, true);
            if (r < rv && crow >= 0 && col < p.N) {
                *(uint2*)((uint8_t*)p.C + (size_t)crow * p.ldc + col) = make_uint2((uint32_t)lo, (uint32_t)hi);
                if ((col & 31) == 0) p.c_bscale[(size_t)crow * p.bs_pitch + col / 32] = (uint8_t)sbyte;
            }
            return;
        }
        if (r >= rv || crow < 0 || col >= p.N) return;
        *(uint4*)((bf16_t*)p.C + (size_t)crow * p.ldc + col) =
            make_uint4(gg_pack_bf16(y[0], y[1]), gg_pack_bf16(y[2], y[3]), gg_pack_bf16(y[4], y[5]), gg_pack_bf16(y[6], y[7]));
        if constexpr (!FP8 && EPI != EPI_NONE && EPI != EPI_GATE) {
            if (p.C2) {  // the values before the activation (rows are never remapped where they are kept)
                constexpr int W2 = EPI == EPI_SWIGLU ? 2 : 1;
                bf16_t* r2 = (bf16_t*)p.C2 + (size_t)crow * p.ldc * W2 + (EPI == EPI_SWIGLU ? gp : col);
                *(uint4*)r2 = make_uint4(gg_pack_bf16(x0[0], x0[1]), gg_pack_bf16(x0[2], x0[3]), gg_pack_bf16(x0[4], x0[5]), gg_pack_bf16(x0[6], x0[7]));
                if constexpr (EPI == EPI_SWIGLU)
                    *(uint4*)(r2 + 32) = make_uint4(gg_pack_bf16(x1[0], x1[1]), gg_pack_bf16(x1[2], x1[3]), gg_pack_bf16(x1[4], x1[5]), gg_pack_bf16(x1[6], x1[7]));
            }
        }
    };
    float* const ws = P > 1 ? (float*)((uint8_t*)p.part_ws + GS_CTR_BYTES) : nullptr;
    constexpr int NQ = FP8 ? 4 : 1;
#pragma unroll
    for (int set = KG - 1; set >= 0; --set) {  // (the second set leaves its sums, the first adds its own)
        if (set == kg) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < NQ; ++v) {
                        // four consecutive rows of the weight tile are four consecutive columns
                        const int r = wm * S::WR + i * MT + (lane & (MT - 1));
                        const int c = gg_packed_col<FP8>(wn * S::WC + j * MT + (FP8 ? 8 * v + 4 * (lane >> 5) : 4 * (lane >> 4)));
                        float4* const at = (float4*)(so + r * GS_LDO + c);
                        float4 a = make_float4(acc[i][j][4 * v], acc[i][j][4 * v + 1], acc[i][j][4 * v + 2], acc[i][j][4 * v + 3]);
                        if (KG > 1 && set == 0) {
                            const float4 b = *at;
                            a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
                        }
                        *at = a;
                    }
        }
        __syncthreads();
    }
    // (whole passes of RPP rows: the threads that hold a block of columns of a row stay together)
    const int r_end = min((rv + RPP - 1) & ~(RPP - 1), BM);
    if (P == 1) {
        for (int r = tid / TPR; r < r_end; r += RPP) {
            float x0[8], x1[8];
            *(float4*)x0 = *(const float4*)(so + r * GS_LDO + pc);
            *(float4*)(x0 + 4) = *(const float4*)(so + r * GS_LDO + pc + 4);
            if constexpr (EPI == EPI_SWIGLU) {
                *(float4*)x1 = *(const float4*)(so + r * GS_LDO + pc + 32);
                *(float4*)(x1 + 4) = *(const float4*)(so + r * GS_LDO + pc + 36);
            }
            finish(r, x0, x1);
        }
        return;
    }
    unsigned long long* const o = (unsigned long long*)(ws + (size_t)unit * (BM * GS_BN));
    for (int i = tid; i < rv * (GS_BN / 2); i += NTH)
        __hip_atomic_store(o + i, *(const unsigned long long*)(so + (i / (GS_BN / 2)) * GS_LDO + 2 * (i % (GS_BN / 2))), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    // arrival: the sums above are written through to memory; once they are acknowledged the part counts itself in.  The
    // counter starts from whatever the workspace holds: only a word that carries this launch's nonce counts.
    gg_wait<0, 0>();
    __syncthreads();
    if (tid == 0) {
        unsigned long long* ctr = (unsigned long long*)p.part_ws + tile;
        unsigned long long seen = __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        while ((seen >> 8) != q.nonce)  // the first to arrive starts the count (once it has, the others add to it without a retry)
            if (__hip_atomic_compare_exchange_strong(ctr, &seen, q.nonce << 8, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
        const bool last = (int)(__hip_atomic_fetch_add(ctr, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 255) == P - 1;
        // (the last part leaves a word without the nonce: a replay of a captured launch carries the same one)
        if (last) __hip_atomic_store(ctr, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = last;
    }
    __syncthreads();
    if (!s_last) return;
    const float* w0 = ws + (size_t)tile * P * (BM * GS_BN);
    for (int r = tid / TPR; r < r_end; r += RPP) {
        float x0[8], x1[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x0[e] = x1[e] = 0.f;
        if (r < rv) {
            const unsigned long long* w = (const unsigned long long*)(w0 + (size_t)r * GS_BN + pc);
            constexpr int NV = EPI == EPI_SWIGLU ? 8 : 4, PU = 32 / NV;  // 64-bit loads per part; parts requested together
            for (int k0 = 0; k0 < P; k0 += PU) {
                unsigned long long v[PU][NV];
#pragma unroll
                for (int k = 0; k < PU; ++k)
                    if (k0 + k < P)
#pragma unroll
                        for (int e = 0; e < NV; ++e)
                            v[k][e] = __hip_atomic_load(w + (size_t)(k0 + k) * (BM * GS_BN / 2) + (e & 3) + (e >> 2) * 16, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                for (int k = 0; k < PU; ++k)
                    if (k0 + k < P)
#pragma unroll
                        for (int e = 0; e < NV; ++e) {
                            float* x = (e >> 2 ? x1 : x0) + 2 * (e & 3);
                            x[0] += __uint_as_float((uint32_t)v[k][e]);
                            x[1] += __uint_as_float((uint32_t)(v[k][e] >> 32));
                        }
            }
        }
        finish(r, x0, x1);
    }
}

// A number no earlier launch of this process used (and no stale workspace word is likely to hold): 56 bits.
static unsigned long long gs_nonce() {
    static const unsigned long long base = [] {
        unsigned long long z = (unsigned long long)(uintptr_t)&gs_nonce ^ (unsigned long long)clock() * 0x9e3779b97f4a7c15ull;
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        return (z ^ (z >> 31)) | (1ull << 40);
    }();
    static std::atomic<unsigned long long> n{0};
    return (base + n.fetch_add(1, std::memory_order_relaxed)) & ((1ull << 56) - 1);
}

// Part tiles of bm rows that a launch may use: one per compute unit at most, as many as the workspace has room and counters for.
static int gs_slots(int bm, int cus) { return (int)std::min<long long>(cus, GS_PART_BYTES / (bm * GS_BN * 4)); }
static int gs_max_units(int bm, const void* part_ws, size_t bytes) {
    if (!part_ws || bytes <= (size_t)GS_CTR_BYTES) return 0;
    return (int)std::min<long long>((long long)(bytes - GS_CTR_BYTES) / (bm * GS_BN * 4), GS_CTR_BYTES / 8);
}

int gs_plan_parts(long long tiles, int bm, int nk, int cus, const void* part_ws, size_t bytes) {
    const int room = gs_max_units(bm, part_ws, bytes);
    return room ? gs_parts(tiles, gs_slots(bm, cus), nk, room) : 1;
}

template <int BM, bool FP8, int EPI, bool BSA, int BMODE>
static void gs_launch(const GsParams& q0, void* part_ws, size_t part_ws_bytes, int cus, hipStream_t s) {
    GsParams q = q0;
    q.slots = gs_slots(BM, cus);
    q.g.max_units = gs_max_units(BM, part_ws, part_ws_bytes);
    q.g.part_ws = q.g.max_units ? (float*)part_ws : nullptr;
    const int nt = (q.ncols + GS_BN - 1) / GS_BN;
    const long long ub = ((long long)q.g.S_rows + (long long)std::min(q.g.E_l, q.g.S_rows) * (BM - 1)) / BM * nt;  // most tiles there can be
    auto units = [&](long long tiles) {
        return (unsigned)((std::max<long long>(tiles, q.g.part_ws ? std::min<long long>(q.slots, tiles * GG_MAX_PARTS) : 0) + 7) / 8 * 8);
    };
    q.nonce = gs_nonce();
    if constexpr (BM == 64) {
        if (q.big_bm) {
            gemm_small_kernel<BM, FP8, EPI, BSA, BMODE, true, 1><<<units((long long)q.g.tail_max * (q.big_bm / BM) * (GG_BN / GS_BN)), GS_THREADS, gs_lds_bytes<BM, BSA, 1>(), s>>>(q);
            return;
        }
    }
    // Two sets of waves to a tile where every tile has a compute unit to itself: what bounds such a launch is how long the weights take to come, and two sets
    // have twice as many stages under way.  Weights from memory: 443 rows of two groups x 2048 x 4096 19.4 -> 18.3 us, x 4096 x 2048 24.6 -> 22.9, 482 of 2 x 3840 x 1664
    // 25.8 -> 22.8; short K gains nothing (1088: 12.0, 12.0) or pays for adding the sets up (576: 7.6 -> 8.1), and so do groups of a few rows
    // (77 rows of 32 x 5440 x 896 50.9 -> 53.8); a second round of such workgroups costs 1.04 to 1.36 times.
    if (ub <= cus && q.g.K * (FP8 ? 1 : 2) >= 54 * ROWB && q.g.S_rows >= 8 * q.g.E_l)
        gemm_small_kernel<BM, FP8, EPI, BSA, BMODE, false, 2><<<units(ub), GS_THREADS * 2, gs_lds_bytes<BM, BSA, 2>(), s>>>(q);
    else
        gemm_small_kernel<BM, FP8, EPI, BSA, BMODE, false, 1><<<units(ub), GS_THREADS, gs_lds_bytes<BM, BSA, 1>(), s>>>(q);
}

template <bool FP8>
static int gs_dispatch(const GsParams& q, int bm, int epi, void* ws, size_t bytes, int cus, hipStream_t s) {
#define GS_MODE(EPIv, BSAv, MODEv)                                                     \
    do {                                                                               \
        if (bm == 32) gs_launch<32, FP8, EPIv, BSAv, MODEv>(q, ws, bytes, cus, s);     \
        else gs_launch<64, FP8, EPIv, BSAv, MODEv>(q, ws, bytes, cus, s);              \
    } while (0)
#define GS_BM(EPIv, BSAv) GS_MODE(EPIv, BSAv, GG_B_PACKED)
    if constexpr (FP8) {
        if (epi == EPI_NONE) GS_BM(EPI_NONE, true);
        else GS_BM(EPI_SWIGLU, false);
    } else if (q.g.b_mode != GG_B_PACKED) {  // weights in the reference layout
        const int mode = q.g.b_mode;
        if (mode == GG_B_T && epi == EPI_NONE) GS_MODE(EPI_NONE, false, GG_B_T);
        else if (mode == GG_B_N && epi == EPI_NONE) GS_MODE(EPI_NONE, false, GG_B_N);
        else if (mode == GG_B_N && epi == EPI_GELU) GS_MODE(EPI_GELU, false, GG_B_N);
        else if (mode == GG_B_N && epi == EPI_SILU) GS_MODE(EPI_SILU, false, GG_B_N);
        else if (mode == GG_B_NP && epi == EPI_SWIGLU) GS_MODE(EPI_SWIGLU, false, GG_B_NP);
        else return moe_fail(MOE_ERR_INVALID, "grouped_gemm: weight mode %d with activation %d", mode, epi);
    } else {
        switch (epi) {
            case EPI_NONE: GS_BM(EPI_NONE, false); break;
            case EPI_GELU: GS_BM(EPI_GELU, false); break;
            case EPI_SILU: GS_BM(EPI_SILU, false); break;
            case EPI_SWIGLU: GS_BM(EPI_SWIGLU, false); break;
            default: GS_BM(EPI_GATE, false); break;
        }
    }
#undef GS_BM
#undef GS_MODE
    return moe_check_launch("grouped_gemm");
}

// What a launch on tiles of bm rows is taken to cost, in us, for gg_choose (grouped_gemm.hip), which says where the coefficients come from: 0.27 / 0.30 us per
// 128 bytes of K while every workgroup has a compute unit to itself, then in proportion to their number (times 1.22 to 1.37: the load path is
// shared), and the hand-over of a split tile.  `tiles`: about as many as there will be.
double gs_estimate(int bm, double tiles, int nk, bool fp8, int cus, const void* part_ws, size_t part_ws_bytes) {
    const int room = std::min(gs_slots(bm, cus), gs_max_units(bm, part_ws, part_ws_bytes));
    const double P = tiles < room ? std::max(1.0, std::min(std::min(floor(room / tiles), floor((double)nk / GS_MIN_PART_STAGES)), (double)GG_MAX_PARTS)) : 1.0;
    const double x = tiles * P / cus;
    if (bm == 32) return nk / 2 / P * 0.27 * std::max(1.0, x * (fp8 ? 1.37 : 1.24)) + 0.5 * std::max(1.0, x / 2) + (P > 1 ? 4 : 0);
    return nk / 2 / P * 0.30 * std::max(1.0, x * (fp8 ? 1.30 : 1.22)) + 1.3 * std::max(1.0, x / 2) + (P > 1 ? 6.5 : 0);
}

size_t gs_workspace_bytes(int cus) { return GS_CTR_BYTES + std::min<size_t>((size_t)cus * 64 * GS_BN * 4, GS_PART_BYTES); }

int launch_gemm_small(const GemmParams& p, bool fp8, int bm, int epi, void* ws, size_t bytes, int cus, hipStream_t s) {
    GsParams q{};
    q.g = p;
    q.ncols = epi == EPI_SWIGLU ? 2 * p.N : p.N;
    return fp8 ? gs_dispatch<true>(q, bm, epi, ws, bytes, cus, s) : gs_dispatch<false>(q, bm, epi, ws, bytes, cus, s);
}

int launch_gemm_tail(const GemmParams& p, bool fp8, int bm_big, int epi, void* ws, size_t bytes, int grid, hipStream_t s) {
    GsParams q{};
    q.g = p;
    q.ncols = epi == EPI_SWIGLU ? 2 * p.N : p.N;
    q.big_bm = bm_big;
    q.big_grid = bm_big == 128 ? 2 * grid : grid;  // (tiles to a round)
    return fp8 ? gs_dispatch<true>(q, 64, epi, ws, bytes, grid, s) : gs_dispatch<false>(q, 64, epi, ws, bytes, grid, s);
}

}  // namespace moe_gg
