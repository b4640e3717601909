// Grouped GEMM for launches that 256-row tiles (grouped_gemm.hip) fill the chip badly with: tiles of 128 x 256, one per workgroup of four waves, two workgroups
// to a compute unit, dealt out by the hardware.
//
// Same operands, packed and raw weights, epilogues and weight-gradient mode as there.  What a persistent workgroup of 256-row tiles pays for every tile -- its
// store, and the first stages and fragments of the next -- runs here beside the other workgroup's K loop; half the rows to a tile lose half as many to the ends of ragged
// groups; and a round is 512 tiles that end when they end.  The price is the load path: a wave's block is 64 x 128, so 1.5 times the bytes go through LDS for the
// same products, and K has three stages in LDS instead of four.  Hence the rule (gg_choose): launches of up to a few rounds, and short K.
// Bound: matrix pipes 0.55 to 0.7 busy at 1.7 to 2.2 GHz, then the load path (0.38 us per 128 bytes of K and two workgroups at the 130 bytes a ns that it takes whole
// lines at, against 0.9 to 1.1 us of products).  Against the better of the other kernels, before: 16384 rows of 8 groups x 2048 x 2048 139 -> 118 us, of 32 groups x 768 x 768 28 -> 24.5;
// 8192 of 4 x 1024 x (2 x 4096) 131 -> 115; 1003 of 2 x 2048 x 4096 31 -> 26.5; fp8 MLP of 1942 x 2048 x 1408 in 15 groups 54 -> 43.5.
#include "gg_common.h"
#include <algorithm>
#include <type_traits>

namespace moe_gg {

constexpr int GD_BM = 128, GD_BN = GG_BN, GD_NST = 3, GD_THREADS = 256;
constexpr int GD_ROUND = 512;  // tiles dealt out to the XCDs at a time

template <int EPI, bool FP8, int BMODE>
__global__ __launch_bounds__(GD_THREADS, 2) void gemm_duo_kernel(const GemmParams p, const int cus) {
    constexpr bool DW = BMODE == GG_B_DW, BT = BMODE == GG_B_T, BN_PAIR = BMODE == GG_B_NP, BN_RAW = BMODE == GG_B_N || BN_PAIR;
    constexpr bool BSA = FP8 && EPI == EPI_NONE, QOUT = FP8 && EPI == EPI_SWIGLU;
    static_assert(!FP8 || BMODE == GG_B_PACKED, "raw weights are a bf16 matter");
    static_assert(!DW || EPI == EPI_NONE, "the weight-gradient mode is a plain GEMM");
    constexpr int ES = FP8 ? 1 : 2, MT = FP8 ? 32 : 16, CF = FP8 ? 2 : 1;
    constexpr int TM = 64 / MT, TN = 128 / MT, NT = TM * TN;
    constexpr int RPA = DW ? 2 : CF, RPB = DW || BN_RAW ? 2 : CF;
    constexpr int NRD = TM * RPA + TN * RPB;
    // Activations come two stages, 128 bytes of their rows, at a time as in grouped_gemm.hip (a stage at a time this kernel took 1.12 to 1.17 times as long), where LDS
    // has room: two slots of pairs and three of weight stages are all of a workgroup's half.
    constexpr bool WIDE = !DW && !BSA;
    constexpr int RA = WIDE ? 4 : 2, RB = 4;           // loads per lane: A, per pair of stages (WIDE) or stage; B, per stage
    constexpr int ASZ = GD_BM * ROWB, BSZ = GD_BN * ROWB, NST = GD_NST, NA = WIDE ? 4 : NST;  // bytes of a stage; slots, in stages
    __shared__ __align__(1024) uint8_t lds[NA * ASZ + NST * BSZ + (BSA ? 4 * 2 * 64 * 4 : 0)];
    uint8_t* const sA = lds;
    uint8_t* const sB = lds + NA * ASZ;
    uint32_t* const s_hsc = (uint32_t*)(lds + NA * ASZ + NST * BSZ);  // (BSA) a wave's scale dwords of two pairs of stages, one per row
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int Nt = p.Npad / GD_BN;
    const int src_rows = DW ? p.dw_src_rows : p.S_rows;

    // ---- this workgroup's tile
    const int dmt = DW ? (p.dw_rows + GD_BM - 1) / GD_BM : 0;
    GgRows gr;
    int mt, ti, mt_all = 0;
    {
        int rows = 0;
        for (int g0 = 0; g0 < p.E_l; g0 += WAVE) {
            gr = gg_rows<false>(p.cnt, g0 + lane, p.E_l, rows, src_rows);
            mt = DW ? (gr.n > 0 ? dmt : 0) : (gr.n + GD_BM - 1) / GD_BM;
            ti = wave_incl_scan(mt);
            mt_all += wave_lane(ti, WAVE - 1);
            rows = gr.end;
            if constexpr (DW) {
                // the gradient of a group without rows is zero (it has no tile), by all workgroups
                unsigned long long none = __ballot(g0 + lane < p.E_l && gr.n == 0);
                while (none) {
                    const int e = g0 + __builtin_ctzll(none);
                    none &= none - 1;
                    const int nv = (p.dw_split ? p.dw_split : p.N) / 8;
                    bf16_t* c = (bf16_t*)p.C + (size_t)e * p.c_group_stride;
                    for (int i = blockIdx.x * GD_THREADS + tid; i < p.dw_rows * nv; i += gridDim.x * GD_THREADS) {
                        bf16_t* o = c + (size_t)(i / nv) * p.ldc + (i % nv) * 8;
                        *(uint4*)o = make_uint4(0, 0, 0, 0);
                        if (p.dw_split) *(uint4*)(o + p.dw_delta) = make_uint4(0, 0, 0, 0);
                    }
                }
            }
        }
        if constexpr (!DW && !FP8) gg_zero_tail(p, rows);
    }
    const int tiles = __builtin_amdgcn_readfirstlane(gg_whole_tiles(mt_all * Nt, 2 * cus, DW ? 0 : p.tail_max));
    // workgroups b, b + 8, ... share an XCD: of every GD_ROUND tiles in walking order it takes 64 in a row (those of the last, part-filled
    // round are dealt out evenly)
    int lin;
    {
        const int x = blockIdx.x & 7, i = blockIdx.x >> 3, r = i / (GD_ROUND / 8), j = i % (GD_ROUND / 8);
        const int left = tiles - r * GD_ROUND, per = left >= GD_ROUND ? GD_ROUND / 8 : (left + 7) / 8;
        lin = r * GD_ROUND + x * per + j;
        if (left <= 0 || j >= per || lin >= tiles) return;
    }
    int g = 0, row0 = 0, rv = 0, nt = 0, k0 = 0, nrows = 0;  // (DW) k0, nrows: the group's rows
    {
        int rows = 0, before = 0;
        for (int g0 = 0; g0 < p.E_l; g0 += WAVE) {
            if (p.E_l > WAVE) {
                gr = gg_rows<false>(p.cnt, g0 + lane, p.E_l, rows, src_rows);
                mt = DW ? (gr.n > 0 ? dmt : 0) : (gr.n + GD_BM - 1) / GD_BM;
                ti = wave_incl_scan(mt);
            }
            const int t0 = (before + ti - mt) * Nt;
            const unsigned long long hit = __ballot(mt > 0 && lin >= t0 && lin < t0 + mt * Nt);
            if (hit) {
                const int l = __builtin_ctzll(hit);
                int m;
                g = g0 + l;
                gg_patch(lin - wave_lane(t0, l), wave_lane(mt, l), Nt, SUP_DUO, m, nt);
                k0 = wave_lane(gr.start, l);
                nrows = wave_lane(gr.n, l);
                row0 = (DW ? 0 : k0) + m * GD_BM;
                rv = min(GD_BM, (DW ? p.dw_rows : nrows) - m * GD_BM);
                break;
            }
            rows = gr.end;
            before += wave_lane(ti, WAVE - 1);
        }
    }
    g = __builtin_amdgcn_readfirstlane(g); nt = __builtin_amdgcn_readfirstlane(nt);
    row0 = __builtin_amdgcn_readfirstlane(row0); rv = __builtin_amdgcn_readfirstlane(rv);
    k0 = __builtin_amdgcn_readfirstlane(k0); nrows = __builtin_amdgcn_readfirstlane(nrows);
    const int nks = DW ? (nrows + 63) / 64 * 2 : p.K * ES / ROWB;  // stages of K: even, two at least

    // ---- addresses: LDS tiles and fragments as in grouped_gemm.hip, but for the weight-gradient mode's A, whose rows are 256 bytes here
    const int lchunk = (lane & 3) ^ gg_swz(lane >> 4);
    const uint32_t ldk = DW ? (uint32_t)p.dw_rows * 2u : (uint32_t)(p.K * ES);
    [[maybe_unused]] const bool pair = p.B2 != nullptr;
    [[maybe_unused]] const uint32_t ldb = BT ? (uint32_t)(pair ? p.K / 2 : p.K) * 2u : (uint32_t)p.N * 2u;
    [[maybe_unused]] const size_t b_group = (size_t)p.K / (BT && pair ? 2 : 1) * p.N * 2;
    [[maybe_unused]] const ptrdiff_t b2_delta = p.B2 - p.B;
    const size_t b_slab = BT ? (size_t)ROWB : DW || BN_RAW ? (size_t)32 * ldb : (size_t)p.Npad * ROWB;
    const uint8_t* Ab = DW ? p.A + (size_t)k0 * ldk + (size_t)row0 * 2 : p.a_map ? p.A : p.A + (size_t)row0 * ldk;
    const size_t b_at = DW ? (size_t)k0 * ldb + (size_t)nt * GD_BN * 2
                      : BT ? (size_t)g * b_group + (size_t)nt * GD_BN * ldb
                      : BN_RAW ? (size_t)g * b_group + (size_t)nt * (BN_PAIR ? GD_BN : 2 * GD_BN)
                               : (size_t)g * p.Npad * ldk + (size_t)nt * GD_BN * ROWB;
    const uint8_t* Bb = p.B + b_at;
    [[maybe_unused]] const long long a_left = (long long)nrows * ldk - (long long)row0 * 2;
    [[maybe_unused]] const long long b_left = DW ? (long long)nrows * ldb - (long long)nt * GD_BN * 2 : (long long)p.E_l * b_group - (long long)b_at;
    uint32_t aoff[RA], boff[RB];
#pragma unroll
    for (int r = 0; r < RA; ++r) {
        if constexpr (DW)
            aoff[r] = (uint32_t)(4 * (r * 4 + wave) + (lane >> 4)) * ldk + (uint32_t)((lane & 15) ^ (2 * ((lane >> 4) + 4 * ((wave >> 1) & 1)))) * 16u;
        else if constexpr (WIDE) {
            const int ar = r * 32 + wave * 8 + (lane >> 3), lr = min(ar, rv - 1);
            aoff[r] = (uint32_t)(p.a_map ? max(p.a_map[row0 + lr], 0) : lr) * ldk + ((lane & 7) ^ gg_swz_wide(ar)) * 16;
        } else {
            const int lr = min(r * 64 + wave * WROWS + (lane >> 2), rv - 1);
            aoff[r] = (uint32_t)(p.a_map ? max(p.a_map[row0 + lr], 0) : lr) * ldk + lchunk * 16;
        }
    }
#pragma unroll
    for (int r = 0; r < RB; ++r) {
        if constexpr (DW) boff[r] = (uint32_t)(2 * (r * 4 + wave) + (lane >> 5)) * ldb + (uint32_t)((lane & 31) ^ (4 * ((2 * wave + (lane >> 5)) & 3))) * 16u;
        else if constexpr (BT) boff[r] = (uint32_t)gg_packed_col<false>(r * 64 + wave * WROWS + (lane >> 2)) * ldb + lchunk * 16;
        else if constexpr (BN_RAW) boff[r] = (uint32_t)(4 * (r % 2 * 4 + wave) + (lane >> 4)) * ldb + (uint32_t)((lane & 15) ^ (4 * (lane >> 4))) * 16u;
        else boff[r] = (uint32_t)(r * 64 + wave * WROWS + (lane >> 2)) * ROWB + lchunk * 16;
    }
    const uint32_t la0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)sA) + wave * WROWS * ROWB;
    const uint32_t lb0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)sB) + wave * WROWS * ROWB;
    [[maybe_unused]] const uint32_t ls0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)(s_hsc + wave * 128));
    [[maybe_unused]] const uint32_t soff = BSA ? (uint32_t)(row0 + min(wm * 64 + lane, rv - 1)) * (uint32_t)p.bs_pitch : 0u;
    typedef typename std::conditional<DW, gg_i32x4, const uint8_t*>::type asrc_t;
    typedef typename std::conditional<BMODE == GG_B_PACKED, const uint8_t*, gg_i32x4>::type bsrc_t;
    struct BSrc {
        bsrc_t b, b2;
    };
    auto asrc = [&](int st) -> asrc_t {
        if constexpr (DW) return gg_range(Ab + (size_t)st * 32 * ldk, a_left - (long long)st * 32 * ldk);
        else return gg_uniform(Ab + (size_t)st * ROWB);
    };
    auto bsrc = [&](int st) {
        BSrc s;
        const size_t so = BT && pair ? (size_t)(st >> 1) * ROWB : (size_t)st * b_slab;
        if constexpr (BMODE == GG_B_PACKED) s.b = gg_uniform(Bb + so);
        else {
            s.b = gg_range(BT && pair && (st & 1) ? Bb + b2_delta + so : Bb + so, b_left - (long long)so);
            if constexpr (BN_RAW) s.b2 = gg_range(Bb + (BN_PAIR ? b2_delta : 256) + so, b_left - (long long)so - (BN_PAIR ? 0 : 256));
        }
        return s;
    };
    auto load_a = [&](int d, const asrc_t& s, uint32_t la) { gg_dma16(s, aoff[d], la + d * 4096); };
    auto load_b = [&](int d, const BSrc& s, uint32_t lb) {
        if constexpr (BN_RAW) gg_dma16(d >= RB / 2 ? s.b2 : s.b, boff[d], lb + d * 4096);
        else gg_dma16(s.b, boff[d], lb + d * 4096);
    };
    auto load_scales = [&](int st) {
        if constexpr (BSA) gg_dma4(gg_uniform(p.a_bscale + ((st >> 1) << 2)), soff, ls0 + ((st >> 1) & 1) * 256);
    };

    // what the epilogue needs from memory per row and column: into a slot of B that is not needed any more
    auto load_tables = [&](uint8_t* to) {
        const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)to) + wave * 256;
        if (wave < 2) {
            const uint32_t t4 = (uint32_t)min(wave * WAVE + gg_lane_now(), rv - 1) * 4u;
            if ((FP8 || EPI == EPI_GATE) && (!BSA || p.row_scale)) gg_dma4(gg_uniform((const uint8_t*)(p.row_scale + row0)), t4, at);
            if (!DW && p.c_map) gg_dma4(gg_uniform((const uint8_t*)(p.c_map + row0)), t4, at + 512);
        }
        if constexpr (FP8) {
            const int ln = gg_lane_now(), pc = gg_packed_col<true>(nt * GD_BN + wave * WAVE + ln);
            int col = EPI == EPI_SWIGLU ? (pc / 64) * 32 + pc % 32 : pc;
            col = col < p.N ? col : 0;  // (columns past N are never stored: any valid scale will do)
            if (EPI == EPI_SWIGLU && ln >= 32) gg_dma4(gg_uniform((const uint8_t*)(p.col_scale2 + (size_t)g * p.ncs)), (uint32_t)col * 4u, at + 1024);
            else gg_dma4(gg_uniform((const uint8_t*)(p.col_scale + (size_t)g * p.ncs)), (uint32_t)col * 4u, at + 1024);
        }
    };

    typedef typename std::conditional<FP8, floatx16, floatx4>::type acc_t;
    acc_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < (FP8 ? 16 : 4); ++v) acc[i][j][v] = 0.f;

    // ---- fragments
    constexpr int FSTEP = FP8 ? 2 : 1;
    const int fpos = (FP8 ? (lane >> 5) : (lane >> 4)) ^ gg_swz(lane >> 2);
    const uint4* fa = (const uint4*)sA + (wm * 64 + (lane & (MT - 1))) * (WIDE ? 2 * CHUNKS : CHUNKS);
    [[maybe_unused]] const int fpos_a = (FP8 ? (lane >> 5) : (lane >> 4)) ^ gg_swz_wide(lane);
    const uint4* fb = (const uint4*)sB + (wn * 128 + (lane & (MT - 1))) * CHUNKS;
    [[maybe_unused]] uint32_t tr_a = 0, tr_b = 0;
    constexpr int BTR = DW ? 512 : 256;
    if constexpr (DW || BN_RAW) {
        const int kq = (lane >> 4) * 8 + ((lane & 15) >> 2), k4 = (lane & 15) >> 2, q4 = lane & 3;
        if constexpr (DW) {
            tr_a = (uint32_t)(uintptr_t)(lds_ptr_t)sA + kq * 256 + (((wm * 8 + (q4 >> 1)) ^ (2 * (k4 + 4 * ((lane >> 4) & 1)))) * 16) + (q4 & 1) * 8;
            tr_b = (uint32_t)(uintptr_t)(lds_ptr_t)sB + kq * 512 + (((wn * 16 + q4) ^ (4 * k4)) * 16);
        } else
            tr_b = (uint32_t)(uintptr_t)(lds_ptr_t)sB + (BN_PAIR ? 0 : wn * (BSZ / 2)) + kq * 256 + ((((BN_PAIR ? wn * 8 : 0) + q4) ^ (4 * k4)) * 16);
    }
    struct Frag {
        uint4 a[TM * CF], b[TN * CF];
    } f0, f1;
    [[maybe_unused]] int sc[TM];
    // fragment read R of a stage: of A in slot sa (a pair's and u, or a stage's), of B in slot sb
    auto read1 = [&](int R, Frag& f, int sa, int u, int sb) {
        if (R < TM * RPA) {
            const int i = R / RPA, h = R % RPA;
            if constexpr (DW) {
                const uint2 v = gg_read_tr<256>((tr_a ^ (i * 32)) + sa * ASZ, h);
                if (h == 0) { f.a[i].x = v.x; f.a[i].y = v.y; } else { f.a[i].z = v.x; f.a[i].w = v.y; }
            } else if constexpr (WIDE) f.a[i * CF + h] = fa[sa * (2 * ASZ / 16) + i * MT * 2 * CHUNKS + (fpos_a ^ (u * CHUNKS + h * FSTEP))];
            else f.a[i * CF + h] = fa[sa * (ASZ / 16) + i * MT * CHUNKS + (fpos ^ (h * FSTEP))];
        } else {
            const int j = (R - TM * RPA) / RPB, h = (R - TM * RPA) % RPB;
            if constexpr (DW || BN_RAW) {
                const uint32_t at = (tr_b ^ (BN_PAIR ? (j >> 2) * 64 : (j >> 1) * 64)) + (BN_PAIR ? ((j >> 1) & 1) * (BSZ / 2) : 0) + sb * BSZ + (j & 1) * 8;
                const uint2 v = gg_read_tr<BTR>(at, h);
                if (h == 0) { f.b[j].x = v.x; f.b[j].y = v.y; } else { f.b[j].z = v.x; f.b[j].w = v.y; }
            } else f.b[j * CF + h] = fb[sb * (BSZ / 16) + j * MT * CHUNKS + (fpos ^ (h * FSTEP))];
        }
    };
    auto read_scales = [&](int q) {  // those of pair q
        if constexpr (BSA) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
                sc[i] = (int)(((s_hsc[wave * 128 + (q & 1) * 64 + i * MT + (lane & 31)] >> ((lane >> 5) * 8)) & 0x00ff00ffu) + (uint32_t)(127 - GG_WSCALE) * 0x00010001u);
        }
    };
    // ---- prologue: the first three stages of B, the first three stages or two pairs of A (clamped: a tile has two stages at least)
#pragma unroll
    for (int d = 0; d < NST; ++d) {
        const int st = min(d, nks - 1);
        if (d != 1) load_scales(st);
        if (!WIDE || d != 1) {
            const asrc_t a = asrc(WIDE ? st & ~1 : st);
#pragma unroll
            for (int l = 0; l < RA; ++l) load_a(l, a, la0 + d * ASZ);
        }
        const BSrc b = bsrc(st);
#pragma unroll
        for (int l = 0; l < RB; ++l) load_b(l, b, lb0 + d * BSZ);
    }
    constexpr int BEHIND = RA + RB + (BSA ? 1 : 0);  // loads of the third
    gg_wait<(WIDE ? RB : RA + RB) + BEHIND, 0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int r = 0; r < NRD; ++r) read1(r, f0, 0, 0, 0);
    read_scales(0);
    gg_wait<BEHIND, 0>();
    __builtin_amdgcn_s_barrier();
    if constexpr (!FP8) __builtin_amdgcn_s_setprio(1);  // (a wave that multiplies goes before one that sets up or stores a tile)
    int slot = 0, pslot = 0;  // slots of stage s (B, and A where it comes by stages), of its pair (WIDE)
    // Block s multiplies stage s, reads the fragments of stage s + 1 and (LOAD) requests stage s + 3 into the slot of stage s; WIDE: A's pair s + 3, s + 4 in
    // odd blocks, into the slot of the pair that ends here.
    auto step = [&](auto load_c, auto odd_c, auto last_c, const Frag& f, Frag& nxt, int s) {
        constexpr bool LOAD = decltype(load_c)::value, ODD = decltype(odd_c)::value;
        constexpr int LEFT = decltype(last_c)::value;  // stages behind this one (3: three or more)
        constexpr int NLA = !LOAD || (WIDE && !ODD) ? 0 : RA, NL = LOAD ? NLA + RB : 0;  // loads of the block, A first
        const int nslot = slot == NST - 1 ? 0 : slot + 1, npslot = WIDE ? (ODD ? pslot ^ 1 : pslot) : nslot;
        asrc_t ap{};
        BSrc bp{};
        if constexpr (LOAD) {
            if constexpr (NLA > 0) ap = asrc(s + 3);
            bp = bsrc(s + 3);
            if constexpr (ODD) load_scales(s + 3);
        }
        if constexpr (LEFT == 1) load_tables(sB + slot * BSZ);
        const uint32_t la = la0 + (WIDE ? pslot * 2 : slot) * ASZ, lb = lb0 + slot * BSZ;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (BSA) asm volatile("s_nop 1");
        __builtin_amdgcn_sched_barrier(0);
        constexpr int RPM = FP8 || NRD > 24 ? 2 : 1;             // reads behind one MFMA
        constexpr int LSTEP = NT / (NL > 0 ? NL : 1) > 0 ? NT / (NL > 0 ? NL : 1) : 1;
        constexpr int LFIRST = NT > NL ? 1 : 0;
#pragma unroll
        for (int m = 0; m < NT; ++m) {
            const int i = m / TN, jj = m % TN, j = (i & 1) ? TN - 1 - jj : jj;
            if constexpr (BSA) {
                mma_fp8_k64_bs<false, ODD ? 2 : 0, true>(acc[i][j], f.b[2 * j], f.b[2 * j + 1], f.a[2 * i], f.a[2 * i + 1], sc[i]);
            } else if constexpr (FP8) mma_fp8_k64(acc[i][j], f.b[2 * j], f.b[2 * j + 1], f.a[2 * i], f.a[2 * i + 1]);
            else mma_bf16_k32(acc[i][j], f.b[j], f.a[i]);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (LOAD) {
                const int d = m >= LFIRST && (m - LFIRST) % LSTEP == 0 ? (m - LFIRST) / LSTEP : NL;
                if (d < NLA) load_a(d, ap, la);
                else if (d < NL) load_b(d - NLA, bp, lb);
            }
            if constexpr (LEFT > 0) {
#pragma unroll
                for (int e = 0; e < RPM; ++e)
                    if (m * RPM + e < NRD) read1(m * RPM + e, nxt, npslot, ODD ? 0 : 1, nslot);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (ODD && LEFT > 0) read_scales((s + 1) >> 1);
        slot = nslot;
        if constexpr (WIDE) pslot = npslot;
        asm volatile("" ::: "memory");
        // hand-over: stage s + 2 has landed, and nobody reads the slot of stage s + 1 any more
        if constexpr (LEFT > 1) {
            gg_wait<NL + (LOAD && BSA && ODD ? 1 : 0), 0>();
            __builtin_amdgcn_s_barrier();
        }
        asm volatile("" ::: "memory");
    };
    typedef std::integral_constant<bool, true> yes;
    typedef std::integral_constant<bool, false> no;
#define GD_LEFT(n) std::integral_constant<int, n>{}
    int s = 0;
    for (; s + 4 < nks; s += 2) {
        step(yes{}, no{}, GD_LEFT(3), f0, f1, s);
        step(yes{}, yes{}, GD_LEFT(3), f1, f0, s + 1);
    }
    if (nks > 2) {
        step(yes{}, no{}, GD_LEFT(3), f0, f1, s);
        step(no{}, yes{}, GD_LEFT(2), f1, f0, s + 1);
        s += 2;
    }
    step(no{}, no{}, GD_LEFT(1), f0, f1, s);
    step(no{}, yes{}, GD_LEFT(0), f1, f0, s + 1);
#undef GD_LEFT
    if constexpr (BSA) asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
    if constexpr (!FP8) __builtin_amdgcn_s_setprio(0);
    // (the tables went to the slot of the last stage but one)
    const uint8_t* const tab = sB + (slot == 0 ? 1 : slot == 1 ? 2 : 0) * BSZ;
    const float* const s_row_scale = (const float*)tab;
    const int* const s_crow = (const int*)(tab + 512);
    const float* const s_col_scale = (const float*)(tab + 1024);
    gg_wait<0, 0>();
    __syncthreads();

    // ---- epilogue: the lane's values, their places and their stores as in grouped_gemm_kernel
    bf16_t* C = (bf16_t*)p.C;
    constexpr int GT = 32 / MT, NG = TN / GT, NU = FP8 ? 2 : 1;
    const int lane_e = gg_lane_now(), rbase = wm * 64, cbase = wn * 128;
    const int lsub = FP8 ? (lane_e >> 5) : (lane_e >> 4);
    constexpr int NR = (FP8 && !QOUT) ? 2 : 1;
    bool ok[TM][NR];
    bf16_t* crow[TM][NR];
    float rs[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        rs[i] = 1.f;
        if constexpr (FP8 || EPI == EPI_GATE) {
            if (!BSA || p.row_scale) rs[i] = s_row_scale[rbase + i * MT + (lane_e & (MT - 1))];
        }
#pragma unroll
        for (int h = 0; h < NR; ++h) {
            const int r = rbase + i * MT + ((FP8 && !QOUT) ? (lane_e & 15) + 16 * h : (lane_e & (MT - 1)));
            ok[i][h] = r < rv;
            const size_t grow = (size_t)(row0 + (ok[i][h] ? r : 0));
            const int crow_i = !DW && p.c_map ? s_crow[r] : 0;
            ok[i][h] = ok[i][h] && crow_i >= 0;
            crow[i][h] = C + (!DW && p.c_map ? (size_t)max(crow_i, 0) : grow) * (QOUT ? (size_t)1 : (size_t)p.ldc) + (DW ? (size_t)g * p.c_group_stride : (size_t)0);
        }
    }
#pragma unroll
    for (int o = 0; o < TM * NG; ++o) {
        const int i = FP8 ? o % TM : o / NG, jg = FP8 ? o / TM : o % NG;
        if constexpr (EPI == EPI_SWIGLU) {
            if (jg % 2 == 1) continue;
        }
        const int pcol = nt * GD_BN + cbase + jg * 32;
        const bool two = EPI == EPI_SWIGLU || (DW && p.dw_split);
        const int colg = two ? (pcol / 64) * 32 : pcol;
        [[maybe_unused]] const long long cshift = DW && p.dw_split && (pcol & 32) ? p.dw_delta : 0;
        [[maybe_unused]] uint4 pk[2];
        [[maybe_unused]] float xq[2][8];
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int col = colg + (FP8 ? 16 * u : 0) + 8 * lsub;
            float x[8];
            [[maybe_unused]] float pre_g[8], pre_u[8];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int j = FP8 ? jg : jg * GT + t, qd = FP8 ? 2 * u + t : 0, ju = j + GT;
                float cg[4] = {1.f, 1.f, 1.f, 1.f}, cu[4] = {1.f, 1.f, 1.f, 1.f};
                if constexpr (FP8) {
                    const int tc = cbase + j * MT + 8 * qd + 4 * lsub;
                    const float4 s0 = *(const float4*)(s_col_scale + tc);
                    cg[0] = s0.x; cg[1] = s0.y; cg[2] = s0.z; cg[3] = s0.w;
                    if constexpr (EPI == EPI_SWIGLU) {
                        const float4 s1 = *(const float4*)(s_col_scale + tc + 32);
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
            } else if (ok[i][0] && col + (two && DW ? pcol - colg : 0) < p.N) {
                *(uint4*)(crow[i][0] + col + (DW ? cshift : 0)) = o4;
                if constexpr (EPI != EPI_NONE && EPI != EPI_GATE) {
                    if (p.C2) {
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
            float am = 0.f;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int e = 0; e < 8; ++e) am = fmaxf(am, fabsf(xq[u][e]));
            {
                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(am), __float_as_uint(am), false, false);
                am = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
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
            const auto s0 = __builtin_amdgcn_permlane32_swap(cd[0][0], cd[1][0], false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(cd[0][1], cd[1][1], false, false);
            const uint4 codes = make_uint4(s0[0], s1[0], s0[1], s1[1]);
            const int col = colg + 16 * lsub;
            if (ok[i][0] && col < p.N) {
                uint8_t* qrow = (uint8_t*)p.C + (size_t)(crow[i][0] - C) * p.ldc;
                *(uint4*)(qrow + col) = codes;
                if (lsub == 0) p.c_bscale[(size_t)(crow[i][0] - C) * p.bs_pitch + colg / 32] = (uint8_t)sbyte;
            }
        } else if constexpr (FP8) {
#define GD_SWAP16(a_, b_)                                                          \
    do {                                                                           \
        const auto sw_ = __builtin_amdgcn_permlane16_swap((a_), (b_), false, false); \
        (a_) = sw_[0];                                                             \
        (b_) = sw_[1];                                                             \
    } while (0)
            GD_SWAP16(pk[0].x, pk[1].x);
            GD_SWAP16(pk[0].y, pk[1].y);
            GD_SWAP16(pk[0].z, pk[1].z);
            GD_SWAP16(pk[0].w, pk[1].w);
#undef GD_SWAP16
            const int col = colg + 16 * ((lane_e >> 4) & 1) + 8 * lsub;
            if (col < p.N) {
                if (ok[i][0]) *(uint4*)(crow[i][0] + col) = pk[0];
                if (ok[i][NR - 1]) *(uint4*)(crow[i][NR - 1] + col) = pk[1];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

int launch_gemm_duo(const GemmParams& p, bool fp8, int epi, int cus, hipStream_t s) {
    const int nt = p.Npad / GD_BN;
    const bool dw = p.dw_rows > 0;
    const long long ub = dw ? (long long)p.E_l * ceil_div(p.dw_rows, GD_BM) * nt
                            : ((long long)p.S_rows + (long long)std::min(p.E_l, p.S_rows) * (GD_BM - 1)) / GD_BM * nt;
    const long long blocks = (ub + GD_ROUND - 1) / GD_ROUND * GD_ROUND;
#define GD_GO(EPIv, FP8v, MODEv) gemm_duo_kernel<EPIv, FP8v, MODEv><<<(unsigned)blocks, GD_THREADS, 0, s>>>(p, cus)
    if (dw) GD_GO(EPI_NONE, false, GG_B_DW);
    else if (fp8) {
        if (epi == EPI_NONE) GD_GO(EPI_NONE, true, GG_B_PACKED);
        else if (epi == EPI_SWIGLU) GD_GO(EPI_SWIGLU, true, GG_B_PACKED);
        else return moe_fail(MOE_ERR_UNSUPPORTED, "grouped_gemm: fp8 with activation %d", epi);
    } else if (p.b_mode == GG_B_PACKED) {
        switch (epi) {
            case EPI_NONE: GD_GO(EPI_NONE, false, GG_B_PACKED); break;
            case EPI_GELU: GD_GO(EPI_GELU, false, GG_B_PACKED); break;
            case EPI_SILU: GD_GO(EPI_SILU, false, GG_B_PACKED); break;
            case EPI_SWIGLU: GD_GO(EPI_SWIGLU, false, GG_B_PACKED); break;
            case EPI_GATE: GD_GO(EPI_GATE, false, GG_B_PACKED); break;
            default: return moe_fail(MOE_ERR_INVALID, "grouped_gemm: activation %d", epi);
        }
    } else if (p.b_mode == GG_B_T && epi == EPI_NONE) GD_GO(EPI_NONE, false, GG_B_T);
    else if (p.b_mode == GG_B_NP && epi == EPI_SWIGLU) GD_GO(EPI_SWIGLU, false, GG_B_NP);
    else if (p.b_mode == GG_B_N && epi == EPI_NONE) GD_GO(EPI_NONE, false, GG_B_N);
    else if (p.b_mode == GG_B_N && epi == EPI_GELU) GD_GO(EPI_GELU, false, GG_B_N);
    else if (p.b_mode == GG_B_N && epi == EPI_SILU) GD_GO(EPI_SILU, false, GG_B_N);
    else return moe_fail(MOE_ERR_INVALID, "grouped_gemm: weight mode %d with activation %d", p.b_mode, epi);
#undef GD_GO
    return moe_check_launch("grouped_gemm");
}
}  // namespace moe_gg
