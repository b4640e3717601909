// What the grouped GEMM kernels (grouped_gemm.hip: large tiles; gemm_small.hip: small ones) share: launch parameters, the packed
// weight layout, MFMA wrappers, activations, HBM -> LDS loads.
#pragma once
#include "common.h"

namespace moe_gg {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int ROWB = 64;   // bytes of K per tile row per LDS ring stage
constexpr int CHUNKS = ROWB / 16;
constexpr int NRING = 4;   // LDS ring stages
constexpr int WROWS = 64 / CHUNKS;  // tile rows moved by one wave-wide 16-byte-per-lane load
constexpr int GG_MAXG = MOE_MAX_EXPERTS;
constexpr int GG_BN = 256;

struct GemmParams {
    const uint8_t* A;         // [S_rows, K] activations (bf16 or fp8)
    const uint8_t* B;         // packed weights [E_l, Npad, K]; or (b_mode) weights in the reference layout, see GgB
    const uint8_t* B2;        // the second matrix of a gate / up pair (GG_B_NP; GG_B_T with a pair, else NULL)
    int b_mode;
    void* C;                  // [S_rows, ldc] bf16
    void* C2;                 // optional (bf16 kernels with an activation): the values BEFORE the activation, bf16, row pitch ldc
                              // (SwiGLU: 2 ldc, in the packed gate / up column order), kept for the backward pass
    const int32_t* cnt;       // [E_l] rows per group
    const float* row_scale;   // fp8: [S_rows] per-row activation scale; bf16 with EPI_GATE: [S_rows] per-row gate
    const float* col_scale;   // fp8: [E_l, ncs] per-output-channel scale (gate for SwiGLU)
    const float* col_scale2;  // fp8 SwiGLU: [E_l, ncs] up scales
    // fp8, block-scaled hidden activation (one power-of-two scale, an E8M0 exponent byte, per row and 32 columns; bs_pitch
    // bytes per row): written beside the codes by the gate/up kernel's epilogue (c_bscale, rows as C's), read by the down
    // kernel as the scale operand of its MFMAs (a_bscale, rows as A's).
    uint8_t* c_bscale;
    const uint8_t* a_bscale;
    int bs_pitch;
    const int32_t* a_map;     // optional: logical row -> row of A (gather while loading), else A is row r itself
    const int32_t* c_map;     // optional: logical row -> row of C (scatter while storing)
    int E_l, K, N, Npad, ldc, S_rows, ncs;
    int zero_tail;            // rows [counted total, S_rows) of C are zeroed (no c_map then)
    // Small tiles (gemm_small.hip): scratch for the fp32 partial sums of tiles whose K range is cut (max_units part tiles), or NULL.
    float* part_ws;
    int max_units;
    // Large tiles: a last round of the persistent grid with at most this many tiles is left to a launch of small ones.
    int tail_max;
    // Weight-gradient mode (template flag DW): C[g] (dw_rows x N, at C + g * c_group_stride elements) = x_g^T dy_g, the reduction
    // running over the rows of group g.  A is x [rows, dw_rows] and B is dy [rows, N], both as they are: the reduction index is
    // the slow one, a K stage is 32 rows of each, and the fragments are transposed on their way out of LDS.  With dw_split (F)
    // dy's columns are in the fused gate / up order (32 gate, 32 up, ...): gate column n of a row goes to column n, up column n
    // to the element dw_delta further.
    int dw_rows;
    int dw_src_rows;  // rows of the operands: the counts are clamped to it
    int dw_split;
    long long dw_delta;
    size_t c_group_stride;
    // Time stamps (the TRACE instantiation only; see moe_diag_gemm_trace): GG_TRACE_TILE_WORDS words per workgroup -- for
    // every tile the wall clock (100 MHz) at the start of its K loop, at the end of its K loop and at the end of its
    // epilogue -- then GG_TRACE_BLOCK_WORDS words of workgroup 0: the clock at the end of each of its MFMA blocks.
    // trace_flags & 1: the epilogue computes but stores nothing.
    unsigned long long* trace;
    int trace_flags;
};
// How a kernel takes its weight operand (template parameter; the rows below are those of [E_l, rows, columns] bf16 tensors in the
// reference layout, read as they are -- for weights that change from call to call, whose re-tiling would cost more than it saves):
//   GG_B_PACKED  re-tiled (moe_prepack_weights): a K stage of a tile is one contiguous piece
//   GG_B_DW      the weight-gradient mode (see dw_rows): columns are output columns, the rows of a group are the reduction
//   GG_B_T       out = a w^T: rows are output columns, columns the reduction, 64 bytes of 256 rows to a stage, like an activation
//                operand; with B2 the stages alternate between B and B2 (the fused gate / up order of a's columns)
//   GG_B_N       out = a w: columns are output columns, rows the reduction: 32 rows of 256 columns to a stage, transposed on the way
//                out of LDS like GG_B_DW's
//   GG_B_NP      the same for a gate / up pair in the fused column order: 128 columns of B and the same 128 of B2 to a stage
// What they cost against the re-tiled operand (33618 rows, 32 groups): a w 901 -> 942 us (K 2048, N 7168) and 872 -> 913 us (K 7168,
// N 2048), a w^T 901 -> 927 and 872 -> 946 us; one group of 32768 rows 5 to 12 %.  Pieces of 64 or 256 bytes of rows far apart
// instead of 16 contiguous KB load the L2 channels less evenly.  Re-tiling one such matrix set takes 0.8 ms per direction.
// Reads past the end of a tensor (its last tile's columns past N) arrive as zeros; elsewhere they are other rows' values, in
// columns that are not stored.
enum { GG_B_PACKED = 0, GG_B_DW = 1, GG_B_T = 2, GG_B_N = 3, GG_B_NP = 4 };

constexpr int GG_TRACE_TILE_WORDS = 256, GG_TRACE_BLOCK_WORDS = 4096;

// Where a packed weight column sits inside its aligned group of 32 rows of the packed matrix.  The MFMA leaves a lane
// with runs of FOUR consecutive rows of the weight operand (bf16 16x16: rows 4q .. 4q+3 of a tile for the lanes 16q ..
// 16q+15; fp8 32x32: rows 8Q + 4h .. + 3 for the register quad Q and the lanes 32h .. 32h+31).  The rows of a group are
// ordered so that two of a lane's runs are EIGHT consecutive output columns, which leave as one 16-byte store:
//   bf16: column 8q + 4t + v of the group (t = 0, 1: the group's two MFMA tiles) at row 16t + 4q + v;
//   fp8 : column 16P + 8h + 4t + v (P = 0, 1; quads 2P + t) at row 8 (2P + t) + 4h + v.
// Runs of four columns that start at a multiple of four stay runs of four rows.
template <bool FP8>
__host__ __device__ inline int gg_col_to_row32(int c) {  // c in [0, 32)
    if (FP8) return ((c >> 4) * 2 + ((c >> 2) & 1)) * 8 + ((c >> 3) & 1) * 4 + (c & 3);
    return ((c >> 2) & 1) * 16 + (c >> 3) * 4 + (c & 3);
}
template <bool FP8>
__host__ __device__ inline int gg_row_to_col32(int r) {  // the inverse
    if (FP8) return (r >> 4) * 16 + ((r >> 2) & 1) * 8 + ((r >> 3) & 1) * 4 + (r & 3);
    return ((r >> 2) & 3) * 8 + (r >> 4) * 4 + (r & 3);
}
template <bool FP8>
__host__ __device__ inline int gg_packed_row(int col) { return (col & ~31) | gg_col_to_row32<FP8>(col & 31); }
template <bool FP8>
__host__ __device__ inline int gg_packed_col(int row) { return (row & ~31) | gg_row_to_col32<FP8>(row & 31); }

// x * sigmoid(x) with the hardware reciprocal (1 ulp) instead of an IEEE division: the SwiGLU epilogue of a
// 128 x 128 wave tile evaluates this 8192 times per lane-row, and the division was most of its cost
// two fp32 -> packed bf16 (round to nearest even) in one hardware conversion
typedef __bf16 gg_bf16x2 __attribute__((ext_vector_type(2)));
typedef float gg_f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t gg_pack_bf16(float lo, float hi) {
    const gg_f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, gg_bf16x2));
}
__device__ __forceinline__ float act_silu_fast(float x) { return x * __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }
__device__ __forceinline__ float act_silu(float x) { return x / (1.0f + __expf(-x)); }
__device__ __forceinline__ float act_gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752440f)); }

typedef float floatx4 __attribute__((ext_vector_type(4)));
// bf16: one 16x16x32 MFMA; lanes 16q .. 16q+15 hold K elements 8q .. 8q+7 (16 bytes) of rows 0 .. 15 of both operands
// (Z: the sum starts here -- the MFMA takes a constant zero as its C operand, so no accumulator is cleared beforehand)
template <bool Z = false>
__device__ __forceinline__ void mma_bf16_k32(floatx4& acc, const uint4& a, const uint4& b) {
    if constexpr (Z) {
        const floatx4 z = {0.f, 0.f, 0.f, 0.f};
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), z, 0, 0, 0);
    } else {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), acc, 0, 0, 0);
    }
}

// fp8: one 32x32x64 MFMA on 32 bytes of K per lane and operand (two 16-byte LDS chunks); both operands
// are split over the lanes and registers in the same way, so every k is multiplied exactly once
typedef int gg_i32x8 __attribute__((ext_vector_type(8)));
template <bool Z = false>
__device__ __forceinline__ void mma_fp8_k64(floatx16& acc, const uint4& a_lo, const uint4& a_hi, const uint4& b_lo, const uint4& b_hi) {
    const gg_i32x8 a = {(int)a_lo.x, (int)a_lo.y, (int)a_lo.z, (int)a_lo.w, (int)a_hi.x, (int)a_hi.y, (int)a_hi.z, (int)a_hi.w};
    const gg_i32x8 b = {(int)b_lo.x, (int)b_lo.y, (int)b_lo.z, (int)b_lo.w, (int)b_hi.x, (int)b_hi.y, (int)b_hi.z, (int)b_hi.w};
    // format selectors 0/0 = fp8 (e4m3) for both operands, no block scales
    if constexpr (Z) {
        const floatx16 z = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, z, 0, 0, 0, 0, 0, 0);
    } else {
        acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, acc, 0, 0, 0, 0, 0, 0);
    }
}

// The same MFMA with block scales on the activation operand (the instruction's B: the kernels multiply transposed, weights
// as A).  For row r of the operand and block b of 32 k (b = 0: the first four registers of the lanes 0-31 and 32-63, i.e. k
// 0-15 and 16-31 of the step; b = 1: the other four registers), the scale is the E8M0 byte OPSEL of the scale register of
// lane 32 b + r (established with a one-wave probe on the chip); the weight operand takes 2^0 everywhere.
constexpr int GG_WSCALE = 64;
// ASMV: the instruction written out, accumulator in ordinary vector registers (the layout of eight waves per workgroup,
// where a wave's 256 registers hold accumulators and fragments alike).  Through the builtin, the compiler moves the scaled
// MFMAs of that layout across the scheduling fences that pin the K loop, bunches them, and spills accumulators and
// fragments inside the loop; a volatile asm statement stays where it is written.  The compiler does not know that the
// statement is an MFMA: what it would insert between such an instruction and a dependent one is added by hand where the
// accumulators are next read (GG_MFMA_SETTLE).
template <bool Z, int OPSEL, bool ASMV = false>
__device__ __forceinline__ void mma_fp8_k64_bs(floatx16& acc, const uint4& a_lo, const uint4& a_hi, const uint4& b_lo, const uint4& b_hi,
                                               int scale_b) {
    const gg_i32x8 a = {(int)a_lo.x, (int)a_lo.y, (int)a_lo.z, (int)a_lo.w, (int)a_hi.x, (int)a_hi.y, (int)a_hi.z, (int)a_hi.w};
    const gg_i32x8 b = {(int)b_lo.x, (int)b_lo.y, (int)b_lo.z, (int)b_lo.w, (int)b_hi.x, (int)b_hi.y, (int)b_hi.z, (int)b_hi.w};
    if constexpr (ASMV) {
        static_assert(!Z, "the written-out form accumulates");
        const int wsc = GG_WSCALE;
        if constexpr (OPSEL == 0)
            asm volatile("v_mfma_scale_f32_32x32x64_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,0,0]" : "+v"(acc) : "v"(a), "v"(b), "v"(wsc), "v"(scale_b));
        else
            asm volatile("v_mfma_scale_f32_32x32x64_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,1,0]" : "+v"(acc) : "v"(a), "v"(b), "v"(wsc), "v"(scale_b));
        return;
    }
    // (the weight operand's scale byte is GG_WSCALE = 64, a constant the instruction can take without a register; the
    // activation side adds the 63 that are missing to 2^0 to its own bytes: the product of the two scales is what counts)
    if constexpr (Z) {
        const floatx16 z = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, z, 0, 0, 0, GG_WSCALE, OPSEL, scale_b);
    } else {
        acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, acc, 0, 0, 0, GG_WSCALE, OPSEL, scale_b);
    }
}

// Block scale of the fp8 hidden activation: the smallest power of two X = 2^(byte - 127) with amax / X <= 448 (the largest
// e4m3 value), from the bits of amax >= 0: amax = m 2^p, 1 <= m < 2, fits when p - e < 8, or p - e = 8 and m <= 1.75 -- so
// byte = p + 127 - 8, one more when the mantissa exceeds that of 1.75; never below 0 (amax = 0, or tiny).  Integer work:
// the CPU checker computes the same byte from the same bits.
__host__ __device__ inline int gg_block_scale_byte(uint32_t amax_bits) {
    const int b = (int)((amax_bits + 0x1fffffu) >> 23) - 8;
    return b < 0 ? 0 : b;
}
// 1 / X as a float: 2^(127 - byte), exact (byte <= 247 for finite amax)
__host__ __device__ inline uint32_t gg_block_inv_bits(int byte) { return (uint32_t)(254 - byte) << 23; }

// EPI_GATE: no activation, and every result row is multiplied by its row's gate (GemmParams::row_scale, one fp32
// multiplication before the rounding to bf16): the down projection of an expert whose rows return already weighted.
// (The fp8 kernels have a row scale as it is: a gate is folded into it by the caller.)
enum { EPI_NONE = 0, EPI_GELU = 1, EPI_SILU = 2, EPI_SWIGLU = 3, EPI_GATE = 4 };

// ---- pieces of the main loop ---------------------------------------------------------------------
// HBM -> LDS, 16 bytes per lane, no register staging.  One instruction moves 16 tile rows of one ring
// stage (64 lanes x 16 B = 16 rows x 64 B); wave w of a round moves rows [w*16, w*16+16) of that round.
// Written as inline assembly to get the scalar-base + 32-bit-lane-offset form (the builtin expands to a
// 64-bit per-lane address); M0 holds the LDS byte address of the wave's 1 KB destination.
// A scalar register that a vector instruction wrote (v_readlane, where the compiler brings a spilled base back) may be a load's base
// only five wait states later, and the compiler does not count them across the start of such a statement.  csrc/build.py goes over the machine
// code and refuses a library with a load that is too early (there is none within eight).  Moving the base to a scalar register of the statement's
// own would make that needless, but the loads wait for the move: mixtral's step 8062 -> 8126 us, its training pass 26111 -> 26437.
// The LDS address is added up in the statement, a constant offset as a literal: with the sums in front of it the compiler keeps one base
// for every load of a stage and reloads most of them from spills (265 instead of 239 instructions around the 128 MFMAs of two stages).  The small-tile
// kernel, which spills nothing, sums in front (198 tokens x 1152, 8 experts of 3392: 52.3 us with literals, 51.7).
__device__ __forceinline__ void gg_dma16(const uint8_t* sbase, uint32_t voff, uint32_t lds_base, uint32_t lds_off = 0) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %0"
                 : : "s"(sbase), "v"(voff), "s"(lds_base), "is"(lds_off) : "memory", "scc");
}

// The same through a buffer descriptor: bytes at or past its range arrive as zeros.
typedef int gg_i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void gg_dma16(const gg_i32x4& srd, uint32_t voff, uint32_t lds_base, uint32_t lds_off = 0) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %0, 0 offen lds"
                 : : "s"(srd), "v"(voff), "s"(lds_base), "is"(lds_off) : "memory", "scc");
}
// Descriptor of `left` bytes at p (none when left <= 0), in scalar registers.
__device__ __forceinline__ gg_i32x4 gg_range(const uint8_t* p, long long left) {
    const uint64_t v = (uint64_t)p;
    const long long n = left < 0 ? 0 : left > 0xfffffff0ll ? 0xfffffff0ll : left;
    const gg_i32x4 d = {__builtin_amdgcn_readfirstlane((int)(uint32_t)v), __builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32)) & 0xffff,
                        __builtin_amdgcn_readfirstlane((int)(uint32_t)n), 0x00020000};
    return d;
}

// LDS tiles of 64-byte rows: 16-byte chunk c of row r lies at position c ^ gg_swz(r / 4).  A 128-bit read by all lanes takes 16 of them
// at a time -- 0-3, 12-15, 20-27 (then the others of the first 32; the upper 32 likewise) -- so the fragment reads (lanes 16 q .. 16 q + 15: chunk q of rows 0 .. 15, or fp8 lanes
// 32 h .. 32 h + 31: chunk h of rows 0 .. 31) meet 64 different banks each time when the swizzle maps 0, 1, 2, 3 to 0, 3, 2, 1.  With
// 0, 1, 2, 3 itself lanes 0-3 and 20-23 share their banks: 303 bytes a ns and compute unit instead of 530 (reads alone).
__device__ __forceinline__ int gg_swz(int r4) { return -r4 & 3; }
// Tiles of 128-byte rows (a pair of stages, 64 bytes of K each).  A compute unit loads pieces of 64 bytes of rows from its L2 at 66 bytes a ns,
// pieces of 128 and more at 127 to 135 (loads alone, 256 workgroups of four waves): an activation operand in whole lines costs the load path half.  Chunk c of row r at position c ^ gg_swz_wide(r), c in 0 .. 7.  Two rows span
// the banks, and the eight even (odd) rows of each such 16 lanes meet eight different positions: rows 0-3 and 12-15 of one chunk have r / 2 % 8 = 0, 1, 6, 7, rows
// 4-11 of the next chunk 2, 3, 4, 5 with the lowest bit flipped; rows 0-3, 12-15, 20-27 of one chunk (fp8) all eight.
__device__ __forceinline__ int gg_swz_wide(int r) { return (r >> 1) & 7; }

// Half h of a fragment of a 16 x 16 x 32 MFMA out of an LDS tile whose rows run along k (row pitch PITCH bytes): lanes 16 q ..
// 16 q + 15 end with k 8 q + 4 h .. + 3 of columns 0 .. 15.  `addr`: the lane's LDS byte address of k = 8 q + (lane % 16) / 4, four
// columns from column 4 (lane % 4) on; the instruction transposes within the 16 lanes.
typedef short gg_i16x4 __attribute__((ext_vector_type(4)));
template <int PITCH>
__device__ __forceinline__ uint2 gg_read_tr(uint32_t addr, int h) {
    typedef __attribute__((address_space(3))) char* lds_char;
    typedef __attribute__((address_space(3))) gg_i16x4* lds_v4;
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4)((lds_char)(uintptr_t)addr + h * 4 * PITCH)));
}

// The lane id read afresh (two instructions) where it is needed.  What the epilogue and the tile set-up derive from it
// is then computed there, once per tile, instead of being hoisted out of the tile loop as a dozen lane-constant
// invariants that occupy -- or spill -- registers across the whole K loop.
__device__ __forceinline__ int gg_lane_now() {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}

// One dword per lane, HBM -> LDS: lane l's value lands at lds_addr + 4 l.
__device__ __forceinline__ void gg_dma4(const uint8_t* sbase, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %1, %0" : : "s"(sbase), "v"(voff), "s"(lds_addr) : "memory");
}

// a wave-uniform value forced into scalar registers
__device__ __forceinline__ const uint8_t* gg_uniform(const uint8_t* p) {
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const uint8_t*)(((uint64_t)hi << 32) | lo);
}

// s_waitcnt through the builtin (not inline asm) so that the compiler's own wait-count bookkeeping
// sees it.  gfx9 encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] << 14.
template <int VM, int LGKM>
__device__ __forceinline__ void gg_wait() {
    static_assert(VM >= 0 && VM <= 63 && LGKM >= 0 && LGKM <= 15, "wait counts");
    __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | (LGKM << 8) | ((VM >> 4) << 14));
}

// Where the rows of group g (one per lane, 64 in a row) lie: its first row, how many it has, and (the same in every lane) the end of the last of the
// 64; `before`: rows of the groups before them.  Counts that claim more rows than the buffers hold are cut at S_rows -- each before they
// are added up, so that no 64 of them wrap up to GG_SCAN_ROWS rows; beyond (ANY_ROWS), one by one.
constexpr int GG_SCAN_ROWS = (1 << 25) - 1;
struct GgRows {
    int start, n, end;
};
template <bool ANY_ROWS>
__device__ __forceinline__ GgRows gg_rows(const int32_t* cnt, int g, int E_l, int before, int S_rows) {
    const int left = S_rows - before, c = g < E_l ? min(max(cnt[g], 0), left) : 0;
    if (ANY_ROWS && S_rows > GG_SCAN_ROWS) {
        GgRows r = {0, 0, before};
#pragma unroll 1
        for (int l = 0; l < WAVE; ++l) {
            const int n = min(__shfl(c, l, WAVE), S_rows - r.end);
            if (lane_id() == l) { r.start = r.end; r.n = n; }
            r.end += n;
        }
        return r;
    }
    const int inc = wave_incl_scan(c);
    const int ex = min(inc - c, left);
    return {before + ex, min(c, left - ex), before + min(wave_lane(inc, WAVE - 1), left)};
}

constexpr int SUP = 16, SUP_DUO = 8;  // super-tile edge, in tiles: of 256 rows, of 128 (gemm_duo.hip)
// Tile idx of a group of Mt x Nt large tiles in the order they are walked: bands of `sup` rows, super-columns of `sup` within them.
__device__ __forceinline__ void gg_patch(int idx, int Mt, int Nt, int sup, int& mt, int& nt) {
    const int band = idx / (sup * Nt), rem = idx % (sup * Nt);
    const int hr = min(sup, Mt - band * sup);
    const int sc = rem / (hr * sup), rem2 = rem % (hr * sup);
    const int wc = min(sup, Nt - sc * sup);
    mt = band * sup + rem2 / wc;
    nt = sc * sup + rem2 % wc;
}

// Tiles of a launch that the large kernel takes: all of them, or whole rounds of the grid when the rest is left to small tiles.
__host__ __device__ inline int gg_whole_tiles(int total, int grid, int tail_max) {
    const int tail = total % grid;
    return tail <= tail_max ? total - tail : total;
}

// Tiles of a last round that fills less than a third of the grid or so: 64 x 128 tiles (gemm_small.hip) fill the chip with them sooner
// than large ones leave it.  Per 64-byte K stage a small tile takes 0.15 us of a compute unit (times 1.2, fp8 1.4, where units
// share the load path), a large one 0.47 us (128 rows: 0.30) while most of the chip idles beside it.  The launch costs 5 us when
// the counts leave it nothing to do, so several groups get it only where the round is long enough for the chance of some
// most / grid to be worth that.  (Before, such tiles were cut along K by a second launch and summed by a third, 9 us without a
// tail: 777 tokens x 2 of 60 fp8 experts 181 -> 153 us, half of it those launches.)
struct GgTail {
    int most;    // tiles left over at most for the small ones to be quicker
    bool worth;  // worth a launch that may find nothing
};
static inline GgTail gg_tail(int nk, int bm, bool fp8, int grid) {
    const double round_us = nk * (bm == 128 ? 0.30 : 0.47) + 4;
    const int most = (int)((round_us - 8) / (0.15 * nk * (fp8 ? 1.4 : 1.225)) * grid / (bm / 64 * 2));
    return {most < 0 ? 0 : most < grid ? most : grid - 1, round_us >= 45};
}

constexpr int GG_MAX_PARTS = 16;       // parts a tile's K range is cut into, at most
// stages per part when nk stages (even) are cut into P parts: even, and P of them cover nk
__host__ __device__ inline int gg_part_stages(int nk, int P) { return ((nk + P - 1) / P + 1) & ~1; }

// GemmParams::zero_tail, by all workgroups of a launch
__device__ __forceinline__ void gg_zero_tail(const GemmParams& p, int total) {
    if (__builtin_expect(!p.zero_tail || total >= p.S_rows, 1)) return;
    const int nv = p.N / 8;
    const size_t n = (size_t)(p.S_rows - total) * nv;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        *(uint4*)((bf16_t*)p.C + (size_t)(total + i / nv) * p.ldc + (i % nv) * 8) = make_uint4(0, 0, 0, 0);
}

// gemm_small.hip: the time of a launch of small tiles (32 or 64 rows) as the choice between the kernels sees it; and that launch.
double gs_estimate(int bm, double tiles, int nk, bool fp8, int cus, const void* part_ws, size_t part_ws_bytes);
int gs_plan_parts(long long tiles, int bm, int nk, int cus, const void* part_ws, size_t bytes);  // parts per tile, as its kernel finds them
size_t gs_workspace_bytes(int cus);  // (what its partial sums take at most)
int launch_gemm_small(const GemmParams& p, bool fp8, int bm, int epi, void* ws, size_t bytes, int cus, hipStream_t s);
// The tiles of a launch of large tiles (bm_big rows, grid workgroups) that GemmParams::tail_max left over.
int launch_gemm_tail(const GemmParams& p, bool fp8, int bm_big, int epi, void* ws, size_t bytes, int grid, hipStream_t s);

// gemm_duo.hip: tiles of 128 rows, two workgroups to a compute unit (GemmParams::tail_max as for 256-row tiles; weight gradients where dw_rows is set).
int launch_gemm_duo(const GemmParams& p, bool fp8, int epi, int cus, hipStream_t s);
}  // namespace moe_gg
