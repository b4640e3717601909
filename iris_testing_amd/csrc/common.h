// Shared device/host helpers for libmoe_gfx950.so (gfx950 only, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>
#include <type_traits>

#include "../../include/moe_gfx950.h"

#define WAVE 64

// ---- error text (per calling thread) ---------------------------------------------------------
char* moe_err_buf();
int moe_fail(int code, const char* fmt, ...);
int moe_check_launch(const char* what);

// dispatch.hip, for step.hip: moe_count_and_offsets and moe_recv_prepare with one launch less
int moe_count_and_prepare(const moe_step_args* a, hipStream_t s);
// ... and where moe_count_with_pack says so, the count (with prepare: both) and the pack in one
bool moe_count_with_pack(int T, int k);
int moe_count_and_pack(const moe_step_args* a, bool prepare, hipStream_t s);
// grouped_gemm.hip, for step.hip: moe_unpack_expert_major of fp32 rows, moe_grouped_mlp and moe_return_pack, in two launches where tiles are small (S_rows > 0)
int moe_mlp_f32_slots(const float* recv, const int32_t* recv_counts, int W, int M, int S_rows, int H, int F, int E_l, int act, const float* w1,
                      const float* w_up, const float* w2, float* rows, int32_t* expert_cnt, float* hidden_ws, float* y, float* ret,
                      hipStream_t s);

#define MOE_REQUIRE(cond, code, ...)                 \
    do {                                             \
        if (!(cond)) return moe_fail(code, __VA_ARGS__); \
    } while (0)

// ---- bf16 as raw bits ------------------------------------------------------------------------
typedef uint16_t bf16_t;

__device__ __forceinline__ float bf16_to_f32(bf16_t v) { return __uint_as_float(((uint32_t)v) << 16); }

// round to nearest even; NaN stays a (quiet) NaN
__device__ __forceinline__ bf16_t f32_to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)((u >> 16) | 0x0040u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
}

template <typename T>
__device__ __forceinline__ float load_f32(const T* p);
template <>
__device__ __forceinline__ float load_f32<float>(const float* p) { return *p; }
template <>
__device__ __forceinline__ float load_f32<bf16_t>(const bf16_t* p) { return bf16_to_f32(*p); }

__device__ __forceinline__ int lane_id() { return threadIdx.x & (WAVE - 1); }

// Inclusive scan over the 64 lanes of a wave, all of them active: OP over the lanes up to the own one, from 0 (its neutral element: sums, maxima
// of values >= 0).  Six DPP moves; a cross-lane read through LDS (__shfl) is a round trip of some 35 ns instead, and the scans
// stand at the start of kernels that have little else to do.
template <typename OP>
__device__ __forceinline__ int wave_scan(int v, OP op) {
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));  // row_shr 1, 2, 4, 8: within 16 lanes
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));  // row_bcast 15: the 16 lanes before, to rows 1 and 3
    return op(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));  // row_bcast 31: the first half, to the second
}
__device__ __forceinline__ int wave_incl_scan(int v) {
    return wave_scan(v, [](int a, int b) { return a + b; });
}
// lane ^ OFF's value, without LDS either (OFF a power of two; all lanes active)
template <int OFF>
__device__ __forceinline__ int wave_xor(int x) {
    static_assert(OFF == 1 || OFF == 2 || OFF == 4 || OFF == 8 || OFF == 16 || OFF == 32, "");
    if constexpr (OFF == 1) return __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xf, 0xf, false);  // quad_perm [1,0,3,2]
    else if constexpr (OFF == 2) return __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xf, 0xf, false);  // quad_perm [2,3,0,1]
    else if constexpr (OFF == 4) {  // row_shl 4 into lanes 0-3 and 8-11 of a row, row_shr 4 into the others
        return __builtin_amdgcn_update_dpp(__builtin_amdgcn_update_dpp(0, x, 0x104, 0xf, 0x5, false), x, 0x114, 0xf, 0xa, false);
    } else if constexpr (OFF == 8) return __builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, false);  // row_ror 8
    else {
        // the swaps leave the pairs' lower (r[0]) and upper (r[1]) rows or halves in both
        if constexpr (OFF == 16) {
            const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
            return (int)((lane_id() & 16) ? r[0] : r[1]);
        } else {
            const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
            return (int)((lane_id() & 32) ? r[0] : r[1]);
        }
    }
}
// f(integral constants 32, 16, 8, 4, 2, 1)
template <typename F>
__device__ __forceinline__ void wave_butterfly(F&& f) {
    f(std::integral_constant<int, 32>{}); f(std::integral_constant<int, 16>{}); f(std::integral_constant<int, 8>{});
    f(std::integral_constant<int, 4>{}); f(std::integral_constant<int, 2>{}); f(std::integral_constant<int, 1>{});
}
// the same value in every lane: lane l's (l the same in all), the sum of all, the largest (of values >= 0)
__device__ __forceinline__ int wave_lane(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ int wave_sum(int v) { return wave_lane(wave_incl_scan(v), WAVE - 1); }
__device__ __forceinline__ int wave_max0(int v) {
    return wave_lane(wave_scan(v, [](int a, int b) { return max(a, b); }), WAVE - 1);
}

static inline int dtype_size(int dtype) { return dtype == MOE_F32 ? 4 : (dtype == MOE_BF16 ? 2 : 0); }
static inline int ceil_div(int a, int b) { return (a + b - 1) / b; }
// whether 16-byte loads and stores may start at p (NULL: there is nothing to load)
static inline bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }
// f(k as a constant where kernels have a form for it, else 0)
template <typename F>
static inline void with_topk(int k, F&& f) {
    switch (k) {
        case 1: return f(std::integral_constant<int, 1>{});
        case 2: return f(std::integral_constant<int, 2>{});
        case 4: return f(std::integral_constant<int, 4>{});
        case 8: return f(std::integral_constant<int, 8>{});
        case 16: return f(std::integral_constant<int, 16>{});
        default: return f(std::integral_constant<int, 0>{});
    }
}
template <int KT>
constexpr int topk_slots() { return KT ? KT : MOE_MAX_TOPK; }

// ---- bf16 rows as e4m3 codes and a scale per row: largest magnitude, codes of eight values -----
__device__ __forceinline__ float fp8_row_amax(const uint4& v, float amax) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        amax = fmaxf(amax, fabsf(__uint_as_float(w[i] << 16)));
        amax = fmaxf(amax, fabsf(__uint_as_float(w[i] & 0xffff0000u)));
    }
    return amax;
}
__device__ __forceinline__ uint2 fp8_row_convert(const uint4& v, float inv) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    float f[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[2 * i] = __fmul_rn(__uint_as_float(w[i] << 16), inv);
        f[2 * i + 1] = __fmul_rn(__uint_as_float(w[i] & 0xffff0000u), inv);
    }
    int lo = 0, hi = 0;
    lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], lo, false);
    lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], lo, true);
    hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], hi, false);
    hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], hi, true);
    return make_uint2((uint32_t)lo, (uint32_t)hi);
}
