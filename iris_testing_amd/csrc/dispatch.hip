// Per-destination counting, offsets, deterministic payload order, and the row-movement kernels
// (pack into [W,M,H], unpack to [E_l,W,CAP,H] / expert-major [S,H], return pack, combine).
//
// Replaces the Python bucket loop of route_and_pack_padding_free (reference utils.py:204-246),
// build_expert_offsets (utils.py:20-31), _build_dst_offsets (benchmark.py:44-49),
// reorder_flat_to_token_buf (baseline.py:178-222) and the intended token_shuffle kernel
// (layers/token_shuffle.py:31-56; kernels.py:179-205).
//
// Order of rows inside a (dst, el) bucket is ascending token index (utils.py:210-219).  An
// atomic-counter scatter would not reproduce that, so the position of every routed slot is
// computed as   expert_start[ex] + (rows of ex in earlier 64-token blocks) + (rows of ex in
// earlier lanes of this block),  with LDS histograms and per-expert lane masks.
// All integer work: results are bit-exact by construction.
#include "common.h"
#include <atomic>
#include <type_traits>

namespace {

constexpr int CB = MOE_COUNT_BLOCK;  // 64 tokens = one wave per counting block

// ---- 1. per-block histogram: hist[b][e] = #slots of block b routed to expert e --------------------
__global__ __launch_bounds__(256) void block_hist_kernel(const int32_t* __restrict__ idx, int32_t* __restrict__ hist,
                                                          int T, int k, int E, int NB) {
    extern __shared__ int32_t lds_hist[];  // [4][E]
    const int wave = threadIdx.x / WAVE;
    int32_t* my = lds_hist + wave * E;
    for (int i = threadIdx.x; i < 4 * E; i += blockDim.x) lds_hist[i] = 0;
    __syncthreads();
    const int b = blockIdx.x * 4 + wave;
    const int t = b * CB + lane_id();
    if (b < NB && t < T) {
        for (int j = 0; j < k; ++j) {
            const int e = idx[(size_t)t * k + j];
            if ((unsigned)e < (unsigned)E) atomicAdd(&my[e], 1);
        }
    }
    __syncthreads();
    if (b < NB)
        for (int e = lane_id(); e < E; e += WAVE) hist[(size_t)b * E + e] = my[e];
}

// ---- 2. expert prefix -> all count/offset outputs (one wave) ---------------------------------------
// A single wave runs it, whatever else its block holds; the lanes hand over through es in LDS.  es[e] = rows of the experts
// before e; with `write` the results also go to memory.
__device__ __forceinline__ void offsets_body(const int32_t* counts /*LDS*/, int E, int W, int32_t* es /*[E+1], LDS*/, bool write,
                                             int32_t* __restrict__ send_counts, int32_t* __restrict__ expert_offs,
                                             int32_t* __restrict__ dst_sizes, int32_t* __restrict__ dst_offsets,
                                             int32_t* __restrict__ caps) {
    const int lane = lane_id();
    const int per = (E + WAVE - 1) / WAVE;
    const int lo = min(lane * per, E), hi = min(lo + per, E);
    int sum = 0, cmax = 0;
    for (int e = lo; e < hi; ++e) { const int c = counts[e]; sum += c; cmax = max(cmax, c); }
    const int incl = wave_incl_scan(sum);
    int run = incl - sum;
    for (int e = lo; e < hi; ++e) { es[e] = run; run += counts[e]; }
    if (lane == WAVE - 1) es[E] = incl;
    if (!write) return;
    cmax = wave_max0(cmax);
    // the lanes' LDS writes above are read by other lanes of the same wave below
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int E_l = E / W;
    for (int e = lane; e < E; e += WAVE) {
        send_counts[e] = counts[e];
        expert_offs[e] = es[e] - es[(e / E_l) * E_l];
    }
    int mmax = 0;
    for (int d = lane; d < W; d += WAVE) {
        const int sz = es[(d + 1) * E_l] - es[d * E_l];
        dst_sizes[d] = sz;
        dst_offsets[d] = es[d * E_l];
        mmax = max(mmax, sz);
    }
    mmax = wave_max0(mmax);
    if (lane == 0) { caps[0] = max(mmax, 1); caps[1] = max(cmax, 1); }
}

// ---- 2b. many tokens: what the blocks before a ranking workgroup hold, by a scan over the histogram.  A workgroup takes SCAN_E experts,
// thread (slice, expert) a run of ranking groups (rank_blocks<false>() rows each): sums per slice, a scan of them over the
// lanes, then base[group][e] = rows of e in the groups before it, and after the last group the totals.  Two reads and a quarter
// of a write per histogram cell, in rows of 64 bytes; bound by the latency of a slice's run (262144 tokens x 8 of 256: the count takes
// 43 us, with the sums below 181, with one wave per expert along all blocks 101).
constexpr int SCAN_E = 16, SCAN_SLICES = 64;
constexpr int RANK_WAVES = 16;
template <bool ONE>
constexpr int rank_blocks() { return ONE ? 16 : 4; }
__global__ __launch_bounds__(SCAN_E * SCAN_SLICES) void scan_hist_kernel(const int32_t* __restrict__ hist, int32_t* __restrict__ base, int NB,
                                                                         int NG, int E) {
    __shared__ int32_t sum[SCAN_E][SCAN_SLICES + 1];
    constexpr int ROWS = rank_blocks<false>();
    static_assert(SCAN_SLICES == WAVE, "a slice per lane, an expert per wave");
    const int c = threadIdx.x % SCAN_E, sl = threadIdx.x / SCAN_E, e = blockIdx.x * SCAN_E + c;
    const int per = (NG + SCAN_SLICES - 1) / SCAN_SLICES, g0 = min(sl * per, NG), g1 = min(g0 + per, NG);
    auto group = [&](int g) {
        int v = 0;
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const int b = g * ROWS + r;
            v += b < NB ? hist[(size_t)b * E + e] : 0;
        }
        return v;
    };
    int all = 0;
    if (e < E) {
#pragma unroll 4
        for (int g = g0; g < g1; ++g) all += group(g);
    }
    sum[c][sl] = all;
    __syncthreads();
    const int wave = threadIdx.x / WAVE;  // (one wave per expert)
    const int mine = sum[wave][lane_id()], incl = wave_incl_scan(mine);
    __syncthreads();
    sum[wave][lane_id()] = incl - mine;
    if (lane_id() == WAVE - 1) sum[wave][SCAN_SLICES] = incl;
    __syncthreads();
    if (e >= E) return;
    int run = sum[c][sl];
#pragma unroll 4
    for (int g = g0; g < g1; ++g) {
        base[(size_t)g * E + e] = run;
        run += group(g);
    }
    if (sl == 0) base[(size_t)NG * E + e] = sum[c][SCAN_SLICES];
}

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
constexpr int PACK_ZR = 8;  // consecutive slots of a [W,M,row] buffer that a wave looks through for padding (see pack_tokens_kernel)


// rows [size_s, M) of every slot s of a [W,M,row] buffer <- 0, size_s = sum over e of rc[s,e]; one wave per run of
// consecutive rows (the slot's size is summed once per run, or twice when the run crosses into the next slot)
__device__ __forceinline__ int slot_size(const int32_t* __restrict__ rc, int s, int E_l, int lane) {
    int size = 0;
    for (int e = lane; e < E_l; e += WAVE) size += rc[s * E_l + e];
    return wave_sum(size);
}
__device__ __forceinline__ void zero_padding_rows(u32x4* __restrict__ buf, const int32_t* __restrict__ rc, int W, int E_l, int M,
                                                  int row_vecs, int block, int run) {
    const int wave = threadIdx.x / WAVE, lane = lane_id();
    const int r0 = (block * (blockDim.x / WAVE) + wave) * run, r1 = min(r0 + run, W * M);
    if (r0 >= r1) return;
    int s = r0 / M, m = r0 % M;
    int size = slot_size(rc, s, E_l, lane);
    const u32x4 z = {0u, 0u, 0u, 0u};
    for (int r = r0; r < r1; ++r) {
        if (m >= size) {
            u32x4* row = buf + (size_t)r * row_vecs;
            for (int c = lane; c < row_vecs; c += WAVE) __builtin_nontemporal_store(z, row + c);
        }
        if (++m == M && r + 1 < r1) { m = 0; size = slot_size(rc, ++s, E_l, lane); }
    }
}

// Expert-major row r of the receive side -> row of the [W,M,H] buffer that holds it (one thread per row, binary search in
// the (expert, source)-major prefix).  The same index serves the way back: the result row of r returns to the slot its input
// came from.  Rows past the received total map to row 0; rows the pack dropped (position in the sender's slot at or past
// the pair capacity M) map to -1: the GEMMs read row 0 for them and store nothing.
// One launch: every block derives the two prefix tables it needs from recv_counts in LDS (at most
// MOE_MAX_EXPERTS entries: a wave's scan) instead of waiting for a table kernel; block 0 also leaves the per-expert totals.
// M = 0: the receive buffer is a padding-free flat payload instead (source-major, expert-minor blocks, the layout
// reorder_flat_to_token_buf of the reference reads, baseline.py:204-218): the row of (e, s, j) is the exclusive prefix of the
// counts over flattened (s, e) plus j, and no row can have been dropped.
// recv_gate / row_gate (both or neither): the gates that arrived with the rows, [rows of the receive buffer], gathered
// into expert-major order for the GEMM that applies them (0 for rows without a source).  recv_scale / row_scale likewise: the
// fp8 row scales (rows without a source take that of row 0, whose codes the GEMM reads for them).
// zbuf (or NULL): the blocks from map_blocks on zero the padding rows of that [W,M,row_vecs] buffer, which depend on the same counts.
// A launch of its own (256 threads to a block) or, in a step, blocks beside the ranking's (1024).
struct RecvPrepare {
    const int32_t* rc;
    int W, E_l, M, n_rows;
    int32_t *map, *expert_cnt;
    const float* recv_gate;
    float* row_gate;
    const float* recv_scale;
    float* row_scale;
    u32x4* zbuf;
    int row_vecs, map_blocks, run;
};
__device__ __forceinline__ void recv_prepare_block(const RecvPrepare& a, int block, int32_t* s_row_off /* [MOE_MAX_EXPERTS + 1] */, int32_t* s_src_off) {
    if (block >= a.map_blocks) {
        zero_padding_rows(a.zbuf, a.rc, a.W, a.E_l, a.M, a.row_vecs, block - a.map_blocks, a.run);
        return;
    }
    const int n = a.W * a.E_l;
    const bool flat = a.M == 0;
    if (threadIdx.x < WAVE) {
        const int lane = lane_id();
        const int per = (n + WAVE - 1) / WAVE;
        const int lo = min(lane * per, n), hi = min(lo + per, n);
        int sum = 0;
        for (int i = lo; i < hi; ++i) sum += a.rc[(i % a.W) * a.E_l + (i / a.W)];
        const int incl = wave_incl_scan(sum);
        int run = incl - sum;
        for (int i = lo; i < hi; ++i) { s_row_off[i] = run; run += a.rc[(i % a.W) * a.E_l + (i / a.W)]; }
        if (lane == WAVE - 1) s_row_off[n] = incl;
        if (flat) {  // exclusive prefix over flattened (s, e): where the block of (s, e) starts in the flat payload
            int fsum = 0;
            for (int i = lo; i < hi; ++i) fsum += a.rc[i];
            const int fincl = wave_incl_scan(fsum);
            int frun = fincl - fsum;
            for (int i = lo; i < hi; ++i) { s_src_off[i] = frun; frun += a.rc[i]; }
        } else {
            for (int sr = lane; sr < a.W; sr += WAVE) {
                int r = 0;
                for (int e = 0; e < a.E_l; ++e) { s_src_off[sr * a.E_l + e] = r; r += a.rc[sr * a.E_l + e]; }
            }
        }
        if (block == 0 && a.expert_cnt)
            for (int e = lane; e < a.E_l; e += WAVE) {
                int c = 0;
                for (int sr = 0; sr < a.W; ++sr) c += a.rc[sr * a.E_l + e];
                a.expert_cnt[e] = c;
            }
    }
    __syncthreads();
    const int r = block * blockDim.x + threadIdx.x;
    if (r >= a.n_rows) return;
    if (r >= s_row_off[n]) {
        a.map[r] = 0;
        if (a.row_gate) a.row_gate[r] = 0.f;
        if (a.row_scale) a.row_scale[r] = a.recv_scale[0];
        return;
    }
    int lo = 0, hi = n;  // s_row_off[0] = 0 <= r; the last of a run of equal offsets owns the row
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (s_row_off[mid] <= r) lo = mid; else hi = mid;
    }
    const int e = lo / a.W, sr = lo % a.W;
    const int m = s_src_off[sr * a.E_l + e] + (r - s_row_off[lo]);
    const int row = flat ? m : (m < a.M ? sr * a.M + m : -1);
    a.map[r] = row;
    if (a.row_gate) a.row_gate[r] = row >= 0 ? a.recv_gate[row] : 0.f;
    if (a.row_scale) a.row_scale[r] = a.recv_scale[max(row, 0)];
}

// ---- 3. stable positions.  A workgroup of 16 waves ranks RBLK consecutive blocks of 64 tokens, 16 / RBLK waves to a block, each with
// every (16 / RBLK)-th of a token's slots: the waves OR their lane bits into a 64-bit mask per block and expert in LDS (a token holds
// an expert at most once), and the rank of a slot inside its expert is the rows of the expert in earlier workgroups' blocks +
// the popcounts of the earlier blocks' masks + the popcount of its own mask below the lane.
// What the earlier blocks hold every workgroup sums up for itself from the histogram (NB x E words from L2: 8 KB for 16384 tokens
// and 8 experts, 256 KB for 16384 and 256, in 16-byte loads where E allows them), and the offsets with it: no scan launch between the
// two (it took 5 to 22 us on its own, one workgroup walking its experts' rows one after the other).  Four blocks to a workgroup:
// with 16 the popcounts of up to 15 masks per slot and four workgroups in all took 22 us for 4096 tokens x 8 of 256, so 9.
// (scan and rank took 22 us as launches of their own.)
// ONE = true (up to 1024 tokens): a single workgroup holds all 16 blocks, counts for itself and is the only launch.
// SIDE: the blocks from rank_blocks_n on prepare the receive side (in a step, where the received counts are there already: a launch less, 2 to 3 us
// beside a ranking that leaves the chip idle).
// base (or NULL): what scan_hist_kernel left, where the sums, which grow with the square of the tokens, are too many (RANK_SUM_CELLS).
// hist == NULL (few enough slots, RANK_SELF_SLOTS): the workgroup counts all slots, those before its blocks and the rest apart, in eight
// copies of the counters, so that lanes with the same expert seldom meet.
constexpr int RANK_COPIES = 8;
template <bool ONE, bool SIDE>
__global__ __launch_bounds__(RANK_WAVES * WAVE) void rank_kernel(const int32_t* __restrict__ idx, const int32_t* __restrict__ hist,
                                                                  const int32_t* __restrict__ base, int T,
                                                                  int k, int E, int W, int NB, int32_t* __restrict__ send_counts,
                                                                  int32_t* __restrict__ expert_offs, int32_t* __restrict__ dst_sizes,
                                                                  int32_t* __restrict__ dst_offsets, int32_t* __restrict__ caps,
                                                                  int32_t* __restrict__ pos, int32_t* __restrict__ row_token, int rank_blocks_n,
                                                                  const RecvPrepare side) {
    constexpr int RBLK = rank_blocks<ONE>(), PARTS = RANK_WAVES / RBLK, SLOTS = MOE_MAX_TOPK / PARTS;
    extern __shared__ unsigned long long masks[];  // [RBLK][E]
    __shared__ int32_t tot[MOE_MAX_EXPERTS], pre[MOE_MAX_EXPERTS], es[MOE_MAX_EXPERTS + 1];
    if (SIDE && (int)blockIdx.x >= rank_blocks_n) {
        recv_prepare_block(side, blockIdx.x - rank_blocks_n, es, pre);
        return;
    }
    const int tid = threadIdx.x, wave = tid / WAVE, lane = lane_id(), blk = wave / PARTS, part = wave % PARTS;
    const int b0 = blockIdx.x * RBLK, t = (b0 + blk) * CB + lane;
    const bool live = b0 + blk < NB && t < T;
    int mine[SLOTS];
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) mine[j] = (live && j * PARTS + part < k) ? idx[(size_t)t * k + j * PARTS + part] : -1;
    for (int e = tid; e < E; e += blockDim.x) {
        tot[e] = !ONE && base ? base[(size_t)rank_blocks_n * E + e] : 0;
        pre[e] = !ONE && base ? base[(size_t)blockIdx.x * E + e] : 0;
    }
    for (int i = tid; i < RBLK * E; i += blockDim.x) masks[i] = 0ull;
    const int stride = E | 1;  // (odd: the copies of a counter lie in different banks)
    int32_t* const tab = reinterpret_cast<int32_t*>(masks + RBLK * E);
    if (!ONE && !hist)
        for (int i = tid; i < 2 * RANK_COPIES * stride; i += blockDim.x) tab[i] = 0;
    __syncthreads();
    unsigned long long* my = masks + blk * E;
#pragma unroll
    for (int j = 0; j < SLOTS; ++j)
        if ((unsigned)mine[j] < (unsigned)E) {
            atomicOr(&my[mine[j]], 1ull << lane);
            if constexpr (ONE) atomicAdd(&tot[mine[j]], 1);
        }
    if constexpr (!ONE) {
        // column sums of the histogram: thread = (V experts, slice of the blocks)
        auto sums = [&](auto vec) {
            constexpr int V = decltype(vec)::value;
            const int cols = E / V, slices = blockDim.x / cols, c = tid % cols, sl = tid / cols;
            if (sl >= slices) return;
            int all[V] = {}, before[V] = {};
#pragma unroll 8
            for (int b = sl; b < NB; b += slices) {
                int v[V];
                if constexpr (V == 4) {
                    const int4 q = reinterpret_cast<const int4*>(hist + (size_t)b * E)[c];
                    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
                } else {
                    v[0] = hist[(size_t)b * E + c];
                }
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    all[i] += v[i];
                    before[i] += b < b0 ? v[i] : 0;
                }
            }
#pragma unroll
            for (int i = 0; i < V; ++i) {
                atomicAdd(&tot[c * V + i], all[i]);
                atomicAdd(&pre[c * V + i], before[i]);
            }
        };
        if (!hist) {
            const int n = T * k, limit = min(b0 * CB, T) * k, copy = lane % RANK_COPIES;
            auto add = [&](int i, int e) {
                if ((unsigned)e < (unsigned)E) atomicAdd(&tab[((i < limit ? 0 : RANK_COPIES) + copy) * stride + e], 1);
            };
            const int vecs = ((uintptr_t)idx & 15) == 0 ? n / 4 : 0;
#pragma unroll 4
            for (int i = tid; i < vecs; i += RANK_WAVES * WAVE) {
                const int4 q = reinterpret_cast<const int4*>(idx)[i];
                add(4 * i, q.x); add(4 * i + 1, q.y); add(4 * i + 2, q.z); add(4 * i + 3, q.w);
            }
            for (int i = 4 * vecs + tid; i < n; i += RANK_WAVES * WAVE) add(i, idx[i]);
            __syncthreads();
            for (int e = tid; e < E; e += RANK_WAVES * WAVE) {
                int before = 0, after = 0;
#pragma unroll
                for (int c = 0; c < RANK_COPIES; ++c) {
                    before += tab[c * stride + e];
                    after += tab[(RANK_COPIES + c) * stride + e];
                }
                pre[e] = before;
                tot[e] = before + after;
            }
        } else if (!base) {
            if (E % 4 == 0 && ((uintptr_t)hist & 15) == 0) sums(std::integral_constant<int, 4>{});
            else sums(std::integral_constant<int, 1>{});
        }
    }
    __syncthreads();
    if (wave == 0) offsets_body(tot, E, W, es, blockIdx.x == 0, send_counts, expert_offs, dst_sizes, dst_offsets, caps);
    __syncthreads();
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (WAVE - lane));
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) {
        const int e = mine[j];
        if ((unsigned)e < (unsigned)E) {
            int p = es[e] + pre[e] + __popcll(my[e] & below);
            for (int w = 0; w < blk; ++w) p += __popcll(masks[w * E + e]);
            pos[(size_t)t * k + j * PARTS + part] = p;
            row_token[p] = t;
        }
    }
}

// ---- small integer helpers --------------------------------------------------------------------------
__global__ void max_floor1_kernel(const int32_t* __restrict__ v, int n, int32_t* __restrict__ out) {
    __shared__ int32_t red[256];
    int m = 1;
    for (int i = threadIdx.x; i < n; i += blockDim.x) m = max(m, v[i]);
    red[threadIdx.x] = m;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] = max(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}



// expert_offs[d,e] = exclusive prefix over e of counts[d,:]; dst_sizes / dst_offsets over d (one wave)
__global__ __launch_bounds__(WAVE) void expert_offsets_kernel(const int32_t* __restrict__ counts, int W, int E_l,
                                                               int32_t* __restrict__ expert_offs, int32_t* __restrict__ dst_sizes,
                                                               int32_t* __restrict__ dst_offsets) {
    __shared__ int32_t sizes[MOE_MAX_EXPERTS];
    const int lane = lane_id();
    for (int d = lane; d < W; d += WAVE) {
        int r = 0;
        for (int e = 0; e < E_l; ++e) { expert_offs[d * E_l + e] = r; r += counts[d * E_l + e]; }
        sizes[d] = r;
        if (dst_sizes) dst_sizes[d] = r;
    }
    __syncthreads();
    if (dst_offsets && lane == 0) {
        int r = 0;
        for (int d = 0; d < W; ++d) { dst_offsets[d] = r; r += sizes[d]; }
    }
}

// ---- row movement: dst[r,:] = src[source_row(r),:], or zeros when the row has no source ---------------
// One wave per output row, 16 bytes per lane.  The source row is resolved inside the kernel (no map
// buffer, no extra launch); every quantity involved is wave-uniform.
enum {
    SRC_MAP = 0,      // map[r]                                  (padding-free payload)
    SRC_PACK = 1,     // send slot (d,m) -> token                (fixed [W,M,H] pack)
    SRC_UNPACK = 2,   // expert-major row r -> recv row          (recv [W,M,H] -> [S,H])
    SRC_TOKBUF = 3,   // token_buf row (e,s,j) -> recv row       (recv [W,M,H] -> [E_l,W,CAP,H])
    SRC_RETURN = 4,   // return slot (s,m) -> expert-major row   ([S,H] -> [W,M,H])
    SRC_REORDER = 5,  // token_buf row (e,s,j) -> flat row       (flat payload -> [E_l,W,CAP,H])
    SRC_SHUFFLE = 6,  // expert-major row r -> token_buf row     ([E_l,W,CAP,H] -> [S,H])
    SRC_UNSHUFFLE = 7 // token_buf row (e,s,j) -> expert-major row ([S,H] -> [E_l,W,CAP,H]; the shuffle's gradient)
};

struct RowSource {
    int mode;
    const int32_t* map;                                   // SRC_MAP / SRC_PACK: row_token
    const int32_t *dst_sizes, *dst_offsets;               // SRC_PACK
    const int32_t *rc, *src_off, *row_off, *flat_off;     // recv-driven modes: tables in LDS (recv_tables)
    int W, E_l, M, CAP;
    int32_t* status;
};

// What the recv-driven modes derive from recv_counts (W E_l <= MOE_MAX_EXPERTS entries; counts are read as
// counts[s * pitch_s + e * pitch_e], so a matrix or its transpose will do):
//   rc[s*E_l+e]      the counts themselves
//   src_off[s*E_l+e] exclusive prefix over e of rc[s,:]                  (row inside slot s)
//   row_off[e*W+s]   exclusive prefix over flattened (e,s)               (expert-major row; total at [E_l*W])
//   flat_off[s*E_l+e] exclusive prefix over flattened (s,e)              (row in a padding-free flat payload)
// Every workgroup of the copy makes its own set in LDS, one table to a wave (2 us with 256 counts, once per workgroup of a
// grid that stays on the chip), instead of a launch of one wave in front of the copy (4.8 us in a graph, 5 to 15 at 256 counts).
struct RecvCounts {
    const int32_t* counts;
    int pitch_s, pitch_e;
    int32_t *pca, *expert_cnt;  // or NULL: counts[e][s], rows per expert (left by the first workgroup)
};
struct RecvTables {
    int32_t rc[MOE_MAX_EXPERTS], src_off[MOE_MAX_EXPERTS], row_off[MOE_MAX_EXPERTS + 1], flat_off[MOE_MAX_EXPERTS];
};
__device__ __forceinline__ void recv_tables(RecvTables& t, const RecvCounts& q, int W, int E_l) {
    const int n = W * E_l, wave = threadIdx.x / WAVE, lane = lane_id();
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int s = i / E_l, e = i % E_l, c = q.counts[(size_t)s * q.pitch_s + (size_t)e * q.pitch_e];
        t.rc[i] = c;
        if (q.pca && blockIdx.x == 0) q.pca[e * W + s] = c;
    }
    __syncthreads();
    const int per = (n + WAVE - 1) / WAVE;
    const int lo = min(lane * per, n), hi = min(lo + per, n);
    if (wave == 0) {
        int sum = 0;
        for (int i = lo; i < hi; ++i) sum += t.rc[(i % W) * E_l + i / W];
        const int incl = wave_incl_scan(sum);
        int run = incl - sum;
        for (int i = lo; i < hi; ++i) { t.row_off[i] = run; run += t.rc[(i % W) * E_l + i / W]; }
        if (lane == WAVE - 1) t.row_off[n] = incl;
    } else if (wave == 1) {
        int sum = 0;
        for (int i = lo; i < hi; ++i) sum += t.rc[i];
        int run = wave_incl_scan(sum) - sum;
        for (int i = lo; i < hi; ++i) { t.flat_off[i] = run; run += t.rc[i]; }
    } else if (wave == 2) {
        for (int s = lane; s < W; s += WAVE) {
            int r = 0;
            for (int e = 0; e < E_l; ++e) { t.src_off[s * E_l + e] = r; r += t.rc[s * E_l + e]; }
        }
    } else if (wave == 3 && q.expert_cnt && blockIdx.x == 0) {
        for (int e = lane; e < E_l; e += WAVE) {
            int c = 0;
            for (int s = 0; s < W; ++s) c += t.rc[s * E_l + e];
            q.expert_cnt[e] = c;
        }
    }
    __syncthreads();
}

// largest i in [0,n) with off[i] <= r (off ascending, off[0] = 0): the whole wave looks at 64 entries
// at a time and counts them with a ballot.  Equal offsets mark empty segments; the last of a run of
// equal offsets is the segment that owns the row.
__device__ __forceinline__ int wave_seg(const int32_t* __restrict__ off, int n, int r) {
    int total = 0;
    for (int base = 0; base < n; base += WAVE) {
        const int i = base + lane_id();
        const bool le = i < n && off[i] <= r;
        total += __popcll(__ballot(le));
    }
    return total - 1;
}

__device__ __forceinline__ int source_row(const RowSource& a, int r) {
    const int n = a.W * a.E_l;
    switch (a.mode) {
        case SRC_MAP: return a.map[r];
        case SRC_PACK: {
            const int d = r / a.M, m = r % a.M;
            const int cnt = a.dst_sizes[d];
            if (m == 0 && cnt > a.M && a.status && lane_id() == 0) *a.status = 1;
            return m < cnt ? a.map[a.dst_offsets[d] + m] : -1;
        }
        case SRC_UNPACK:
        case SRC_SHUFFLE: {
            if (r >= a.row_off[n]) return -1;
            const int seg = wave_seg(a.row_off, n + 1, r);  // seg = e*W + s
            const int e = seg / a.W, s = seg % a.W, j = r - a.row_off[seg];
            if (a.mode == SRC_SHUFFLE) return (e * a.W + s) * a.CAP + j;
            // a row past the pair capacity never reached the slot (the pack dropped it): it reads as zeros
            const int m = a.src_off[s * a.E_l + e] + j;
            if (m >= a.M) {
                if (a.status && lane_id() == 0) *a.status = 1;
                return -1;
            }
            return s * a.M + m;
        }
        case SRC_TOKBUF:
        case SRC_REORDER: {
            const int j = r % a.CAP, s = (r / a.CAP) % a.W, e = r / (a.CAP * a.W);
            const int c = a.rc[s * a.E_l + e];
            if (j == 0 && c > a.CAP && a.status && lane_id() == 0) *a.status = 1;
            if (j >= c) return -1;
            if (a.mode == SRC_REORDER) return a.flat_off[s * a.E_l + e] + j;
            const int m = a.src_off[s * a.E_l + e] + j;  // row inside the sender's slot; past M it was dropped by the pack
            if (m >= a.M) {
                if (a.status && lane_id() == 0) *a.status = 1;
                return -1;
            }
            return s * a.M + m;
        }
        case SRC_UNSHUFFLE: {
            const int j = r % a.CAP, s = (r / a.CAP) % a.W, e = r / (a.CAP * a.W);
            return j < a.rc[s * a.E_l + e] ? a.row_off[e * a.W + s] + j : -1;
        }
        default: {  // SRC_RETURN
            const int s = r / a.M, m = r % a.M;
            const int32_t* so = a.src_off + s * a.E_l;
            const int tot = so[a.E_l - 1] + a.rc[s * a.E_l + a.E_l - 1];
            if (m >= tot) return -1;
            const int e = wave_seg(so, a.E_l, m);
            return a.row_off[e * a.W + s] + (m - so[e]);
        }
    }
}

// Rows of a copy that a wave takes together: of 2 to 4 KB two (eight 16-byte loads of a lane in flight instead of four), from as many rows on as
// keep every place on the chip taken, up to where the waves of single rows fill the memory's queues by themselves.  One by one / together, us: 4096 rows
// of 3 KB payload 7.4 / 6.4, unpack 8.1 / 7.7, return 8.1 / 7.8; 8192 of 3.5 KB 13.0 / 11.4, 14.2 / 12.1, 14.5 / 12.8; 12288 of 3 KB 14.6 / 13.3, 16.1 / 14.8,
// 16.5 / 16.0; 13500 payload 3 to 9 % more, the others 1 to 7 % less; but 14800 the others equal, 24576 26.8 / 28.2, 28.4 / 30.0, 28.9 / 30.4, 65536 68 / 71, 69 / 74, 70 / 75.  The fixed-slot pack
// of rows up to 2.5 KB gains at any number (65536 of 2 KB 57 / 51).  Shorter rows gain nothing (8192 of 1 KB 5 to 10 % more).
inline int copy_rows(int mode, int n_rows, int row_vec) {
    if (row_vec <= 2 * WAVE || row_vec > 4 * WAVE || n_rows < 4096) return 1;
    return n_rows <= (mode == SRC_MAP ? 12288 : 14336) || (mode == SRC_PACK && row_vec <= 160) ? 2 : 1;
}
// RPW rows of at most 8 / RPW vectors a lane, row j from src[from[j]] (below 0: zeros) to dst[j]; NT_STORE: non-temporal stores
template <int RPW, bool NT_STORE>
__device__ __forceinline__ void copy_rows_together(const u32x4* const (&from)[RPW], u32x4* const (&to)[RPW], int row_vec, int lane) {
    constexpr int V = 8 / RPW;
    u32x4 v[RPW][V];
#pragma unroll
    for (int j = 0; j < RPW; ++j)
#pragma unroll
        for (int u = 0; u < V; ++u) {
            v[j][u] = u32x4{0u, 0u, 0u, 0u};
            if (from[j] && lane + u * WAVE < row_vec) v[j][u] = __builtin_nontemporal_load(from[j] + lane + u * WAVE);
        }
#pragma unroll
    for (int j = 0; j < RPW; ++j)
#pragma unroll
        for (int u = 0; u < V; ++u)
            if (to[j] && lane + u * WAVE < row_vec) {
                if constexpr (NT_STORE) __builtin_nontemporal_store(v[j][u], to[j] + lane + u * WAVE);
                else to[j][lane + u * WAVE] = v[j][u];
            }
}

template <int WPB, bool RECV, int RPW>
__global__ __launch_bounds__(WPB * WAVE) void gather_rows_kernel(const u32x4* __restrict__ src, u32x4* __restrict__ dst,
                                                                  const RowSource src_of, int n_rows,
                                                                  int row_vec /* 16-byte units per row */, const RecvCounts q) {
    RowSource a = src_of;
    if constexpr (RECV) {
        static_assert(WPB == 4, "one wave per table");
        __shared__ RecvTables tables;
        recv_tables(tables, q, a.W, a.E_l);
        a.rc = tables.rc; a.src_off = tables.src_off; a.row_off = tables.row_off; a.flat_off = tables.flat_off;
    }
    // (row by row the wave's number stays in a vector register: in a scalar one the look-up of a row becomes a chain of scalar loads and divisions
    // that short rows do not cover; 32768 rows of 256 bytes, fixed-slot pack 12.7 us and 11.7, payload 10.3 and 9.8, receive layout 12.9 and 12.1)
    const int wave = RPW > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE) : threadIdx.x / WAVE, lane = lane_id();
    if constexpr (RPW > 1) {
        for (unsigned r0 = (blockIdx.x * WPB + wave) * RPW; r0 < (unsigned)n_rows; r0 += gridDim.x * WPB * RPW) {
            const u32x4* from[RPW];
            u32x4* to[RPW];
#pragma unroll
            for (int j = 0; j < RPW; ++j) {
                const bool live = r0 + j < (unsigned)n_rows;
                const int m = live ? source_row(a, (int)(r0 + j)) : -1;
                from[j] = m >= 0 ? src + (size_t)m * row_vec : nullptr;
                to[j] = live ? dst + (size_t)(r0 + j) * row_vec : nullptr;
            }
            copy_rows_together<RPW, true>(from, to, row_vec, lane);
        }
        return;
    }
    for (int r = blockIdx.x * WPB + wave; r < n_rows; r += gridDim.x * WPB) {
        const int m = source_row(a, r);
        u32x4* d = dst + (size_t)r * row_vec;
        if (m >= 0) {
            // streaming copy: every byte is touched once, so loads and stores bypass cache retention
            const u32x4* s = src + (size_t)m * row_vec;
            int c = lane;
            for (; c + 7 * WAVE < row_vec; c += 8 * WAVE) {
                u32x4 v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = __builtin_nontemporal_load(s + c + u * WAVE);
#pragma unroll
                for (int u = 0; u < 8; ++u) __builtin_nontemporal_store(v[u], d + c + u * WAVE);
            }
            for (; c < row_vec; c += WAVE) __builtin_nontemporal_store(__builtin_nontemporal_load(s + c), d + c);
        } else {
            const u32x4 z = {0u, 0u, 0u, 0u};
            for (int c = lane; c < row_vec; c += WAVE) __builtin_nontemporal_store(z, d + c);
        }
    }
}

// ---- pack, token-major: every token row is read once and stored to its k send slots ------------------
// Units [0, T) of the launch are tokens (one wave each); the units after them are runs of PACK_ZR consecutive send
// slots each, which only get zeros where they are padding (a wave per slot was mostly wave start-up: with skewed
// routing most of the send buffer is padding).  Same bytes in send_buf as the slot-major gather (SRC_PACK), with x
// read once instead of k times.
// Waves per token row of the kernels that give a token to a wave: with few tokens a row is cut into runs of columns (64 vectors at
// least), so that the chip holds some 2048 waves whatever the token count (24 rows of 14 KB, top-8: pack 12.8 -> 7.7 us, combine
// 23 -> 5.8 us: a wave alone walks its row by 1 to 8 KB a memory round trip).
inline int row_parts(int tokens, int row_vec) {
    return max(1, min(2048 / max(tokens, 1), (row_vec + WAVE - 1) / WAVE));
}
// The combine's: also with many tokens, so that the rows of fewer tokens are read at a time -- with a row to a wave 4096 x 8 rows of 14 KB
// are 32768 places in memory at once.  Runs of 2 KB at least and at most four to a row (k = 8: 4096 x 14 KB 104 -> 97 us, 5.5 TB/s;
// 8192 x 4 KB 61 -> 57; k = 2: 8192 x 8 KB 41 -> 36; eight runs 55 where four take 51 and one 54, runs of 1 KB 20 where one takes 17).
// The pack's too (2048 x 14 KB, top-4 43.8 -> 39.1 us, 3000 x 10 KB, top-2 23.4 -> 22.3, 2500 x 14 KB, top-8 78 -> 74; 4096 x 14 KB, top-8 127 -> 129 by
// itself, between the router and the combine 2 us quicker).
inline int combine_parts(int tokens, int row_vec) {
    return tokens < 2048 ? row_parts(tokens, row_vec) : max(1, min(min(16384 / tokens, row_vec / (2 * WAVE)), 4));
}
// Columns [c_lo, c_hi) of a token's row to the rows of send that slots(drow) names (k of them; -1: none).  Eight 16-byte loads in flight per lane (fewer
// at the end of a row, or when the row is shorter than 8 KB), the first ones under way while the slots are looked up.
// KT: the top-k, or 0 for any.  With few tokens the launch is a chain of round trips to memory, and sixteen slots spelt out, most of them jumped
// over, are more of them, for instructions: 256 x 1 KB, top-2, 4.3 -> 3.6 us, 512 x 4 KB, top-1, 5.3 -> 4.6, 24 x 14 KB, top-8, 6.7 -> 6.3; with
// many tokens of short rows they are work: 65536 x 1 KB, top-2, 74 -> 42, 8192 x 1.5 KB, top-2, 13.9 -> 8.6; 4096 x 14 KB, top-8, 115 -> 110.
template <int KT, typename F>
__device__ __forceinline__ void pack_row(const u32x4* __restrict__ src, u32x4* __restrict__ send, int k, int row_vec, int c_lo, int c_hi, int lane, F&& slots) {
    constexpr int KM = topk_slots<KT>();
    u32x4 v[8];
    auto load = [&](int c) {
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (c + u * WAVE < c_hi) v[u] = __builtin_nontemporal_load(src + c + u * WAVE);
    };
    if (KT) load(c_lo + lane);
    int drow[KM];
    slots(drow);
    for (int c = c_lo + lane; c < c_hi; c += 8 * WAVE) {
        if (!KT || c >= c_lo + 8 * WAVE) load(c);
#pragma unroll
        for (int j = 0; j < KM; ++j) {
            if ((KT || j < k) && drow[j] >= 0) {
                u32x4* o = send + (size_t)drow[j] * row_vec + c;
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (c + u * WAVE < c_hi) __builtin_nontemporal_store(v[u], o + u * WAVE);
            }
        }
    }
}
template <int WPB, int KT>
__global__ __launch_bounds__(WPB * WAVE) void pack_tokens_kernel(const u32x4* __restrict__ x, u32x4* __restrict__ send,
                                                                  const int32_t* __restrict__ idx, const int32_t* __restrict__ pos,
                                                                  const int32_t* __restrict__ dst_sizes,
                                                                  const int32_t* __restrict__ dst_offsets, int T, int k_rt, int E_l,
                                                                  int W, int M, int row_vec, int32_t* __restrict__ status,
                                                                  const float* __restrict__ gate, float* __restrict__ send_gate, int parts) {
    // gate / send_gate (both or neither): the slot's top-k gate travels with its row, send_gate[d,m] = gate[t,kk], zero
    // in the padding slots -- for a destination that applies the gate to the expert's result before sending it back
    // parts: waves per token, each with its own run of columns (see row_parts)
    constexpr int KM = topk_slots<KT>();
    const int wave = threadIdx.x / WAVE, lane = lane_id(), k = KT ? KT : k_rt;
    const int n_slots = W * M, n_tok = T * parts;
    const int per = ((row_vec + parts - 1) / parts + WAVE - 1) / WAVE * WAVE;
    const int n_units = n_tok + (n_slots + PACK_ZR - 1) / PACK_ZR;
    for (int unit = blockIdx.x * WPB + wave; unit < n_units; unit += gridDim.x * WPB) {
        if (unit >= n_tok) {
            const int s0 = (unit - n_tok) * PACK_ZR, s1 = min(s0 + PACK_ZR, n_slots);
            int d = s0 / M, m = s0 % M;
            int cnt = dst_sizes[d];
            const u32x4 z = {0u, 0u, 0u, 0u};
            for (int sl = s0; sl < s1; ++sl) {
                if (m == 0 && cnt > M && status && lane == 0) *status = 1;
                if (m >= cnt) {
                    u32x4* o = send + (size_t)sl * row_vec;
                    // (ordinary stores: measured 4 to 10 % faster here than non-temporal ones, which win for the copies below)
                    for (int c = lane; c < row_vec; c += WAVE) o[c] = z;
                    if (send_gate && lane == 0) send_gate[sl] = 0.f;
                }
                if (++m == M && sl + 1 < s1) { m = 0; cnt = dst_sizes[++d]; }
            }
            continue;
        }
        const int r = unit / parts, c_lo = (unit % parts) * per, c_hi = min(c_lo + per, row_vec);
        // destination rows of the token's k slots (-1: beyond the pair capacity, dropped like the gather drops it)
        pack_row<KT>(x + (size_t)r * row_vec, send, k, row_vec, c_lo, c_hi, lane, [&](int (&drow)[KM]) {
#pragma unroll
            for (int j = 0; j < KM; ++j) {
                drow[j] = -1;
                if (KT || j < k) {
                    const int d = idx[(size_t)r * k + j] / E_l;
                    const bool d_ok = (unsigned)d < (unsigned)W;  // (an expert id outside [0, W E_l): no slot, and no read of its offset)
                    const int m = pos[(size_t)r * k + j] - dst_offsets[d_ok ? d : 0];
                    if (d_ok && (unsigned)m < (unsigned)M) drow[j] = d * M + m;
                    if (send_gate && drow[j] >= 0 && lane == 0 && c_lo == 0) send_gate[drow[j]] = gate[(size_t)r * k + j];
                }
            }
        });
    }
}

// ---- quantise and pack in one pass: the token rows leave the source as fp8 codes and one scale per row -----------------
// Per-row quantisation commutes with moving rows: send_q / send_scale hold, slot for slot, what quantize_rows_fp8 would make
// of the bf16 send buffer (padding slots: codes 0, scale 1, as for an all-zero row) -- so the destination can feed them to
// the fp8 GEMM as they arrive, and half the bytes cross.  Units [0, T) of the launch are tokens (one wave each: the row is
// read once, quantised in registers, stored to its k slots); the units after them are runs of PACK_ZR slots that are
// written only where they are padding.
// A token: its row of nv 16-byte vectors, asked for before its slots are looked up (NV to a lane in registers; 0: read twice), a form for each usual
// top-k (see pack_row): 3500 x 4 KB, top-8 22.7 -> 19.7 us, 3000 x 10 KB, top-2 22.0 -> 19.0, 16384 x 2 KB, top-8 44 -> 40; 4096 x 8 KB, top-4 27.7 -> 28.6.
template <int KT, int NV, typename F>
__device__ __forceinline__ void pack_row_fp8(const uint4* __restrict__ src, uint8_t* __restrict__ send_q, float* __restrict__ send_scale, int k, int nv,
                                             int lane, F&& slots) {
    constexpr int KM = topk_slots<KT>();
    const size_t cols = (size_t)nv * 8;
    uint4 held[NV > 0 ? NV : 1];
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = lane + i * WAVE;
        held[i] = c < nv ? src[c] : make_uint4(0, 0, 0, 0);
    }
    int drow[KM];
    slots(drow);
    if constexpr (NV > 0) {
#pragma unroll
        for (int i = 0; i < NV; ++i) amax = fp8_row_amax(held[i], amax);
    } else {
        for (int c = lane; c < nv; c += WAVE) amax = fp8_row_amax(src[c], amax);
    }
    amax = __int_as_float(wave_max0(__float_as_int(amax)));  // (never NaN, never below 0: the bits are ordered alike)
    const bool zero = amax == 0.f;
    const float inv = zero ? 1.f : __fdiv_rn(448.f, amax);
    const float sc = zero ? 1.f : __fdiv_rn(amax, 448.f);
    if constexpr (NV > 0) {
        uint2 code[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) code[i] = fp8_row_convert(held[i], inv);
#pragma unroll
        for (int j = 0; j < KM; ++j) {
            if ((KT || j < k) && drow[j] >= 0) {
                uint2* o = (uint2*)(send_q + (size_t)drow[j] * cols);
#pragma unroll
                for (int i = 0; i < NV; ++i) {
                    const int c = lane + i * WAVE;
                    if (c < nv) o[c] = code[i];
                }
                if (lane == 0) send_scale[drow[j]] = sc;
            }
        }
    } else {
        for (int c = lane; c < nv; c += WAVE) {
            const uint2 code = fp8_row_convert(src[c], inv);
#pragma unroll
            for (int j = 0; j < KM; ++j)
                if ((KT || j < k) && drow[j] >= 0) ((uint2*)(send_q + (size_t)drow[j] * cols))[c] = code;
        }
#pragma unroll
        for (int j = 0; j < KM; ++j)
            if ((KT || j < k) && drow[j] >= 0 && lane == 0) send_scale[drow[j]] = sc;
    }
}
template <int KT, int NV>
__global__ __launch_bounds__(256) void pack_tokens_fp8_kernel(const bf16_t* __restrict__ x, int T, int cols,
                                                               const int32_t* __restrict__ idx, const int32_t* __restrict__ pos,
                                                               const int32_t* __restrict__ dst_sizes,
                                                               const int32_t* __restrict__ dst_offsets, int k_rt, int E_l, int W, int M,
                                                               uint8_t* __restrict__ send_q, float* __restrict__ send_scale,
                                                               int32_t* __restrict__ status, const float* __restrict__ gate,
                                                               float* __restrict__ send_gate) {
    // (gate / send_gate, both or neither: the slot's top-k gate travels with its row, zero in the padding slots)
    constexpr int KM = topk_slots<KT>();
    const int wave = threadIdx.x / WAVE, lane = lane_id(), k = KT ? KT : k_rt;
    const int nv = cols / 8;  // 16-byte vectors of bf16 per row = 8-byte vectors of codes
    const int n_slots = W * M;
    const int n_units = T + (n_slots + PACK_ZR - 1) / PACK_ZR;
    for (int r = blockIdx.x * 4 + wave; r < n_units; r += gridDim.x * 4) {
        if (r >= T) {
            const int s0 = (r - T) * PACK_ZR, s1 = min(s0 + PACK_ZR, n_slots);
            int d = s0 / M, m = s0 % M;
            int cnt = dst_sizes[d];
            for (int sl = s0; sl < s1; ++sl) {
                if (m == 0 && cnt > M && status && lane == 0) *status = 1;
                if (m >= cnt) {
                    uint2* o = (uint2*)(send_q + (size_t)sl * cols);
                    for (int c = lane; c < nv; c += WAVE) o[c] = make_uint2(0u, 0u);
                    if (lane == 0) send_scale[sl] = 1.f;
                    if (send_gate && lane == 0) send_gate[sl] = 0.f;
                }
                if (++m == M && sl + 1 < s1) { m = 0; cnt = dst_sizes[++d]; }
            }
            continue;
        }
        pack_row_fp8<KT, NV>((const uint4*)(x + (size_t)r * cols), send_q, send_scale, k, nv, lane, [&](int (&drow)[KM]) {
#pragma unroll
            for (int j = 0; j < KM; ++j) {
                drow[j] = -1;
                if (KT || j < k) {
                    const int d = idx[(size_t)r * k + j] / E_l;
                    const bool d_ok = (unsigned)d < (unsigned)W;
                    const int m = pos[(size_t)r * k + j] - dst_offsets[d_ok ? d : 0];
                    if (d_ok && (unsigned)m < (unsigned)M) drow[j] = d * M + m;
                    if (send_gate && drow[j] >= 0 && lane == 0) send_gate[drow[j]] = gate[(size_t)r * k + j];
                }
            }
        });
    }
}

// Count and pack of few tokens in one launch: every wave works out for itself where its token's rows go, from the expert ids of all slots (a few
// KB, from L2), so nothing has to wait for a ranking in front.  The row of a slot is the slots of lower experts plus those of its own in earlier
// tokens; with key = expert * T k + slot (a token holds an expert at most once) that is the number of smaller keys, and the keys below the first of
// its destination's experts are the rows in front of the destination: a compare, a ballot and a bit count for 64 slots.
// Block 0 counts the experts and leaves the tables; blocks 1 to side_blocks prepare the receive side (see rank_kernel); the others are the
// units of pack_tokens_kernel, whose bytes these are.  M = 0: the padding-free payload, row = position.
// What it saves is the ranking's launch, most of whose time is its start and a chain of small steps.  A step of 256 fp32 tokens x 1 KB, top-2, 34.7 -> 31.8 us;
// 512 x 4 KB, top-1, 66.6 -> 63.8; 24 x 14 KB, top-8, 352 -> 349; 777 x 4 KB, top-2, flat, 111.5 -> 106.8; quantised, 64 x 4 KB, top-2 of 64, 36.9 -> 33.5.
struct CountOut {
    int32_t *send_counts, *expert_offs, *dst_sizes, *dst_offsets, *caps, *pos, *row_token;
};
template <int KT, int NV /* -1: the rows as they are, 16-byte vectors; else quantised (pack_row_fp8), 8-byte vectors of codes */>
__global__ __launch_bounds__(256) void count_pack_kernel(const u32x4* __restrict__ x, void* __restrict__ send, float* __restrict__ send_scale, const int32_t* __restrict__ idx, int T, int k_rt,
                                                          int E, int W, int M, int row_vec, const CountOut out, int32_t* __restrict__ status,
                                                          const float* __restrict__ gate, float* __restrict__ send_gate, int parts, int side_blocks,
                                                          const RecvPrepare side) {
    __shared__ int32_t tot[MOE_MAX_EXPERTS], es[MOE_MAX_EXPERTS + 1];
    extern __shared__ int32_t copies[];  // [RANK_COPIES][E | 1]
    constexpr int KM = topk_slots<KT>();
    const int tid = threadIdx.x, lane = lane_id(), k = KT ? KT : k_rt, n = T * k, E_l = E / W;
    if (blockIdx.x == 0) {
        const int stride = E | 1;
        for (int i = tid; i < RANK_COPIES * stride; i += 256) copies[i] = 0;
        __syncthreads();
#pragma unroll 4
        for (int i = tid; i < n; i += 256) {
            const int e = idx[i];
            if ((unsigned)e < (unsigned)E) atomicAdd(&copies[lane % RANK_COPIES * stride + e], 1);
        }
        __syncthreads();
        for (int e = tid; e < E; e += 256) {
            int c = 0;
#pragma unroll
            for (int i = 0; i < RANK_COPIES; ++i) c += copies[i * stride + e];
            tot[e] = c;
        }
        __syncthreads();
        if (tid < WAVE) offsets_body(tot, E, W, es, true, out.send_counts, out.expert_offs, out.dst_sizes, out.dst_offsets, out.caps);
        return;
    }
    if ((int)blockIdx.x <= side_blocks) {
        recv_prepare_block(side, blockIdx.x - 1, es, tot);
        return;
    }
    // f(keys of 8 x 64 slots: a lane's own; ids outside [0, E) and slots past the end above all others)
    auto keys = [&](auto f) {
        for (int i0 = 0; i0 < n; i0 += 8 * WAVE) {
            unsigned key[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int i = i0 + u * WAVE + lane;
                const int e = i < n ? idx[i] : -1;
                key[u] = (unsigned)e < (unsigned)E ? (unsigned)(e * n + i) : ~0u;
            }
            f(key);
        }
    };
    const int n_slots = W * M, n_tok = T * parts, per = ((row_vec + parts - 1) / parts + WAVE - 1) / WAVE * WAVE;
    const int n_units = n_tok + (n_slots + PACK_ZR - 1) / PACK_ZR, first = ((int)blockIdx.x - 1 - side_blocks) * 4 + tid / WAVE;
    for (int unit = __builtin_amdgcn_readfirstlane(first); unit < n_units; unit += (gridDim.x - 1 - side_blocks) * 4) {
        if (unit >= n_tok) {
            const int s0 = (unit - n_tok) * PACK_ZR, s1 = min(s0 + PACK_ZR, n_slots);
            int d = s0 / M, m = s0 % M;
            auto size_of = [&](int q) {
                int c = 0;
                keys([&](const unsigned (&key)[8]) {
#pragma unroll
                    for (int u = 0; u < 8; ++u) c += __popcll(__ballot(key[u] - (unsigned)(q * E_l * n) < (unsigned)(E_l * n)));
                });
                return c;
            };
            int cnt = size_of(d);
            typedef typename std::conditional<(NV < 0), u32x4, uint2>::type vec;
            const vec z = {};
            for (int sl = s0; sl < s1; ++sl) {
                if (m == 0 && cnt > M && status && lane == 0) *status = 1;
                if (m >= cnt) {
                    vec* o = (vec*)send + (size_t)sl * row_vec;
                    for (int c = lane; c < row_vec; c += WAVE) o[c] = z;
                    if (NV >= 0 && lane == 0) send_scale[sl] = 1.f;
                    if (send_gate && lane == 0) send_gate[sl] = 0.f;
                }
                if (++m == M && sl + 1 < s1) { m = 0; cnt = size_of(++d); }
            }
            continue;
        }
        const int r = unit / parts, c_lo = (unit % parts) * per, c_hi = min(c_lo + per, row_vec);
        auto slots = [&](int (&drow)[KM]) {
            int e[KM], p[KM] = {}, before[KM] = {};
#pragma unroll
            for (int j = 0; j < KM; ++j) e[j] = KT || j < k ? idx[r * k + j] : -1;
            keys([&](const unsigned (&key)[8]) {
#pragma unroll
                for (int j = 0; j < KM; ++j) {
                    if (KT || j < k) {
                        const unsigned own = (unsigned)(e[j] * n + r * k), dst = (unsigned)(e[j] / E_l * E_l * n);
#pragma unroll
                        for (int u = 0; u < 8; ++u) {
                            p[j] += __popcll(__ballot(key[u] < own));
                            before[j] += __popcll(__ballot(key[u] < dst));
                        }
                    }
                }
            });
#pragma unroll
            for (int j = 0; j < KM; ++j) {
                drow[j] = -1;
                if ((KT || j < k) && (unsigned)e[j] < (unsigned)E) {
                    const int m = p[j] - before[j];
                    drow[j] = M == 0 ? p[j] : m < M ? e[j] / E_l * M + m : -1;
                    if (c_lo == 0 && lane == 0) {
                        out.pos[r * k + j] = p[j];
                        out.row_token[p[j]] = r;
                        if (send_gate && drow[j] >= 0) send_gate[drow[j]] = gate[r * k + j];
                    }
                }
            }
        };
        if constexpr (NV < 0) pack_row<KT>(x + (size_t)r * row_vec, (u32x4*)send, k, row_vec, c_lo, c_hi, lane, slots);
        else pack_row_fp8<KT, NV>((const uint4*)x + (size_t)r * row_vec, (uint8_t*)send, send_scale, k, row_vec, lane, slots);
    }
}

// ---- combine: out[t,:] = sum_kk gate[t,kk] * ret[slot(t,kk),:] --------------------------------------
template <typename XT>
struct Vec16;
template <>
struct Vec16<bf16_t> {
    static constexpr int N = 8;
    __device__ static void unpack(const uint4& v, float* f) {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) { f[2 * i] = __uint_as_float(w[i] << 16); f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u); }
    }
    __device__ static uint4 pack(const float* f) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = (uint32_t)f32_to_bf16(f[2 * i]) | ((uint32_t)f32_to_bf16(f[2 * i + 1]) << 16);
        return make_uint4(w[0], w[1], w[2], w[3]);
    }
};
template <>
struct Vec16<float> {
    static constexpr int N = 4;
    __device__ static void unpack(const uint4& v, float* f) {
        f[0] = __uint_as_float(v.x); f[1] = __uint_as_float(v.y); f[2] = __uint_as_float(v.z); f[3] = __uint_as_float(v.w);
    }
    __device__ static uint4 pack(const float* f) {
        return make_uint4(__float_as_uint(f[0]), __float_as_uint(f[1]), __float_as_uint(f[2]), __float_as_uint(f[3]));
    }
};

// KT = compile-time top-k (1,2,4,8) or 0 for a run-time k up to MOE_MAX_TOPK.  All k row reads of a
// 16-byte column are issued before the first is used.
template <typename XT, int KT, int WPB>
__global__ __launch_bounds__(WPB * WAVE) void combine_kernel(const uint4* __restrict__ ret, const int32_t* __restrict__ idx,
                                                              const int32_t* __restrict__ pos, const float* __restrict__ gate,
                                                              const int32_t* __restrict__ dst_offsets, int T, int k_rt, int E_l,
                                                              int W, int M, int row_vec, uint4* __restrict__ out,
                                                              int32_t* __restrict__ status, int parts) {
    constexpr int N = Vec16<XT>::N;
    constexpr int KMAX = KT ? KT : MOE_MAX_TOPK;
    const int k = KT ? KT : k_rt;
    const int wave = threadIdx.x / WAVE, lane = lane_id();
    const int per = ((row_vec + parts - 1) / parts + WAVE - 1) / WAVE * WAVE;  // columns per wave (see combine_parts)
    for (int unit = blockIdx.x * WPB + wave; unit < T * parts; unit += gridDim.x * WPB) {
        const int t = unit / parts, c_lo = (unit % parts) * per, c_hi = min(c_lo + per, row_vec);
        // a slot whose destination or row lies outside the [W,M] layout was dropped by the pack (pair capacity
        // exceeded) and has no returned row: it is skipped, like the pack skipped it, and the status word is raised
        size_t rows[KMAX];
        float g[KMAX];
        bool have[KMAX];
#pragma unroll
        for (int j = 0; j < KMAX; ++j) {
            have[j] = false;
            if (j < k) {
                const int d = idx[(size_t)t * k + j] / E_l;
                const bool d_ok = (unsigned)d < (unsigned)W;
                const int m = pos[(size_t)t * k + j] - dst_offsets[d_ok ? d : 0];
                have[j] = d_ok && (unsigned)m < (unsigned)M;
                rows[j] = have[j] ? ((size_t)d * M + m) * row_vec : 0;
                g[j] = gate ? gate[(size_t)t * k + j] : 1.f;  // (no gates: the rows arrive weighted, 1 * x is x exactly)
                if (!have[j] && status && lane == 0) *status = 1;
            }
        }
        // U columns per lane and pass, so that sixteen 16-byte row reads are in flight per lane whatever k is
        constexpr int U = KT == 0 || KT >= 16 ? 1 : 16 / (KT ? KT : 1);
        for (int c0 = c_lo + lane; c0 < c_hi; c0 += U * WAVE) {
            uint4 v[U][KMAX];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int c = c0 + u * WAVE;
#pragma unroll
                for (int j = 0; j < KMAX; ++j)
                    if (j < k && have[j] && c < c_hi) {
                        // every returned row is read once: no cache retention wanted
                        const u32x4 raw = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(ret + rows[j] + c));
                        v[u][j] = make_uint4(raw.x, raw.y, raw.z, raw.w);
                    }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int c = c0 + u * WAVE;
                if (c >= c_hi) break;
                float acc[N];
#pragma unroll
                for (int i = 0; i < N; ++i) acc[i] = 0.f;
#pragma unroll
                for (int j = 0; j < KMAX; ++j) {
                    if (j < k && have[j]) {
                        float f[N];
                        Vec16<XT>::unpack(v[u][j], f);
#pragma unroll
                        for (int i = 0; i < N; ++i) acc[i] = __fadd_rn(acc[i], __fmul_rn(g[j], f[i]));
                    }
                }
                const uint4 o = Vec16<XT>::pack(acc);
                const u32x4 ov = {o.x, o.y, o.z, o.w};
                // (non-temporal: an ordinary store is 2 to 4 % faster with 8 KB and 14 KB rows and 6 to 11 % slower with 4 KB rows)
                __builtin_nontemporal_store(ov, reinterpret_cast<u32x4*>(out + (size_t)t * row_vec + c));
            }
        }
    }
}

// ---- gradient of the combine: out[t] = sum_kk gate[t,kk] * ret[slot(t,kk)] ------------------------------------------
//   d ret[slot(t,kk)] = gate[t,kk] * d out[t]        (every slot belongs to one (t,kk): a scatter, like the pack)
//   d gate[t,kk]      = < d out[t], ret[slot(t,kk)] > (fp32 sum over the row: per-lane partial sums in column order, then
//                                                     a butterfly over the lanes -- reproducible from call to call)
// The first workgroups take the tokens: a wave each (WPT = 1) or all waves together, whose sums then meet in LDS in wave order; the
// others take runs of PACK_ZR slots of d ret, which only get zeros when they are padding (no (t,kk) maps there) -- as in
// pack_tokens_kernel.  Dropped slots (outside [W,M]) get no
// gradient.  A pass takes U columns of the token's d out and of its k slot rows together (some sixteen 16-byte loads in flight
// per lane): d out is read once, not k times (4096 tokens x 8 rows of 14 KB: 299 -> 266 us, 4.4 TB/s with the padding).
// dst_sizes == NULL: a destination's rows end where the next one's start (n_routed rows in all).
template <typename XT, int KT, int WPB, int WPT /* waves per token: 1 or WPB */>
__global__ __launch_bounds__(WPB * WAVE) void combine_backward_kernel(const uint4* __restrict__ dout, const uint4* __restrict__ ret,
                                                                       const int32_t* __restrict__ idx, const int32_t* __restrict__ pos,
                                                                       const float* __restrict__ gate,
                                                                       const int32_t* __restrict__ dst_sizes,
                                                                       const int32_t* __restrict__ dst_offsets, int T, int k_rt, int E_l,
                                                                       int W, int M, int row_vec, uint4* __restrict__ dret,
                                                                       float* __restrict__ dgate) {
    constexpr int N = Vec16<XT>::N;
    constexpr int KMAX = KT ? KT : MOE_MAX_TOPK;
    constexpr int U = KT ? (KT >= 8 ? 2 : KT >= 4 ? 4 : 8) : 1;
    const int k = KT ? KT : k_rt;
    static_assert(WPT == 1 || WPT == WPB, "a token to a wave or to a workgroup");
    __shared__ float part[WPT == 1 ? 1 : WPT][KMAX];
    const int wave = threadIdx.x / WAVE, lane = lane_id();
    // token rows first, WPB / WPT to a workgroup, in workgroups of their own; then the runs of slots, WPB to a workgroup
    const int n_slots = W * M, n_runs = (n_slots + PACK_ZR - 1) / PACK_ZR;
    const int tok_blocks = (T + WPB / WPT - 1) / (WPB / WPT), n_blocks = tok_blocks + (n_runs + WPB - 1) / WPB;
    for (int b = blockIdx.x; b < n_blocks; b += gridDim.x) {
        const int r = WPT == 1 ? b * WPB + wave : b, c_first = WPT == 1 ? lane : (int)threadIdx.x;
        if (b >= tok_blocks) {
            const int run = (b - tok_blocks) * WPB + wave;
            if (run >= n_runs) continue;
            const int s0 = run * PACK_ZR, s1 = min(s0 + PACK_ZR, n_slots);
            int d = s0 / M, m = s0 % M;
            auto size_of = [&](int q) { return dst_sizes ? dst_sizes[q] : (q + 1 < W ? dst_offsets[q + 1] : T * k) - dst_offsets[q]; };
            int cnt = size_of(d);
            for (int sl = s0; sl < s1; ++sl) {
                if (m >= cnt) {
                    uint4* o = dret + (size_t)sl * row_vec;
                    for (int c = lane; c < row_vec; c += WAVE) o[c] = make_uint4(0, 0, 0, 0);
                }
                if (++m == M && sl + 1 < s1) { m = 0; cnt = size_of(++d); }
            }
            continue;
        }
        if (r >= T) continue;
        const uint4* drow = dout + (size_t)r * row_vec;
        size_t slot[KMAX];
        float g[KMAX], dot[KMAX];
        bool have[KMAX];
#pragma unroll
        for (int j = 0; j < KMAX; ++j) {
            have[j] = false;
            dot[j] = 0.f;
            if (j < k) {
                const int d = idx[(size_t)r * k + j] / E_l;
                const bool d_ok = (unsigned)d < (unsigned)W;
                const int m = pos[(size_t)r * k + j] - dst_offsets[d_ok ? d : 0];
                have[j] = d_ok && (unsigned)m < (unsigned)M;
                slot[j] = have[j] ? ((size_t)d * M + m) * row_vec : 0;
                g[j] = gate[(size_t)r * k + j];
            }
        }
        constexpr int CS = WPT * WAVE;  // columns from one to the next of a lane
        for (int c0 = c_first; c0 < row_vec; c0 += U * CS) {
            uint4 dv4[U], rv4[U][KMAX];
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (c0 + u * CS < row_vec) {
                    dv4[u] = drow[c0 + u * CS];
#pragma unroll
                    for (int j = 0; j < KMAX; ++j)
                        if (j < k && have[j]) {
                            const u32x4 raw = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(ret + slot[j] + c0 + u * CS));
                            rv4[u][j] = make_uint4(raw.x, raw.y, raw.z, raw.w);
                        }
                }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (c0 + u * CS >= row_vec) break;
                float dv[N];
                Vec16<XT>::unpack(dv4[u], dv);
#pragma unroll
                for (int j = 0; j < KMAX; ++j)
                    if (j < k && have[j]) {
                        float rv[N], ov[N];
                        Vec16<XT>::unpack(rv4[u][j], rv);
#pragma unroll
                        for (int i = 0; i < N; ++i) {
                            dot[j] = __fadd_rn(dot[j], __fmul_rn(dv[i], rv[i]));
                            ov[i] = __fmul_rn(g[j], dv[i]);
                        }
                        const uint4 o = Vec16<XT>::pack(ov);
                        const u32x4 o4 = {o.x, o.y, o.z, o.w};
                        __builtin_nontemporal_store(o4, reinterpret_cast<u32x4*>(dret + slot[j] + c0 + u * CS));
                    }
            }
        }
#pragma unroll
        for (int j = 0; j < KMAX; ++j)
            if (j < k) {
                wave_butterfly([&](auto off) { dot[j] = __fadd_rn(dot[j], __int_as_float(wave_xor<decltype(off)::value>(__float_as_int(dot[j])))); });
                if (lane == 0) {
                    if constexpr (WPT == 1) dgate[(size_t)r * k + j] = dot[j];
                    else part[wave][j] = dot[j];
                }
            }
        if constexpr (WPT > 1) {
            __syncthreads();
            if ((int)threadIdx.x < k) {
                float sum = part[0][threadIdx.x];
#pragma unroll
                for (int w = 1; w < WPT; ++w) sum = __fadd_rn(sum, part[w][threadIdx.x]);
                dgate[(size_t)r * k + threadIdx.x] = sum;
            }
            __syncthreads();
        }
    }
}

template <typename XT>
int launch_combine(const void* ret, const int32_t* idx, const int32_t* pos, const float* gate, const int32_t* dst_offsets, int T,
                   int k, int E_l, int W, int M, int row_vec, void* out, int32_t* status, hipStream_t s) {
    const int parts = combine_parts(T, row_vec);
    const int blocks = min(ceil_div(T * parts, 4), 65535 * 8);
#define MOE_COMBINE(KT) \
    combine_kernel<XT, KT, 4><<<blocks, 4 * WAVE, 0, s>>>((const uint4*)ret, idx, pos, gate, dst_offsets, T, k, E_l, W, M, row_vec, (uint4*)out, status, parts)
    switch (k) {
        case 1: MOE_COMBINE(1); break;
        case 2: MOE_COMBINE(2); break;
        case 4: MOE_COMBINE(4); break;
        case 8: MOE_COMBINE(8); break;
        default: MOE_COMBINE(0); break;
    }
#undef MOE_COMBINE
    return moe_check_launch("combine");
}

int gather_rows(const void* src, void* dst, const RowSource& a, int n_rows, int row_bytes, hipStream_t s) {
    if (n_rows == 0) return MOE_OK;
    const int rpw = copy_rows(a.mode, n_rows, row_bytes / 16), blocks = min(ceil_div(n_rows, 4 * rpw), 65535 * 8);
#define MOE_GATHER(R) gather_rows_kernel<4, false, R><<<blocks, 4 * WAVE, 0, s>>>((const u32x4*)src, (u32x4*)dst, a, n_rows, row_bytes / 16, RecvCounts{})
    if (rpw == 2) MOE_GATHER(2);
    else MOE_GATHER(1);
#undef MOE_GATHER
    return moe_check_launch("gather_rows");
}
__global__ __launch_bounds__(256) void zero_padding_rows_kernel(u32x4* __restrict__ buf, const int32_t* __restrict__ rc, int W, int E_l,
                                                                 int M, int row_vecs, int run) {
    zero_padding_rows(buf, rc, W, E_l, M, row_vecs, blockIdx.x, run);
}

__global__ __launch_bounds__(256) void row_map_from_counts_kernel(const RecvPrepare a) {
    __shared__ int32_t s_row_off[MOE_MAX_EXPERTS + 1];
    __shared__ int32_t s_src_off[MOE_MAX_EXPERTS];
    recv_prepare_block(a, blockIdx.x, s_row_off, s_src_off);
}

int check_rows(const char* who, int dtype, int H) {
    if (dtype != MOE_F32 && dtype != MOE_BF16) return moe_fail(MOE_ERR_INVALID, "%s: dtype %d", who, dtype);
    if (H <= 0 || (H * dtype_size(dtype)) % 16 != 0)
        return moe_fail(MOE_ERR_INVALID, "%s: rows must be 16-byte multiples (H=%d)", who, H);
    return MOE_OK;
}

// The exchange of a simulated world (moe_a2a_place), up to A2A_SRC sources to a launch (their pointers travel as kernel
// arguments).  A workgroup makes the tables of its sources in LDS, then its waves copy or zero rows (e, s, j) of token_buf.
constexpr int A2A_SRC = MOE_A2A_SOURCES;
struct A2aSources {
    moe_a2a_source src[A2A_SRC];
};
__device__ __forceinline__ int a2a_count(const moe_a2a_source& q, int e) { return q.payload ? max(q.counts[e], 0) : 0; }

// A value for a waiting host (moe_wait_i32): visible as soon as it is stored, not only when the kernel ends.
__device__ __forceinline__ void tell_host(int32_t* out, int32_t v) {
    __threadfence_system();  // (what was written for the host before goes first)
    __hip_atomic_store(out, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// out[0] <- the result (last launch only: the host may be waiting for it), out[1]: what earlier launches found
__global__ __launch_bounds__(256) void a2a_max_count_kernel(const A2aSources q, int ns, int E_l, int32_t* __restrict__ out, bool first,
                                                             bool last) {
    __shared__ int32_t most;
    if (threadIdx.x == 0) most = first ? 0 : out[1];
    __syncthreads();
    int c = 0;
    for (int i = threadIdx.x; i < ns * E_l; i += blockDim.x) c = max(c, a2a_count(q.src[i / E_l], i % E_l));
    c = wave_max0(c);  // (one atomic a wave: 256 of them on one word follow each other)
    if (lane_id() == 0) atomicMax(&most, c);
    __syncthreads();
    if (threadIdx.x == 0) {
        if (last) tell_host(out, most);
        else out[1] = most;
    }
}

template <int RPW>
__global__ __launch_bounds__(256) void a2a_place_kernel(const A2aSources q, int s0, int ns, int W, int E_l, int CAP, int row_vec,
                                                         u32x4* __restrict__ token_buf, int32_t* __restrict__ pca,
                                                         int32_t* __restrict__ counts_ready, int n_ready,
                                                         int32_t* __restrict__ token_sync, int n_sync) {
    // Every workgroup finds the places of all rows, in front of its first one: all counts and starts in one trip to memory, then a scan for each source.  (Counts, then
    // starts, then a source's experts one after the other: 24000 rows of 1.5 KB from 8 sources to 32 experts 16.7 us, now 16.1.)
    __shared__ int32_t cnt[MOE_MAX_EXPERTS], off[MOE_MAX_EXPERTS], start[A2A_SRC];
    __shared__ bool over[256 / WAVE];
    const int tid = threadIdx.x, lane = lane_id();
    bool mine = false;
    for (int i = tid; i < ns * E_l; i += blockDim.x) {
        const int c = a2a_count(q.src[i / E_l], i % E_l);
        cnt[i] = c;
        mine |= c > CAP;
    }
    if (tid < ns) start[tid] = q.src[tid].payload ? *q.src[tid].start : 0;
    const bool any = __ballot(mine) != 0;
    if (lane == 0) over[tid / WAVE] = any;
    __syncthreads();
    if (over[0] || over[1] || over[2] || over[3]) return;
    for (int s = tid / WAVE; s < ns; s += blockDim.x / WAVE) {
        int run = start[s];
        for (int e0 = 0; e0 < E_l; e0 += WAVE) {
            const int e = e0 + lane, c = e < E_l ? cnt[s * E_l + e] : 0, incl = wave_incl_scan(c);
            if (e < E_l) off[s * E_l + e] = run + incl - c;
            run += wave_lane(incl, WAVE - 1);
        }
    }
    if (blockIdx.x == 0) {
        for (int i = tid; i < ns * E_l; i += blockDim.x) pca[(i % E_l) * W + s0 + i / E_l] = cnt[i];
        for (int i = tid; i < n_ready; i += blockDim.x) counts_ready[i] = W;
        for (int i = tid; i < n_sync; i += blockDim.x) token_sync[i] = W;
    }
    __syncthreads();
    const int wave = RPW > 1 ? __builtin_amdgcn_readfirstlane(tid / WAVE) : tid / WAVE, wpb = blockDim.x / WAVE;  // (as in gather_rows_kernel: 65536 rows of 3 KB 67 and 60 us)
    const unsigned n_rows = (unsigned)(E_l * ns * CAP);
    // row r of the launch: (e, s, j); the source's row, or NULL: zeros
    auto row = [&](unsigned r, u32x4*& to) -> const u32x4* {
        const int j = (int)(r % CAP), s = (int)(r / CAP) % ns, e = (int)(r / CAP) / ns;
        to = token_buf + (((size_t)e * W + s0 + s) * CAP + j) * row_vec;
        const long long at = (long long)off[s * E_l + e] + j;
        return j < cnt[s * E_l + e] && at >= 0 && at < q.src[s].rows ? (const u32x4*)q.src[s].payload + (size_t)at * row_vec : nullptr;
    };
    for (unsigned r0 = (blockIdx.x * wpb + wave) * RPW; r0 < n_rows; r0 += gridDim.x * wpb * RPW) {
        const u32x4* from[RPW];
        u32x4* to[RPW];
#pragma unroll
        for (int i = 0; i < RPW; ++i) {
            from[i] = nullptr;
            to[i] = nullptr;
            if (r0 + i < n_rows) from[i] = row(r0 + i, to[i]);
        }
        if constexpr (RPW > 1) {
            copy_rows_together<RPW, false>(from, to, row_vec, lane);
        } else if (from[0]) {
            int c = lane;
            for (; c + 3 * WAVE < row_vec; c += 4 * WAVE) {
                u32x4 v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = __builtin_nontemporal_load(from[0] + c + u * WAVE);
#pragma unroll
                for (int u = 0; u < 4; ++u) to[0][c + u * WAVE] = v[u];
            }
            for (; c < row_vec; c += WAVE) to[0][c] = __builtin_nontemporal_load(from[0] + c);
        } else {
            const u32x4 z = {0u, 0u, 0u, 0u};
            for (int c = lane; c < row_vec; c += WAVE) to[0][c] = z;
        }
    }
}

__global__ __launch_bounds__(256) void shuffle_totals_kernel(const int32_t* __restrict__ pca, int n, const int32_t* __restrict__ sync,
                                                              int n_sync, int32_t* __restrict__ out) {
    __shared__ int32_t sum, least;
    if (threadIdx.x == 0) { sum = 0; least = 0x7fffffff; }
    __syncthreads();
    int s = 0, m = 0x7fffffff;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += pca[i];
    for (int i = threadIdx.x; i < n_sync; i += blockDim.x) m = min(m, sync[i]);
    s = wave_sum(s);
    wave_butterfly([&](auto off) { m = min(m, wave_xor<decltype(off)::value>(m)); });
    if (lane_id() == 0) {
        atomicAdd(&sum, s);
        atomicMin(&least, m);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        out[1] = least;
        tell_host(out, sum);
    }
}

}  // namespace

// Histogram cells that the ranking workgroups may read in all (the square of the tokens) before the scan in front of them, a third launch,
// is the better choice.  Sums against scan in us: 8 experts 10.4 / 13.2 (65536 tokens, 2 M cells) and 14.0 / 12.6 (131072, 8 M);
// 256 experts 11.7 / 12.7 (8192, 1 M), 13.5 / 13.1 (16384, 4 M), 17.2 / 14.0 (32768, 16 M) and 181 / 43 (262144, 1 G); 512 experts
// 14.4 / 13.6 (8192, 2 M) and 18.1 / 14.0 (16384, 8 M).
constexpr long long RANK_SUM_CELLS = 6ll << 20;
// Slots that every ranking workgroup counts for itself instead of summing up the histogram, which is then no launch.  With the histogram against
// without, us: 1100 tokens x 1 of 8 8.4 / 3.7, 2048 x 8 of 32 8.7 / 6.8, 8192 x 2 of 256 8.3 / 5.8, 16384 x 2 of 8 9.1 / 6.5, 4096 x 8 of 256
// 10.5 / 9.0, 8192 x 4 of 512 11.6 / 8.6; but 8192 x 8 of 256 10.8 / 11.9, of 60 9.2 / 11.2, 16384 x 8 of 256 12.6 / 18.0.
constexpr long long RANK_SELF_SLOTS = 32768;

// Slots, and slots x top-k (the comparisons of a wave of count_pack_kernel), up to which a step's count goes with its pack.  A step of rows of 2 KB with
// launches apart against together, us: 2048 x 1 of 8 41.7 / 40.1, 1024 x 2 of 8 43.9 / 42.4, 512 x 4 of 64 48.4 / 47.2, 128 x 8 of 256 52.4 / 51.2; but
// 2048 x 2 of 8 44.9 / 50.3, of 64 57.2 / 61.0, 4096 x 1 of 256 83.3 / 86.9, 1024 x 4 of 64 57.6 / 59.2, 256 x 8 of 256 58.0 / 59.0.
constexpr long long COUNT_PACK_SLOTS = 2048, COUNT_PACK_WORK = 8192;

extern "C" size_t moe_count_workspace_bytes(int T, int k, int E) {
    (void)k;
    const size_t NB = (size_t)ceil_div(T > 0 ? T : 1, CB);
    // hist[NB][E], base[NG + 1][E] (NG = ranking groups); the size callers were always asked for
    return sizeof(int32_t) * (2 * (size_t)E * NB + 2 * (size_t)E + 1);
}

static int check_count(const int32_t* topk_idx, int T, int k, int E, int W, const int32_t* send_counts, const int32_t* expert_offs,
                       const int32_t* dst_sizes, const int32_t* dst_offsets, const int32_t* caps, const int32_t* pos, const int32_t* row_token,
                       const void* ws, size_t ws_bytes) {
    MOE_REQUIRE(T >= 0 && E > 0 && W > 0, MOE_ERR_INVALID, "count: bad shape T=%d E=%d W=%d", T, E, W);
    MOE_REQUIRE(E % W == 0, MOE_ERR_INVALID, "num_experts_total must be divisible by world_size (E=%d W=%d)", E, W);
    MOE_REQUIRE(k >= 1 && k <= MOE_MAX_TOPK, MOE_ERR_UNSUPPORTED, "count: topk=%d outside [1,%d]", k, MOE_MAX_TOPK);
    MOE_REQUIRE(E <= MOE_MAX_EXPERTS, MOE_ERR_UNSUPPORTED, "count: E=%d > %d", E, MOE_MAX_EXPERTS);
    MOE_REQUIRE(send_counts && expert_offs && dst_sizes && dst_offsets && caps && ws, MOE_ERR_INVALID, "count: null pointer");
    MOE_REQUIRE(T == 0 || (topk_idx && pos && row_token), MOE_ERR_INVALID, "count: null pointer");
    MOE_REQUIRE(ws_bytes >= moe_count_workspace_bytes(T, k, E), MOE_ERR_WORKSPACE, "count: workspace %zu < %zu", ws_bytes,
                moe_count_workspace_bytes(T, k, E));
    return MOE_OK;
}

static int count_and_offsets(const int32_t* topk_idx, int T, int k, int E, int W, int32_t* send_counts, int32_t* expert_offs,
                             int32_t* dst_sizes, int32_t* dst_offsets, int32_t* caps, int32_t* pos, int32_t* row_token, void* ws,
                             size_t ws_bytes, const RecvPrepare* side, int side_blocks, hipStream_t s) {
    const int rc = check_count(topk_idx, T, k, E, W, send_counts, expert_offs, dst_sizes, dst_offsets, caps, pos, row_token, ws, ws_bytes);
    if (rc) return rc;
    const int NB = ceil_div(T > 0 ? T : 1, CB);
    int32_t* hist = (int32_t*)ws;
    auto lds = [&](int blocks) { return (size_t)blocks * E * sizeof(unsigned long long); };
#define MOE_RANK(ONE, SIDE, blocks, hist, base, more)                                                                                    \
    rank_kernel<ONE, SIDE><<<(blocks) + side_blocks, RANK_WAVES * WAVE, lds(rank_blocks<ONE>()) + (more), s>>>(                           \
        topk_idx, hist, base, T, k, E, W, NB, send_counts, expert_offs, dst_sizes, dst_offsets, caps, pos, row_token, blocks,           \
        side ? *side : RecvPrepare{})
    if (NB <= rank_blocks<true>()) {  // (few tokens: one workgroup holds everything)
        if (side) MOE_RANK(true, true, 1, nullptr, nullptr, 0);
        else MOE_RANK(true, false, 1, nullptr, nullptr, 0);
        return moe_check_launch("count_and_offsets");
    }
    const int NG = ceil_div(NB, rank_blocks<false>());
    if ((long long)T * k <= RANK_SELF_SLOTS) {
        const size_t tabs = 2 * RANK_COPIES * (size_t)(E | 1) * sizeof(int32_t);
        if (side) MOE_RANK(false, true, NG, nullptr, nullptr, tabs);
        else MOE_RANK(false, false, NG, nullptr, nullptr, tabs);
        return moe_check_launch("count_and_offsets");
    }
    block_hist_kernel<<<ceil_div(NB, 4), 256, 4 * E * sizeof(int32_t), s>>>(topk_idx, hist, T, k, E, NB);
    int32_t* base = nullptr;
    if ((long long)NG * NB * E > RANK_SUM_CELLS) {
        base = hist + (size_t)NB * E;
        scan_hist_kernel<<<ceil_div(E, SCAN_E), SCAN_E * SCAN_SLICES, 0, s>>>(hist, base, NB, NG, E);
    }
    if (side) MOE_RANK(false, true, NG, hist, base, 0);
    else MOE_RANK(false, false, NG, hist, base, 0);
#undef MOE_RANK
    return moe_check_launch("count_and_offsets");
}

extern "C" int moe_count_and_offsets(const int32_t* topk_idx, int T, int k, int E, int W, int32_t* send_counts,
                                     int32_t* expert_offs, int32_t* dst_sizes, int32_t* dst_offsets, int32_t* caps,
                                     int32_t* pos, int32_t* row_token, void* ws, size_t ws_bytes, moe_stream_t stream) {
    return count_and_offsets(topk_idx, T, k, E, W, send_counts, expert_offs, dst_sizes, dst_offsets, caps, pos, row_token, ws, ws_bytes, nullptr,
                             0, (hipStream_t)stream);
}

// ---- the same entry point for callers that may not allocate: the workspace is a fixed array in the library's own
// device image instead of a caller buffer.  Each GPU holds its own copy of the array at its own address; the address
// is looked up once per device, with that device current, and kept.
static __device__ __align__(256) unsigned char scratch[MOE_COUNT_SCRATCH_BYTES];

namespace {
constexpr int MAX_DEVICES = 64;
std::atomic<void*> g_scratch_ptr[MAX_DEVICES];

int count_scratch(void** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return moe_fail(MOE_ERR_LAUNCH, "count_and_offsets_static: hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= MAX_DEVICES) return moe_fail(MOE_ERR_UNSUPPORTED, "count_and_offsets_static: device %d", dev);
    void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!ptr) {
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return moe_fail(MOE_ERR_LAUNCH, "count_and_offsets_static: hipGetSymbolAddress: %s", hipGetErrorString(e));
        g_scratch_ptr[dev].store(ptr, std::memory_order_release);  // (racing first calls look up the same address)
    }
    *out = ptr;
    return MOE_OK;
}
}  // namespace

extern "C" size_t moe_count_static_scratch_bytes(void) { return MOE_COUNT_SCRATCH_BYTES; }

extern "C" int moe_count_and_offsets_static(const int32_t* topk_idx, int T, int k, int E, int W, int32_t* send_counts,
                                            int32_t* expert_offs, int32_t* dst_sizes, int32_t* dst_offsets, int32_t* caps,
                                            int32_t* pos, int32_t* row_token, moe_stream_t stream) {
    MOE_REQUIRE(T >= 0 && E > 0 && k >= 1, MOE_ERR_INVALID, "count_and_offsets_static: bad shape T=%d E=%d k=%d", T, E, k);
    const size_t need = moe_count_workspace_bytes(T, k, E);
    MOE_REQUIRE(need <= (size_t)MOE_COUNT_SCRATCH_BYTES, MOE_ERR_WORKSPACE,
                "count_and_offsets_static: T=%d tokens with E=%d experts need %zu bytes of scratch, the built-in array holds %zu "
                "(use moe_count_and_offsets with a workspace of your own)", T, E, need, (size_t)MOE_COUNT_SCRATCH_BYTES);
    void* ws = nullptr;
    const int rc = count_scratch(&ws);
    if (rc) return rc;
    // every cell of the workspace that the kernels read is written earlier in the same call (histogram cells by the
    // block that owns them, prefixes by the scan): nothing has to start at zero, stale contents of an earlier call
    // are never read
    return moe_count_and_offsets(topk_idx, T, k, E, W, send_counts, expert_offs, dst_sizes, dst_offsets, caps, pos, row_token, ws,
                                 (size_t)MOE_COUNT_SCRATCH_BYTES, stream);
}

extern "C" int moe_build_expert_offsets(const int32_t* counts, int W, int E_l, int32_t* expert_offs, int32_t* dst_sizes,
                                        int32_t* dst_offsets, moe_stream_t stream) {
    MOE_REQUIRE(W > 0 && E_l > 0 && W <= MOE_MAX_EXPERTS, MOE_ERR_INVALID, "build_expert_offsets: bad shape W=%d E_l=%d", W, E_l);
    MOE_REQUIRE(counts && expert_offs, MOE_ERR_INVALID, "build_expert_offsets: null pointer");
    expert_offsets_kernel<<<1, WAVE, 0, (hipStream_t)stream>>>(counts, W, E_l, expert_offs, dst_sizes, dst_offsets);
    return moe_check_launch("build_expert_offsets");
}

extern "C" int moe_max_floor1(const int32_t* values, int n, int32_t* out, moe_stream_t stream) {
    MOE_REQUIRE(n >= 0 && out && (n == 0 || values), MOE_ERR_INVALID, "max_floor1: bad arguments");
    max_floor1_kernel<<<1, 256, 0, (hipStream_t)stream>>>(values, n, out);
    return moe_check_launch("max_floor1");
}

static int check_pack_payload(const void* x, int dtype, int T, int H, const int32_t* row_token, int R, const void* payload) {
    const int rc = check_rows("pack_payload", dtype, H);
    if (rc) return rc;
    MOE_REQUIRE(R >= 0 && T >= 0, MOE_ERR_INVALID, "pack_payload: bad shape");
    MOE_REQUIRE(R == 0 || (x && row_token && payload), MOE_ERR_INVALID, "pack_payload: null pointer");
    return MOE_OK;
}

extern "C" int moe_pack_payload(const void* x, int dtype, int T, int H, const int32_t* row_token, int R, void* payload,
                                moe_stream_t stream) {
    const int rc = check_pack_payload(x, dtype, T, H, row_token, R, payload);
    if (rc) return rc;
    if (R == 0) return MOE_OK;
    RowSource a{};
    a.mode = SRC_MAP;
    a.map = row_token;
    return gather_rows(x, payload, a, R, H * dtype_size(dtype), (hipStream_t)stream);
}

extern "C" int moe_pack(const void* x, int dtype, int T, int H, const int32_t* row_token, const int32_t* dst_sizes,
                        const int32_t* dst_offsets, int W, int M, void* send_buf, int32_t* map_ws, int32_t* status,
                        moe_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    int rc = check_rows("pack", dtype, H);
    if (rc) return rc;
    MOE_REQUIRE(W > 0 && M >= 1 && T >= 0, MOE_ERR_INVALID, "pack: bad shape W=%d M=%d", W, M);
    MOE_REQUIRE((long long)W * M < (1ll << 31), MOE_ERR_UNSUPPORTED, "pack: W*M too large");
    MOE_REQUIRE(send_buf && dst_sizes && dst_offsets, MOE_ERR_INVALID, "pack: null pointer");
    (void)map_ws;
    RowSource a{};
    a.mode = SRC_PACK;
    a.map = row_token;
    a.dst_sizes = dst_sizes;
    a.dst_offsets = dst_offsets;
    a.M = M;
    a.status = status;
    return gather_rows(x, send_buf, a, W * M, H * dtype_size(dtype), s);
}

static int check_pack_tokens(const void* x, int dtype, int T, int H, const int32_t* topk_idx, const int32_t* pos, const float* gate, int k, int E_l,
                             const int32_t* dst_sizes, const int32_t* dst_offsets, int W, int M, const void* send_buf, const float* send_gate) {
    const int rc = check_rows("pack_tokens", dtype, H);
    MOE_REQUIRE((gate == nullptr) == (send_gate == nullptr), MOE_ERR_INVALID, "pack_tokens: gate and send_gate go together");
    if (rc) return rc;
    MOE_REQUIRE(W > 0 && M >= 1 && T >= 0 && E_l > 0, MOE_ERR_INVALID, "pack_tokens: bad shape W=%d M=%d E_l=%d", W, M, E_l);
    MOE_REQUIRE(k >= 1 && k <= MOE_MAX_TOPK, MOE_ERR_UNSUPPORTED, "pack_tokens: topk=%d outside [1,%d]", k, MOE_MAX_TOPK);
    MOE_REQUIRE((long long)W * M + T < (1ll << 31), MOE_ERR_UNSUPPORTED, "pack_tokens: W*M + T too large");
    MOE_REQUIRE(send_buf && dst_sizes && dst_offsets, MOE_ERR_INVALID, "pack_tokens: null pointer");
    MOE_REQUIRE(T == 0 || (x && topk_idx && pos), MOE_ERR_INVALID, "pack_tokens: null pointer");
    return MOE_OK;
}

extern "C" int moe_pack_tokens_gated(const void* x, int dtype, int T, int H, const int32_t* topk_idx, const int32_t* pos,
                                     const float* gate, int k, int E_l, const int32_t* dst_sizes, const int32_t* dst_offsets, int W,
                                     int M, void* send_buf, float* send_gate, int32_t* status, moe_stream_t stream) {
    const int rc = check_pack_tokens(x, dtype, T, H, topk_idx, pos, gate, k, E_l, dst_sizes, dst_offsets, W, M, send_buf, send_gate);
    if (rc) return rc;
    const int row_vec = H * dtype_size(dtype) / 16, parts = combine_parts(T, row_vec);
    const int n_units = T * parts + ceil_div(W * M, PACK_ZR);
    const int blocks = min(ceil_div(n_units, 4), 65535 * 8);
    with_topk(k, [&](auto kt) {
        pack_tokens_kernel<4, decltype(kt)::value><<<blocks, 4 * WAVE, 0, (hipStream_t)stream>>>(
            (const u32x4*)x, (u32x4*)send_buf, topk_idx, pos, dst_sizes, dst_offsets, T, k, E_l, W, M, H * dtype_size(dtype) / 16, status, gate, send_gate, parts);
    });
    return moe_check_launch("pack_tokens");
}

extern "C" int moe_pack_tokens(const void* x, int dtype, int T, int H, const int32_t* topk_idx, const int32_t* pos, int k,
                               int E_l, const int32_t* dst_sizes, const int32_t* dst_offsets, int W, int M, void* send_buf,
                               int32_t* status, moe_stream_t stream) {
    return moe_pack_tokens_gated(x, dtype, T, H, topk_idx, pos, nullptr, k, E_l, dst_sizes, dst_offsets, W, M, send_buf, nullptr,
                                 status, stream);
}

// f(16-byte vectors of a row of H bf16 values to a lane, 0: too many for the registers)
template <typename F>
static void with_row_vectors(int H, F&& f) {
    const int nv = ceil_div(H / 8, WAVE);
    if (nv <= 2) f(std::integral_constant<int, 2>{});
    else if (nv <= 4) f(std::integral_constant<int, 4>{});
    else if (nv <= 8) f(std::integral_constant<int, 8>{});
    else if (nv <= 16) f(std::integral_constant<int, 16>{});
    else f(std::integral_constant<int, 0>{});
}

static int check_pack_tokens_fp8(const void* x_bf16, int T, int H, const int32_t* topk_idx, const int32_t* pos, const float* gate, int k, int E_l,
                                 const int32_t* dst_sizes, const int32_t* dst_offsets, int W, int M, const void* send_q, const float* send_scale,
                                 const float* send_gate) {
    MOE_REQUIRE((gate == nullptr) == (send_gate == nullptr), MOE_ERR_INVALID, "pack_tokens_fp8: gate and send_gate go together");
    MOE_REQUIRE(T >= 0 && H > 0 && H % 8 == 0 && W > 0 && M >= 1 && E_l > 0, MOE_ERR_INVALID, "pack_tokens_fp8: bad shape");
    MOE_REQUIRE(k >= 1 && k <= MOE_MAX_TOPK, MOE_ERR_UNSUPPORTED, "pack_tokens_fp8: topk=%d outside [1,%d]", k, MOE_MAX_TOPK);
    MOE_REQUIRE((long long)W * M + T < (1ll << 31), MOE_ERR_UNSUPPORTED, "pack_tokens_fp8: W*M + T too large");
    MOE_REQUIRE(send_q && send_scale && dst_sizes && dst_offsets, MOE_ERR_INVALID, "pack_tokens_fp8: null pointer");
    MOE_REQUIRE(T == 0 || (x_bf16 && topk_idx && pos), MOE_ERR_INVALID, "pack_tokens_fp8: null pointer");
    return MOE_OK;
}

extern "C" int moe_pack_tokens_fp8(const void* x_bf16, int T, int H, const int32_t* topk_idx, const int32_t* pos, int k, int E_l,
                                   const int32_t* dst_sizes, const int32_t* dst_offsets, int W, int M, uint8_t* send_q,
                                   float* send_scale, int32_t* status, moe_stream_t stream) {
    return moe_pack_tokens_fp8_gated(x_bf16, T, H, topk_idx, pos, nullptr, k, E_l, dst_sizes, dst_offsets, W, M, send_q, send_scale,
                                     nullptr, status, stream);
}

extern "C" int moe_pack_tokens_fp8_gated(const void* x_bf16, int T, int H, const int32_t* topk_idx, const int32_t* pos,
                                         const float* gate, int k, int E_l, const int32_t* dst_sizes, const int32_t* dst_offsets,
                                         int W, int M, uint8_t* send_q, float* send_scale, float* send_gate, int32_t* status,
                                         moe_stream_t stream) {
    const int rc = check_pack_tokens_fp8(x_bf16, T, H, topk_idx, pos, gate, k, E_l, dst_sizes, dst_offsets, W, M, send_q, send_scale, send_gate);
    if (rc) return rc;
    const int n_units = T + ceil_div(W * M, PACK_ZR);
    const int blocks = min(ceil_div(n_units, 4), 65535 * 8);
    hipStream_t s = (hipStream_t)stream;
    with_topk(k, [&](auto kt) {
        with_row_vectors(H, [&](auto nv) {
            pack_tokens_fp8_kernel<decltype(kt)::value, decltype(nv)::value><<<blocks, 256, 0, s>>>(
                (const bf16_t*)x_bf16, T, H, topk_idx, pos, dst_sizes, dst_offsets, k, E_l, W, M, send_q, send_scale, status, gate, send_gate);
        });
    });
    return moe_check_launch("pack_tokens_fp8");
}

static int recv_driven(const char* who, int mode, const void* src, void* dst, int dtype, int H, const RecvCounts& q, int W, int E_l, int M,
                       int CAP, int n_out, int32_t* status, hipStream_t s) {
    int rc = check_rows(who, dtype, H);
    if (rc) return rc;
    MOE_REQUIRE(W > 0 && E_l > 0 && W * E_l <= MOE_MAX_EXPERTS, MOE_ERR_INVALID, "%s: bad W=%d E_l=%d", who, W, E_l);
    MOE_REQUIRE(n_out >= 0 && q.counts, MOE_ERR_INVALID, "%s: bad arguments", who);
    // (an empty flat payload or gradient has no storage: every output row is then padding and the source is never read)
    MOE_REQUIRE(n_out == 0 || (dst && (src || mode == SRC_REORDER || mode == SRC_UNSHUFFLE)), MOE_ERR_INVALID, "%s: null pointer", who);
    RowSource a{};
    a.mode = mode;
    a.W = W; a.E_l = E_l; a.M = M; a.CAP = CAP;
    a.status = status;
    // (one workgroup at least, for pca and the totals; at most what the chip holds at once, which then walks the rows)
    const int row_vec = H * dtype_size(dtype) / 16, rpw = copy_rows(mode, n_out, row_vec), blocks = max(1, min(ceil_div(n_out, 4 * rpw), 256 * 7));
#define MOE_GATHER(R) gather_rows_kernel<4, true, R><<<blocks, 4 * WAVE, 0, s>>>((const u32x4*)src, (u32x4*)dst, a, n_out, row_vec, q)
    if (rpw == 2) MOE_GATHER(2);
    else MOE_GATHER(1);
#undef MOE_GATHER
    return moe_check_launch(who);
}

extern "C" size_t moe_recv_map_ints(int W, int E_l, int n_out) {
    (void)n_out;  // (nothing needs it any more: tables and rows are resolved inside the copies; callers keep allocating what they did)
    return (size_t)3 * (W * E_l + 1) + (size_t)W * E_l;
}

extern "C" int moe_unpack_token_buf(const void* recv, int dtype, int W, int M, int H, const int32_t* recv_counts,
                                    int E_l, int CAP, void* token_buf, int32_t* pca, int32_t* map_ws, int32_t* status,
                                    moe_stream_t stream) {
    MOE_REQUIRE(M >= 1 && CAP >= 1, MOE_ERR_INVALID, "unpack_token_buf: M=%d CAP=%d", M, CAP);
    MOE_REQUIRE((long long)E_l * W * CAP < (1ll << 31), MOE_ERR_UNSUPPORTED, "unpack_token_buf: too many rows");
    (void)map_ws;
    return recv_driven("unpack_token_buf", SRC_TOKBUF, recv, token_buf, dtype, H, {recv_counts, E_l, 1, pca, nullptr}, W, E_l, M, CAP,
                       E_l * W * CAP, status, (hipStream_t)stream);
}

extern "C" int moe_reorder_flat_to_token_buf(const void* flat, int dtype, int R, int H, const int32_t* recv_counts,
                                             int W, int E_l, int CAP, void* token_buf, int32_t* map_ws, int32_t* status,
                                             moe_stream_t stream) {
    (void)R, (void)map_ws;
    MOE_REQUIRE(CAP >= 1, MOE_ERR_INVALID, "reorder: CAP=%d", CAP);
    MOE_REQUIRE((long long)E_l * W * CAP < (1ll << 31), MOE_ERR_UNSUPPORTED, "reorder: too many rows");
    return recv_driven("reorder_flat_to_token_buf", SRC_REORDER, flat, token_buf, dtype, H, {recv_counts, E_l, 1, nullptr, nullptr}, W, E_l, 1,
                       CAP, E_l * W * CAP, status, (hipStream_t)stream);
}

extern "C" int moe_unpack_expert_major(const void* recv, int dtype, int W, int M, int H, const int32_t* recv_counts,
                                       int E_l, void* shuffled, int S_rows, int32_t* expert_cnt, int32_t* map_ws,
                                       moe_stream_t stream) {
    (void)map_ws;
    MOE_REQUIRE(M >= 1, MOE_ERR_INVALID, "unpack_expert_major: M=%d", M);
    return recv_driven("unpack_expert_major", SRC_UNPACK, recv, shuffled, dtype, H, {recv_counts, E_l, 1, nullptr, expert_cnt}, W, E_l, M, 1,
                       S_rows, nullptr, (hipStream_t)stream);
}

// Rows of a [W,M] buffer that a wave looks through for padding: PACK_ZR, in small buffers no more than 16 KB (8 x 60 rows of 14 KB 6.7 -> 3.5 us).
static int padding_run(int rows, int row_bytes) { return rows >= 2048 * PACK_ZR ? PACK_ZR : max(1, min(16384 / row_bytes, PACK_ZR)); }
static RecvPrepare recv_prepare_args(const int32_t* rc, int W, int E_l, int M, int n_rows, int32_t* map, int32_t* expert_cnt,
                                     const float* recv_gate, float* row_gate, const float* recv_scale, float* row_scale, void* zbuf, int row_bytes,
                                     int threads, int& blocks) {
    // (at least one block, for the per-expert totals)
    const int map_blocks = max(ceil_div(n_rows, threads), 1);
    const int run = zbuf ? padding_run(W * M, row_bytes) : 1;
    blocks = map_blocks + (zbuf ? ceil_div(ceil_div(W * M, run), threads / WAVE) : 0);
    return {rc, W, E_l, M, n_rows, map, expert_cnt, recv_gate, row_gate, recv_scale, row_scale, (u32x4*)zbuf, row_bytes / 16, map_blocks, run};
}

static int launch_row_map(const int32_t* rc, int W, int E_l, int M, int n_rows, int32_t* map, int32_t* expert_cnt, const float* recv_gate,
                          float* row_gate, const float* recv_scale, float* row_scale, void* zbuf, int row_bytes, hipStream_t s) {
    int blocks;
    const RecvPrepare a = recv_prepare_args(rc, W, E_l, M, n_rows, map, expert_cnt, recv_gate, row_gate, recv_scale, row_scale, zbuf, row_bytes, 256, blocks);
    row_map_from_counts_kernel<<<blocks, 256, 0, s>>>(a);
    return moe_check_launch("recv_row_map");
}

static int check_recv_prepare(const int32_t* recv_counts, int W, int E_l, int M, int n_rows, const float* recv_gate, const float* recv_scale,
                              const int32_t* row_map, const float* row_gate, const float* row_scale, const void* ret, int dtype, int H) {
    MOE_REQUIRE(W > 0 && E_l > 0 && W * E_l <= MOE_MAX_EXPERTS, MOE_ERR_INVALID, "recv_prepare: bad W=%d E_l=%d", W, E_l);
    MOE_REQUIRE(M >= 0 && n_rows >= 0 && recv_counts, MOE_ERR_INVALID, "recv_prepare: bad arguments");
    MOE_REQUIRE((recv_gate == nullptr) == (row_gate == nullptr) && (recv_scale == nullptr) == (row_scale == nullptr), MOE_ERR_INVALID,
                "recv_prepare: received and row-ordered values go together");
    MOE_REQUIRE(n_rows == 0 || row_map, MOE_ERR_INVALID, "recv_prepare: null pointer");
    if (ret) {
        const int rc = check_rows("recv_prepare", dtype, H);
        if (rc) return rc;
        MOE_REQUIRE(M >= 1 && (long long)W * M < (1ll << 31), MOE_ERR_UNSUPPORTED, "recv_prepare: %d x %d rows", W, M);
    }
    return MOE_OK;
}

extern "C" int moe_recv_prepare(const int32_t* recv_counts, int W, int E_l, int M, int n_rows, const float* recv_gate, const float* recv_scale,
                                int32_t* row_map, float* row_gate, float* row_scale, int32_t* expert_cnt, void* ret, int dtype, int H,
                                moe_stream_t stream) {
    const int rc = check_recv_prepare(recv_counts, W, E_l, M, n_rows, recv_gate, recv_scale, row_map, row_gate, row_scale, ret, dtype, H);
    if (rc) return rc;
    return launch_row_map(recv_counts, W, E_l, M, n_rows, row_map, expert_cnt, recv_gate, row_gate, recv_scale, row_scale, ret,
                          H * dtype_size(dtype), (hipStream_t)stream);
}

// The receive side's preparation for a step, as blocks of `threads` beside another launch's
static int step_recv_prepare(const moe_step_args* a, int threads, RecvPrepare* side, int* blocks) {
    const int E_l = a->experts / a->world, M = a->flat ? 0 : a->M;
    const float *recv_gate = a->gated ? a->recv_gate : nullptr, *recv_scale = a->q_dispatch ? a->recv_scale : nullptr;
    float *row_gate = a->gated ? a->row_gate : nullptr, *row_scale = a->q_dispatch ? a->xs : nullptr;
    void* ret = a->flat ? nullptr : a->ret;
    const int rc = check_recv_prepare(a->recv_counts, a->world, E_l, M, a->S, recv_gate, recv_scale, a->row_map, row_gate, row_scale, ret, a->dtype,
                                      a->hidden);
    if (rc) return rc;
    *side = recv_prepare_args(a->recv_counts, a->world, E_l, M, a->S, a->row_map, a->expert_cnt, recv_gate, row_gate, recv_scale, row_scale, ret,
                              a->hidden * dtype_size(a->dtype), threads, *blocks);
    return MOE_OK;
}

int moe_count_and_prepare(const moe_step_args* a, hipStream_t s) {
    RecvPrepare side;
    int blocks;
    const int rc = step_recv_prepare(a, RANK_WAVES * WAVE, &side, &blocks);
    if (rc) return rc;
    return count_and_offsets(a->idx, a->tokens, a->topk, a->experts, a->world, a->send_counts, a->expert_offs, a->dst_sizes, a->dst_offsets, a->caps,
                             a->pos, a->row_token, a->count_ws, a->count_ws_bytes, &side, blocks, s);
}

bool moe_count_with_pack(int T, int k) { return T > 0 && k >= 1 && k <= MOE_MAX_TOPK && (long long)T * k <= COUNT_PACK_SLOTS && (long long)T * k * k <= COUNT_PACK_WORK; }

int moe_count_and_pack(const moe_step_args* a, bool prepare, hipStream_t s) {
    const int T = a->tokens, k = a->topk, E = a->experts, W = a->world, E_l = E / W, H = a->hidden, M = a->flat ? 0 : a->M;
    const float* gate = a->gated ? a->gate : nullptr;
    float* send_gate = a->gated ? a->send_gate : nullptr;
    RecvPrepare side{};
    int blocks = 0, rc = prepare ? step_recv_prepare(a, 256, &side, &blocks) : MOE_OK;
    if (!rc)
        rc = check_count(a->idx, T, k, E, W, a->send_counts, a->expert_offs, a->dst_sizes, a->dst_offsets, a->caps, a->pos, a->row_token, a->count_ws,
                         a->count_ws_bytes);
    if (!rc)
        rc = a->flat ? check_pack_payload(a->x, a->dtype, T, H, a->row_token, T * k, a->send)
             : a->q_dispatch
                 ? check_pack_tokens_fp8(a->x, T, H, a->idx, a->pos, gate, k, E_l, a->dst_sizes, a->dst_offsets, W, M, a->send, a->send_scale, send_gate)
                 : check_pack_tokens(a->x, a->dtype, T, H, a->idx, a->pos, gate, k, E_l, a->dst_sizes, a->dst_offsets, W, M, a->send, send_gate);
    if (rc) return rc;
    const CountOut out = {a->send_counts, a->expert_offs, a->dst_sizes, a->dst_offsets, a->caps, a->pos, a->row_token};
    auto launch = [&](auto kt, auto nv, int row_vec, int parts) {
        const int units = T * parts + ceil_div(W * M, PACK_ZR), grid = 1 + blocks + min(ceil_div(units, 4), 65535 * 8);
        count_pack_kernel<decltype(kt)::value, decltype(nv)::value><<<grid, 256, RANK_COPIES * (size_t)(E | 1) * sizeof(int32_t), s>>>(
            (const u32x4*)a->x, a->send, a->send_scale, a->idx, T, k, E, W, M, row_vec, out, a->status, gate, send_gate, parts, blocks, side);
    };
    with_topk(k, [&](auto kt) {
        const int row_vec = H * dtype_size(a->dtype) / 16;
        if (a->q_dispatch) with_row_vectors(H, [&](auto nv) { launch(kt, nv, H / 8, 1); });
        else launch(kt, std::integral_constant<int, -1>{}, row_vec, row_parts(T, row_vec));
    });
    return moe_check_launch("count_and_pack");
}

extern "C" int moe_recv_row_map(const int32_t* recv_counts, int W, int E_l, int M, int n_rows, int32_t* row_map,
                                int32_t* expert_cnt, int32_t* map_ws, moe_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    MOE_REQUIRE(W > 0 && E_l > 0 && W * E_l <= MOE_MAX_EXPERTS, MOE_ERR_INVALID, "recv_row_map: bad W=%d E_l=%d", W, E_l);
    MOE_REQUIRE(M >= 1 && n_rows >= 0 && recv_counts, MOE_ERR_INVALID, "recv_row_map: bad arguments");
    (void)map_ws;  // (the tables of earlier versions live in LDS now)
    MOE_REQUIRE(n_rows == 0 || row_map, MOE_ERR_INVALID, "recv_row_map: null pointer");
    // (one launch: every block rebuilds the prefix tables in LDS; at least one block, for the per-expert totals)
    return launch_row_map(recv_counts, W, E_l, M, n_rows, row_map, expert_cnt, nullptr, nullptr, nullptr, nullptr, nullptr, 0, s);
}

extern "C" int moe_recv_row_map_gated(const int32_t* recv_counts, int W, int E_l, int M, int n_rows, const float* recv_gate,
                                      int32_t* row_map, float* row_gate, int32_t* expert_cnt, moe_stream_t stream) {
    MOE_REQUIRE(W > 0 && E_l > 0 && W * E_l <= MOE_MAX_EXPERTS, MOE_ERR_INVALID, "recv_row_map_gated: bad W=%d E_l=%d", W, E_l);
    MOE_REQUIRE(M >= 0 && n_rows >= 0 && recv_counts, MOE_ERR_INVALID, "recv_row_map_gated: bad arguments");
    MOE_REQUIRE((recv_gate == nullptr) == (row_gate == nullptr), MOE_ERR_INVALID, "recv_row_map_gated: recv_gate and row_gate go together");
    MOE_REQUIRE(n_rows == 0 || row_map, MOE_ERR_INVALID, "recv_row_map_gated: null pointer");
    return launch_row_map(recv_counts, W, E_l, M, n_rows, row_map, expert_cnt, recv_gate, row_gate, nullptr, nullptr, nullptr, 0, (hipStream_t)stream);
}

extern "C" int moe_recv_row_map_flat(const int32_t* recv_counts, int W, int E_l, int n_rows, int32_t* row_map, int32_t* expert_cnt,
                                     moe_stream_t stream) {
    return moe_recv_row_map_gated(recv_counts, W, E_l, 0, n_rows, nullptr, row_map, nullptr, expert_cnt, stream);
}

// (E_l = 0: no row is one)
static int zero_padding(void* buf, int dtype, int W, int M, int H, const int32_t* recv_counts, int E_l, hipStream_t s) {
    const int run = padding_run(W * M, H * dtype_size(dtype));
    zero_padding_rows_kernel<<<ceil_div(ceil_div(W * M, run), 4), 256, 0, s>>>((u32x4*)buf, recv_counts, W, E_l, M, H * dtype_size(dtype) / 16, run);
    return moe_check_launch("zero_padding_rows");
}

extern "C" int moe_zero_padding_rows(void* buf, int dtype, int W, int M, int H, const int32_t* recv_counts, int E_l,
                                     moe_stream_t stream) {
    int rc = check_rows("zero_padding_rows", dtype, H);
    if (rc) return rc;
    MOE_REQUIRE(W > 0 && E_l > 0 && M >= 1 && buf && recv_counts, MOE_ERR_INVALID, "zero_padding_rows: bad arguments");
    MOE_REQUIRE((long long)W * M < (1ll << 31), MOE_ERR_UNSUPPORTED, "zero_padding_rows: too many rows");
    return zero_padding(buf, dtype, W, M, H, recv_counts, E_l, (hipStream_t)stream);
}

extern "C" int moe_shuffle(const void* token_buf, int dtype, int E_l, int W, int CAP, int H, const int32_t* pca,
                           void* shuffled, int S_rows, int32_t* expert_cnt, int32_t* map_ws, moe_stream_t stream) {
    (void)map_ws;
    hipStream_t s = (hipStream_t)stream;
    MOE_REQUIRE(W > 0 && E_l > 0 && W * E_l <= MOE_MAX_EXPERTS && CAP >= 1 && S_rows >= 0 && pca,
                MOE_ERR_INVALID, "shuffle: bad arguments");
    // (pca[e,s] = recv_counts[s,e])
    return recv_driven("shuffle", SRC_SHUFFLE, token_buf, shuffled, dtype, H, {pca, 1, W, nullptr, expert_cnt}, W, E_l, 1, CAP, S_rows,
                       nullptr, s);
}

// gradient of moe_shuffle: grad_token_buf[e,s,j,:] = grad_rows[off[e,s] + j,:] for j < pca[e,s], zeros elsewhere
extern "C" int moe_shuffle_backward(const void* grad_rows, int dtype, int E_l, int W, int CAP, int H, const int32_t* pca,
                                    void* grad_token_buf, int32_t* map_ws, moe_stream_t stream) {
    (void)map_ws;
    hipStream_t s = (hipStream_t)stream;
    MOE_REQUIRE(W > 0 && E_l > 0 && W * E_l <= MOE_MAX_EXPERTS && CAP >= 1 && pca, MOE_ERR_INVALID,
                "shuffle_backward: bad arguments");
    MOE_REQUIRE((long long)E_l * W * CAP < (1ll << 31), MOE_ERR_UNSUPPORTED, "shuffle_backward: too many rows");
    return recv_driven("shuffle_backward", SRC_UNSHUFFLE, grad_rows, grad_token_buf, dtype, H, {pca, 1, W, nullptr, nullptr}, W, E_l, 1, CAP,
                       E_l * W * CAP, nullptr, s);
}

extern "C" int moe_return_pack(const void* y, int dtype, int S_rows, int H, const int32_t* recv_counts, int W, int E_l,
                               int M, void* ret, int32_t* map_ws, moe_stream_t stream) {
    (void)map_ws;
    MOE_REQUIRE(M >= 1, MOE_ERR_INVALID, "return_pack: M=%d", M);
    MOE_REQUIRE((long long)W * M < (1ll << 31), MOE_ERR_UNSUPPORTED, "return_pack: W*M too large");
    if (S_rows == 0) {  // (a rank that received nothing: no result rows, which then have no storage either, and every slot is padding)
        const int rc = check_rows("return_pack", dtype, H);
        if (rc) return rc;
        MOE_REQUIRE(W > 0 && E_l > 0 && W * E_l <= MOE_MAX_EXPERTS && recv_counts && ret, MOE_ERR_INVALID, "return_pack: bad arguments");
        return zero_padding(ret, dtype, W, M, H, recv_counts, 0, (hipStream_t)stream);
    }
    return recv_driven("return_pack", SRC_RETURN, y, ret, dtype, H, {recv_counts, E_l, 1, nullptr, nullptr}, W, E_l, M, 1, W * M, nullptr,
                       (hipStream_t)stream);
}

extern "C" int moe_combine_backward(const void* d_out, const void* ret, int dtype, int W, int M, int H, const int32_t* topk_idx,
                                    const int32_t* pos, const float* gate, const int32_t* dst_sizes, const int32_t* dst_offsets,
                                    int T, int k, int E_l, void* d_ret, float* d_gate, moe_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    int rc = check_rows("combine_backward", dtype, H);
    if (rc) return rc;
    MOE_REQUIRE(W > 0 && M >= 1 && T >= 0 && E_l > 0, MOE_ERR_INVALID, "combine_backward: bad shape");
    MOE_REQUIRE(k >= 1 && k <= MOE_MAX_TOPK, MOE_ERR_UNSUPPORTED, "combine_backward: topk=%d outside [1,%d]", k, MOE_MAX_TOPK);
    MOE_REQUIRE((long long)W * M + T < (1ll << 31), MOE_ERR_UNSUPPORTED, "combine_backward: W*M + T too large");
    MOE_REQUIRE(d_ret && dst_offsets, MOE_ERR_INVALID, "combine_backward: null pointer");
    MOE_REQUIRE(T == 0 || (d_out && ret && topk_idx && pos && gate && d_gate), MOE_ERR_INVALID, "combine_backward: null pointer");
    const int row_vec = H * dtype_size(dtype) / 16;
    // (a token to a workgroup where its rows give every wave some 8 KB to move: 8192 tokens x 8 rows of 4 KB 138 -> 116 us, 4096 x 4 of
    // 8 KB 78 -> 66, 64 x 8 of 14 KB 48 -> 18; rows of 1 KB 22 -> 41, 4096 x 2 of 4 KB 24 -> 26)
    const bool wide = row_vec >= 512 || (row_vec >= 256 && k >= 4);
    const int blocks = min(ceil_div(T, wide ? 1 : 4) + ceil_div(ceil_div(W * M, PACK_ZR), 4), 65535 * 8);
#define MOE_CBW(XT, KT, WPT)                                                                                                           \
    combine_backward_kernel<XT, KT, 4, WPT><<<blocks, 4 * WAVE, 0, s>>>((const uint4*)d_out, (const uint4*)ret, topk_idx, pos, gate,     \
                                                                        dst_sizes, dst_offsets, T, k, E_l, W, M, row_vec, (uint4*)d_ret, \
                                                                        d_gate)
#define MOE_CB(XT, KT)             \
    if (wide) MOE_CBW(XT, KT, 4);  \
    else MOE_CBW(XT, KT, 1)
#define MOE_CBK(XT)                                    \
    switch (k) {                                       \
        case 1: MOE_CB(XT, 1); break;                  \
        case 2: MOE_CB(XT, 2); break;                  \
        case 4: MOE_CB(XT, 4); break;                  \
        case 8: MOE_CB(XT, 8); break;                  \
        default: MOE_CB(XT, 0); break;                 \
    }
    if (dtype == MOE_F32) MOE_CBK(float)
    else MOE_CBK(bf16_t)
#undef MOE_CBK
#undef MOE_CB
#undef MOE_CBW
    return moe_check_launch("combine_backward");
}

extern "C" int moe_combine(const void* ret, int dtype, int W, int M, int H, const int32_t* topk_idx, const int32_t* pos,
                           const float* gate, const int32_t* dst_offsets, int T, int k, int E_l, void* out,
                           int32_t* status, moe_stream_t stream) {
    hipStream_t s = (hipStream_t)stream;
    int rc = check_rows("combine", dtype, H);
    if (rc) return rc;
    MOE_REQUIRE(W > 0 && M >= 1 && T >= 0 && E_l > 0, MOE_ERR_INVALID, "combine: bad shape");
    MOE_REQUIRE(k >= 1 && k <= MOE_MAX_TOPK, MOE_ERR_UNSUPPORTED, "combine: topk=%d outside [1,%d]", k, MOE_MAX_TOPK);
    if (T == 0) return MOE_OK;
    MOE_REQUIRE(ret && topk_idx && pos && dst_offsets && out, MOE_ERR_INVALID, "combine: null pointer");  // (gate may be NULL)
    const int row_vec = H * dtype_size(dtype) / 16;
    if (dtype == MOE_F32) return launch_combine<float>(ret, topk_idx, pos, gate, dst_offsets, T, k, E_l, W, M, row_vec, out, status, s);
    return launch_combine<bf16_t>(ret, topk_idx, pos, gate, dst_offsets, T, k, E_l, W, M, row_vec, out, status, s);
}

// ---- the exchange of a simulated world -----------------------------------------------------------
static int a2a_check(const char* who, const moe_a2a_source* src, int W, int E_l) {
    MOE_REQUIRE(src && W > 0 && E_l > 0 && W * E_l <= MOE_MAX_EXPERTS, MOE_ERR_INVALID, "%s: bad W=%d E_l=%d", who, W, E_l);
    for (int s = 0; s < W; ++s)
        MOE_REQUIRE(!src[s].payload || (src[s].counts && src[s].start && src[s].rows >= 0 && aligned16(src[s].payload)), MOE_ERR_INVALID,
                    "%s: source %d is incomplete, or its payload not at a multiple of 16 bytes", who, s);
    return MOE_OK;
}
static A2aSources a2a_slice(const moe_a2a_source* src, int s0, int ns) {
    A2aSources q{};
    for (int i = 0; i < ns; ++i) q.src[i] = src[s0 + i];
    return q;
}

extern "C" int moe_a2a_max_count(const moe_a2a_source* sources, int W, int E_l, int32_t* max_count, moe_stream_t stream) {
    const int rc = a2a_check("a2a_max_count", sources, W, E_l);
    if (rc) return rc;
    MOE_REQUIRE(max_count, MOE_ERR_INVALID, "a2a_max_count: null pointer");
    for (int s0 = 0; s0 < W; s0 += A2A_SRC) {
        const int ns = min(A2A_SRC, W - s0);
        a2a_max_count_kernel<<<1, 256, 0, (hipStream_t)stream>>>(a2a_slice(sources, s0, ns), ns, E_l, max_count, s0 == 0, s0 + ns == W);
    }
    return moe_check_launch("a2a_max_count");
}

// Rows of the exchange that a wave takes together: two of up to 3 KB (few rows: 4 KB), from where they keep the chip busy to
// where the waves of single rows do, and four of very many short ones.
// One by one / together, us (n rows copied, 1.1 to 1.2 n slots): 8192 rows of 1.5 KB 9.2 / 8.4, 2 KB 10.9 / 9.9; 16384 of 1 KB 11.7 / 11.0, 1.5 KB
// 16.2 / 14.3; 32768 of 512 bytes 14.5 / 14.4, 1.5 KB 23.1 / 19.9, 2.3 KB 27.7 / 26.3; 4096 of 3 KB 9.4 / 7.9; but of 2.3 KB 6.6 / 7.1, 6000 of 2 KB 7.0 / 7.6, 8192 of 1 KB
// 6.5 / 7.0, of 256 bytes 5.5 / 6.1, 32768 of 256 bytes 10.7 / 12.2, 65536 of 3 KB 60 / 64, 24576 of 3.5 KB 31.5 / 34.7.  Four together cost 0 to 10 % more
// than two, but 65536 of 512 bytes 25.7 / 23.6 / 22.4 (two, four), of 1 KB 29.3 / 27.0 / 25.5, of 1.5 KB 38.6 / 36.3 / 38.2.
static int place_rows(int n, int row_vec) {
    const long long vecs = (long long)n * row_vec;
    if (row_vec > 2 * WAVE) return n >= (row_vec <= 160 ? 6144 : 4096) && ((row_vec <= 3 * WAVE && vecs <= 8ll << 20) || (row_vec <= 4 * WAVE && n <= 6144)) ? 2 : 1;
    if (n >= 49152 && row_vec <= 80) return 4;
    return n >= 8192 && vecs >= (row_vec >= 48 ? 3ll : 4ll) << 18 && vecs <= 8ll << 20 ? 2 : 1;
}

extern "C" int moe_a2a_place(const moe_a2a_source* sources, int dtype, int W, int E_l, int CAP, int H, void* token_buf, int32_t* pca,
                             int32_t* counts_ready, int n_ready, int32_t* token_sync, int n_sync, moe_stream_t stream) {
    int rc = a2a_check("a2a_place", sources, W, E_l);
    if (!rc) rc = check_rows("a2a_place", dtype, H);
    if (rc) return rc;
    MOE_REQUIRE(CAP >= 1 && (long long)E_l * W * CAP < (1ll << 31), MOE_ERR_UNSUPPORTED, "a2a_place: CAP=%d", CAP);
    MOE_REQUIRE(token_buf && pca, MOE_ERR_INVALID, "a2a_place: null pointer");
    for (int s0 = 0; s0 < W; s0 += A2A_SRC) {
        const int ns = min(A2A_SRC, W - s0);
        const int row_vec = H * dtype_size(dtype) / 16, n = E_l * ns * CAP, rpw = place_rows(n, row_vec);
        const int blocks = min(ceil_div(n, 4 * rpw), 256 * 8);
#define MOE_PLACE(R)                                                                                                                      \
    a2a_place_kernel<R><<<blocks, 256, 0, (hipStream_t)stream>>>(a2a_slice(sources, s0, ns), s0, ns, W, E_l, CAP, row_vec, (u32x4*)token_buf, \
                                                                 pca, counts_ready, counts_ready && !s0 ? n_ready : 0, token_sync,        \
                                                                 token_sync && !s0 ? n_sync : 0)
        if (rpw == 4) MOE_PLACE(4);
        else if (rpw == 2) MOE_PLACE(2);
        else MOE_PLACE(1);
#undef MOE_PLACE
    }
    return moe_check_launch("a2a_place");
}

extern "C" int moe_shuffle_totals(const int32_t* pca, int n, const int32_t* token_sync, int n_sync, int32_t* out, moe_stream_t stream) {
    MOE_REQUIRE(n >= 0 && n_sync >= 0 && out && (n == 0 || pca) && (n_sync == 0 || token_sync), MOE_ERR_INVALID, "shuffle_totals: bad arguments");
    shuffle_totals_kernel<<<1, 256, 0, (hipStream_t)stream>>>(pca, n, token_sync, n_sync, out);
    return moe_check_launch("shuffle_totals");
}
