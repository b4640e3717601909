// One step of the hot path as one call: host code only, every stage is an entry point of its own.
#include "common.h"

struct Range {
    const void* at;
    size_t bytes;
};
static bool meet(const Range& r, const Range& q) {
    return r.at && q.at && (uintptr_t)r.at < (uintptr_t)q.at + q.bytes && (uintptr_t)q.at < (uintptr_t)r.at + r.bytes;
}

// True if nothing that the receive side's preparation reads or writes lies in a buffer of the source side up to the pack: a caller that
// loops its own rows back (received counts, gates or scales are the sent ones) or shares scratch between the sides needs them in order.
static bool sides_apart(const moe_step_args* a) {
    const size_t T = a->tokens, H = a->hidden, E = a->experts, W = a->world, R = T * a->topk, S = a->S, n = W * (size_t)a->M;
    const size_t row = H * (a->dtype == MOE_BF16 ? 2 : 4);
    const Range receive[] = {{a->recv_counts, E * 4}, {a->gated ? a->recv_gate : nullptr, n * 4}, {a->q_dispatch ? a->recv_scale : nullptr, n * 4},
                             {a->row_map, S * 4}, {a->expert_cnt, E / W * 4}, {a->gated ? a->row_gate : nullptr, S * 4},
                             {a->q_dispatch ? a->xs : nullptr, S * 4}, {a->flat ? nullptr : a->ret, n * row}};
    const Range source[] = {{a->x, T * row}, {a->idx, R * 4}, {a->gate, R * 4}, {a->send_counts, E * 4}, {a->expert_offs, E * 4},
                            {a->dst_sizes, W * 4}, {a->dst_offsets, W * 4}, {a->caps, 8}, {a->pos, R * 4}, {a->row_token, R * 4},
                            {a->count_ws, a->count_ws_bytes}, {a->send, a->flat ? R * row : a->q_dispatch ? n * H : n * row},
                            {a->send_scale, n * 4}, {a->send_gate, n * 4}, {a->status, 4}};
    for (const Range& r : receive)
        for (const Range& q : source)
            if (meet(r, q)) return false;
    return true;
}

// True if a launch writes nothing that it reads, and nothing twice.
template <int NR, int NW>
static bool own_writes(const Range (&reads)[NR], const Range (&writes)[NW]) {
    for (int i = 0; i < NW; ++i) {
        for (const Range& r : reads)
            if (meet(r, writes[i])) return false;
        for (int j = 0; j < i; ++j)
            if (meet(writes[j], writes[i])) return false;
    }
    return true;
}

// True if the GEMMs of fp32 experts may move the rows themselves.  One launch then unpacks and runs the up projection, the next runs the
// down projection and fills the returned buffer: scratch that takes the place of something the other half of such a launch still reads
// (the hidden activation over the received rows; the returned rows over the hidden activation, or over the counts per expert, by which
// every workgroup finds its tile) needs the copies, which stand before and behind the GEMMs.
static bool f32_apart(const moe_step_args* a) {
    const size_t H = a->hidden, F = a->ffn, S = a->S, E_l = a->experts / a->world, slots = (size_t)a->world * a->M * H * 4, w = E_l * H * F * 4;
    const Range recv = {a->recv, slots}, ret = {a->ret, slots}, hidden = {a->hidden_ws, S * F * 4}, rows = {a->rows, S * H * 4}, y = {a->y, S * H * 4};
    const Range sent = {a->recv_counts, (size_t)a->experts * 4}, counts = {a->expert_cnt, E_l * 4}, w1 = {a->w1, w}, w2 = {a->w2, w};
    const Range up = {a->act == MOE_ACT_SWIGLU ? a->w_up : nullptr, w};
    return own_writes({recv, sent, w1, up}, {rows, counts, hidden}) && own_writes({hidden, counts, sent, w2}, {y, ret});
}

// True if the count may share a launch with the pack, which then does not read what the count leaves: nothing that the two write is read by
// either or written twice.
static bool count_pack_apart(const moe_step_args* a) {
    const size_t T = a->tokens, H = a->hidden, E = a->experts, W = a->world, R = T * a->topk, n = W * (size_t)a->M, row = H * (a->dtype == MOE_BF16 ? 2 : 4);
    const size_t sent = a->flat ? R * row : n * (a->q_dispatch ? H : row);
    return own_writes({{a->x, T * row}, {a->idx, R * 4}, {a->gated ? a->gate : nullptr, R * 4}},
                      {{a->send_counts, E * 4}, {a->expert_offs, E * 4}, {a->dst_sizes, W * 4}, {a->dst_offsets, W * 4}, {a->caps, 8}, {a->pos, R * 4},
                       {a->row_token, R * 4}, {a->send, sent}, {a->q_dispatch ? a->send_scale : nullptr, n * 4}, {a->gated ? a->send_gate : nullptr, n * 4},
                       {a->status, 4}});
}

// How a step goes: the receive side prepared in the launch that ranks the tokens; the rows of fp32 experts moved by their GEMMs (plumbing:
// 42.9 -> 38 us a step); the tokens ranked by the pack.
struct StepPlan {
    bool together, f32_slots, count_pack;
};
static int step_plan(const moe_step_args* a, StepPlan* plan) {
    MOE_REQUIRE(a, MOE_ERR_INVALID, "step: null arguments");
    MOE_REQUIRE(a->world > 0 && a->experts > 0 && a->experts % a->world == 0, MOE_ERR_INVALID, "step: %d experts on %d ranks", a->experts, a->world);
    MOE_REQUIRE(a->fused || !(a->flat || a->gated || a->q_dispatch), MOE_ERR_INVALID, "step: flat / gated / q_dispatch are fused modes");
    MOE_REQUIRE(!a->q_dispatch || (a->quant && !a->flat), MOE_ERR_INVALID, "step: q_dispatch needs fp8 experts and fixed slots");
    MOE_REQUIRE(!(a->flat && a->gated), MOE_ERR_INVALID, "step: flat and gated are separate modes");
    plan->together = a->fused && sides_apart(a);
    plan->f32_slots = a->f32_weights && !a->fused && !a->quant && a->dtype == MOE_F32 && a->S > 0 && f32_apart(a);
    plan->count_pack = moe_count_with_pack(a->tokens, a->topk) && count_pack_apart(a);
    return MOE_OK;
}

extern "C" int moe_step_plan(const moe_step_args* a, int32_t* out) {
    MOE_REQUIRE(out, MOE_ERR_INVALID, "step_plan: null result");
    StepPlan plan;
    const int rc = step_plan(a, &plan);
    if (rc != MOE_OK) return rc;
    out[0] = plan.together;
    out[1] = plan.f32_slots;
    return MOE_OK;
}

// Stage by stage from Python a step costs 8 to 10 foreign calls with some fifteen arguments each (about 80 us of host time);
// here one, so an eager step of a small model waits for the GPU and not for the host.  The destination side derives the row map, the
// row scales, the gates and the zeroed padding rows from the received counts in one launch, the one that ranks the tokens (a launch
// costs some 4.5 us even when it has nothing to do).
extern "C" int moe_step(const moe_step_args* a, moe_stream_t stream) {
    StepPlan plan;
    int rc = step_plan(a, &plan);
    if (rc != MOE_OK) return rc;
    const int T = a->tokens, H = a->hidden, E = a->experts, k = a->topk, W = a->world, F = a->ffn, M = a->M, S = a->S;
    const int E_l = E / W;
    const float* out_gate = a->gated ? a->gate : nullptr;
#define MOE_STAGE(call)                           \
    do {                                          \
        if ((rc = (call)) != MOE_OK) return rc;   \
    } while (0)
    MOE_STAGE(moe_route_topk(a->x, a->router, a->bias, a->dtype, T, H, E, k, a->logits, a->idx, a->gate, a->route_ws, a->route_ws_bytes,
                             stream));
    if (plan.count_pack)
        MOE_STAGE(moe_count_and_pack(a, plan.together, (hipStream_t)stream));
    else if (plan.together)
        MOE_STAGE(moe_count_and_prepare(a, (hipStream_t)stream));
    else
        MOE_STAGE(moe_count_and_offsets(a->idx, T, k, E, W, a->send_counts, a->expert_offs, a->dst_sizes, a->dst_offsets, a->caps, a->pos,
                                        a->row_token, a->count_ws, a->count_ws_bytes, stream));
    if (plan.count_pack) {
    } else if (a->q_dispatch)
        MOE_STAGE(moe_pack_tokens_fp8_gated(a->x, T, H, a->idx, a->pos, out_gate, k, E_l, a->dst_sizes, a->dst_offsets, W, M,
                                            (uint8_t*)a->send, a->send_scale, a->gated ? a->send_gate : nullptr, a->status, stream));
    else if (a->flat)
        MOE_STAGE(moe_pack_payload(a->x, a->dtype, T, H, a->row_token, T * k, a->send, stream));
    else if (a->gated)
        MOE_STAGE(moe_pack_tokens_gated(a->x, a->dtype, T, H, a->idx, a->pos, a->gate, k, E_l, a->dst_sizes, a->dst_offsets, W, M, a->send,
                                        a->send_gate, a->status, stream));
    else
        MOE_STAGE(moe_pack_tokens(a->x, a->dtype, T, H, a->idx, a->pos, k, E_l, a->dst_sizes, a->dst_offsets, W, M, a->send, a->status,
                                  stream));
    // destination: rows in expert-major order
    if (a->fused && !plan.together)
        MOE_STAGE(moe_recv_prepare(a->recv_counts, W, E_l, a->flat ? 0 : M, S, a->gated ? a->recv_gate : nullptr,
                                   a->q_dispatch ? a->recv_scale : nullptr, a->row_map, a->gated ? a->row_gate : nullptr,
                                   a->q_dispatch ? a->xs : nullptr, a->expert_cnt, a->flat ? nullptr : a->ret, a->dtype, H, stream));
    else if (!a->fused && !plan.f32_slots)
        MOE_STAGE(moe_unpack_expert_major(a->recv, a->dtype, W, M, H, a->recv_counts, E_l, a->rows, S, a->expert_cnt, a->unpack_map, stream));
    const void* src = a->fused ? a->recv : a->rows;
    void* dst = a->fused ? a->ret : a->y;
    const int n_buf = a->fused && !a->flat ? W * M : S;
    const int32_t* map = a->fused ? a->row_map : nullptr;
    const float* row_gate = a->gated ? a->row_gate : nullptr;
    if (a->q_dispatch)
        MOE_STAGE(moe_grouped_mlp_fp8_q_mapped((const uint8_t*)src, nullptr, n_buf, map, a->expert_cnt, S, H, F, E_l, (const uint8_t*)a->w1,
                                               a->s1, a->s_up, (const uint8_t*)a->w2, a->s2, a->xs, a->hq, a->hscale, row_gate, dst, n_buf,
                                               map, a->part_ws, a->part_ws_bytes, stream));
    else if (a->quant)
        MOE_STAGE(moe_grouped_mlp_fp8_mapped(src, n_buf, map, a->expert_cnt, S, H, F, E_l, (const uint8_t*)a->w1, a->s1, a->s_up,
                                             (const uint8_t*)a->w2, a->s2, a->xq, a->xs, a->hq, a->hscale, row_gate, dst, n_buf, map,
                                             a->part_ws, a->part_ws_bytes, stream));
    else if (plan.f32_slots)
        MOE_STAGE(moe_mlp_f32_slots((const float*)a->recv, a->recv_counts, W, M, S, H, F, E_l, a->act, (const float*)a->w1,
                                    (const float*)a->w_up, (const float*)a->w2, (float*)a->rows, a->expert_cnt, (float*)a->hidden_ws,
                                    (float*)a->y, (float*)a->ret, (hipStream_t)stream));
    else if (a->f32_weights)
        MOE_STAGE(moe_grouped_mlp(src, a->expert_cnt, a->dtype, S, H, F, E_l, a->act, a->w1, a->w_up, a->w2, a->hidden_ws, dst, stream));
    else {
        MOE_STAGE(moe_grouped_gemm_mapped(src, n_buf, map, a->w1, a->expert_cnt, S, H, F, E_l, a->act, a->hidden_ws, S, nullptr, a->part_ws,
                                          a->part_ws_bytes, stream));
        if (a->gated)
            MOE_STAGE(moe_grouped_gemm_mapped_gated(a->hidden_ws, S, nullptr, a->w2, a->expert_cnt, S, F, H, E_l, row_gate, dst, n_buf, map,
                                                    a->part_ws, a->part_ws_bytes, stream));
        else
            MOE_STAGE(moe_grouped_gemm_mapped(a->hidden_ws, S, nullptr, a->w2, a->expert_cnt, S, F, H, E_l, MOE_ACT_NONE, dst, n_buf, map,
                                              a->part_ws, a->part_ws_bytes, stream));
    }
    if (!a->fused && !plan.f32_slots) MOE_STAGE(moe_return_pack(a->y, a->dtype, S, H, a->recv_counts, W, E_l, M, a->ret, a->ret_map, stream));
    // the flat returned payload is indexed by position: one "destination" that holds all experts, offset 0
    if (a->flat)
        return moe_combine(a->returned, a->dtype, 1, T * k, H, a->idx, a->pos, a->gate, a->zero_off, T, k, E, a->out, a->status, stream);
    return moe_combine(a->returned, a->dtype, W, M, H, a->idx, a->pos, a->gated ? nullptr : a->gate, a->dst_offsets, T, k, E_l, a->out,
                       a->status, stream);
#undef MOE_STAGE
}
