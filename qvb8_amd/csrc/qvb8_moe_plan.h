// Routing plan of the expert stack, shared by the kernels that group the (token, choice) pairs by expert.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qvb8 {

// Pairs of one expert that the many-token kernels multiply together (qvb8_moe_group.hip): a slot with more pairs is worked
// on in several blocks.
constexpr int kGroupTokens = 64;

// Workspace layout (bytes from the start): plan | H | Yd
//   plan: i32 n_bad, i32 slots in use, i32 token blocks of all slots (+1 pad), int4 slot[n_slots] = {expert, first pair, end pair, token blocks of
//   the slots before it} for the experts that have pairs (end == first for unused slots), i32 order[npairs] (pair numbers
//   grouped by expert)
struct MoePlan {
    int32_t* n_bad; int4* slot; int32_t* order;
};
__host__ __device__ inline int64_t moe_slots(int64_t E, int64_t npairs) { return E < npairs ? E : npairs; }
__host__ __device__ inline size_t moe_plan_bytes(int64_t E, int64_t npairs) {
    return (size_t)(16 + moe_slots(E, npairs) * 16 + npairs * 4 + 255) & ~(size_t)255;
}
__host__ __device__ inline MoePlan moe_plan_at(void* ws, int64_t E, int64_t npairs) {
    unsigned char* p = reinterpret_cast<unsigned char*>(ws);
    return MoePlan{reinterpret_cast<int32_t*>(p), reinterpret_cast<int4*>(p + 16),
                   reinterpret_cast<int32_t*>(p + 16 + moe_slots(E, npairs) * 16)};
}

// One projection of the expert stack for many tokens (qvb8_moe_group.hip).
struct MoeGroupArgs {
    const void* X;                 // up: (tokens, P) activations; down: H (pairs, P) f32
    MoePlan plan;
    const uint8_t* ids; int64_t ids_bytes;
    const float* min_s; const float* tau_s; const uint8_t* nbits; const int64_t* bit_off;   // (E, Q)
    float* out;                    // up: H (pairs, units); down: Yd (pairs, Q)
    int E, Q, P, topk;
    int units, gated;              // up: outputs per expert; whether the rows come as (gate, up) halves
    int keep_inf;                  // up: an infinity among fp16 activations stays one
    int planes;                    // every 16-row tile is stored in planes (a regular stack; bit_off marked)
    int row_blocks, items;         // set by the launcher
};
bool moe_group_shapes_ok(int64_t P_up, int64_t Q_dn, int64_t P_dn);
int launch_moe_group(bool down, int x_dtype, MoeGroupArgs a, int64_t npairs, hipStream_t s);

}  // namespace qvb8
