// What the layer call hands to the expert kernels beyond the public entry points.
#pragma once
#include "common.h"

namespace moe {

constexpr int kTailTokens = 16;          // tokens up to which the down projection may combine (the thin kernel's rows)

// The combine of a layer call, for a down projection that can end with it
struct CombineTail {
    const int32_t *pos, *topk_idx;       // [n, k]
    const float* topk_w;
    const uint16_t* residual;            // may be NULL
    uint16_t* out;                       // [n, hidden]
    int32_t* arrivals;                   // [ceil(hidden / 16)], set by the dispatch (DispatchOut)
    int n, k, mode;
};
constexpr int tail_arrivals(int hidden) { return (hidden + 15) / 16; }

// Whether a down projection of n_rows rows (and of a shared expert) in layer_experts may combine: no call for which this is false does
bool layer_may_combine(int32_t n_experts, int32_t n_rows, bool shared, int32_t hidden);

// moe_grouped_swiglu_joint, both phases (shared may be NULL); combined: the down projection has also done what `tail` says
int layer_experts(const moe_mlp_group& routed, const moe_mlp_group* shared, int32_t hidden, int32_t fp8, const CombineTail* tail,
                  bool* combined, void* stream);

}  // namespace moe
