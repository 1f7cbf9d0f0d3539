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

// The shared expert's gate and up projection of a few tokens, which needs nothing of the router: its waves run in the router's
// launch, which leaves most of the chip and all of the memory's rate idle (layer_shared_first).  Layers, us, in the routed experts' launch
// -> here: DeepSeek-V2-Lite 1 / 3 / 8 / 16 tokens 49.3 / 64.2 / 79.9 / 92.3 -> 48.1 / 62.8 / 77.2 / 91.8, DeepSeek-V2-236B 2 / 8 / 16 139.4 /
// 245.8 / 338.5 -> 131.7 / 241.5 / 330.0, DeepSeek-V3 1 / 5 / 14 123.0 / 328.6 / 655.1 -> 121.7 / 327.9 / 652.3.
struct SharedFirst {
    const void *const *w_gate, *const *w_up;
    const float *const *s_gate, *const *s_up;
    const uint16_t* x;
    uint16_t* act;
    int rows, hidden, inter, fp8;
    int first_block;                     // of the launch
};
constexpr int shared_first_blocks(int inter) { return (inter + 15) / 16; }

// Whether it may run there: the thin kernel then serves the call, whose gate and up launch leaves it out.
//  * One workgroup per CU is the line, those of the router that find no tokens counted: a workgroup is one wave that streams, in an LDS of
//    70 KiB, and past it a CU has a second one to wait for, where the thin kernel runs six.  Layers, us, in the routed experts' launch ->
//    here, 1 and 8 tokens: 64 fp8 experts (16 workgroups in front), shared 3840 wide 89 / 122 -> 90 / 112, 3968 90 / 114 -> 114 / 129, 16384
//    204 / 394 -> 219 / 419; 256 (64), 3072 90 / 138 -> 91 / 136, 3584 92 / 140 -> 116 / 160; DeepSeek-V2-236B's router (40) and bf16,
//    3072 73 / 97 -> 70 / 86, 3584 74 / 98 -> 86 / 100.
//  * And the router has to take long enough: its chain grows with the hidden size, a shared wave of few stages is mostly its own start.
//    Graph replays of 9 layers of 1 to 16 tokens each, ratio: bf16, hidden size 512 1.037, 1024 1.016, 1536 0.992, 2048 0.983, 4096 and more
//    0.97; fp8 512 1.049, 2048 1.027, 4096 1.015, 5120 1.000, 7168 0.992.
bool layer_shared_first(const moe_mlp_group& routed, const moe_mlp_group& shared, int32_t hidden);

// moe_grouped_swiglu_joint, both phases (shared may be NULL), as a part of a layer call
struct LayerCall {
    const CombineTail* tail = nullptr;   // the combine, for a down projection that can end with it
    bool combined = false;               // (result) it did
    bool shared_gate_up_done = false;
    int32_t* claims = nullptr;           // counters that the dispatch sets to 0, kClaimInts for each launch of the call; NULL: none
};
// Whether a launch of the call can have use for them: one with both kinds of tiles.  shared: NULL, or a shared expert with launches of its own
bool layer_claims(const moe_mlp_group& routed, const moe_mlp_group* shared, int32_t hidden);
bool layer_joins(const moe_mlp_group& routed, const moe_mlp_group& shared, int32_t hidden);      // moe_shared_joins
constexpr int kClaimStride = 32, kClaimInts = 8 * kClaimStride;      // a line per XCD
constexpr int kLayerClaims = 4 * kClaimInts;                         // two projections, the shared expert's apart
int layer_experts(const moe_mlp_group& routed, const moe_mlp_group* shared, int32_t hidden, int32_t fp8, LayerCall* call, void* stream);

}  // namespace moe
