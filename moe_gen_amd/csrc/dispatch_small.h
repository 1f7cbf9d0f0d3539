// Token-to-expert dispatch of a short index list by ONE workgroup of 16 waves (a decode or small prefill batch: three
// dependent launches of a few microseconds each cost more than their work).  Shared by dispatch_small and by the
// selection kernel for few tokens, which runs it on the indices it has just chosen.
#pragma once
#include "common.h"
#include "layer.h"

namespace moe {

constexpr int kDispatchMaxE = 256;
constexpr int SMALL_WAVES = 16;

struct DispatchOut {
    int32_t *counts, *offsets, *perm, *pos;
    int32_t* row_map;        // perm / k, may be NULL
    int32_t* one_group;      // [2]: {0, tokens}, the row range of a group that holds every token (the shared expert); may be NULL
    // [n_arrivals]: set to minus the experts that have rows and the one of one_group (CombineTail; one workgroup's form only)
    int32_t* arrivals = nullptr;
    int n_arrivals = 0;
    int32_t* claims = nullptr;   // [n_claims]: set to 0 (LayerCall)
    int n_claims = 0;
};

// (NW waves.)  Wave w owns the w-th slice of the list (a multiple of 64 entries, at most IT of them): counts it, the first 256 threads
// turn the 16 x E counts into counts[], offsets[] and one cursor per (wave, expert) -- offsets[e] + entries of e in
// earlier slices -- and every wave ranks its slice 64 entries at a time.  The sorted position of an entry is the same
// pure function of the list as in the three-kernel form.  get(i): entry i of the list, i < nk.
template <int IT, int NW = SMALL_WAVES, typename F>
__device__ __forceinline__ void dispatch_one_workgroup(int nk, int E, const DispatchOut& out, int k, F get) {
    static_assert(64 * NW >= kDispatchMaxE, "a thread per expert");
    __shared__ int whist[NW][kDispatchMaxE];
    __shared__ int wtot[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int slice = (nk + NW * 64 - 1) / (NW * 64) * 64;
    const int wbase = wave * slice;
    // the lane's entries of the slice, all requested at once (both passes use them: a load per step would put the
    // memory latency into every step); -1 marks an entry past the list or an id outside [0, E)
    int ev[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) ev[it] = get(min(wbase + 64 * it + lane, nk - 1));
    for (int e = tid; e < NW * kDispatchMaxE; e += 64 * NW) (&whist[0][0])[e] = 0;
    __syncthreads();
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int g = wbase + 64 * it + lane;
        if (64 * it >= slice || g >= nk || (unsigned)ev[it] >= (unsigned)E) ev[it] = -1;
        if (ev[it] >= 0) atomicAdd(&whist[wave][ev[it]], 1);
    }
    __syncthreads();
    int cv = 0, inc = 0;
    if (tid < kDispatchMaxE) {                 // waves 0 .. 3, whole waves
        if (tid < E) {
#pragma unroll
            for (int w = 0; w < NW; ++w) cv += whist[w][tid];
        }
        inc = cv;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(inc, d);
            if (lane >= d) inc += o;
        }
        if (lane == 63) wtot[wave] = inc;
    }
    __syncthreads();
    if (tid < E) {
        int run = inc - cv;
        for (int w = 0; w < wave; ++w) run += wtot[w];
        out.counts[tid] = cv;
        out.offsets[tid] = run;
        if (tid == E - 1) out.offsets[E] = run + cv;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const int c = whist[w][tid];
            whist[w][tid] = run;
            run += c;
        }
    }
    if (out.one_group && tid < 2) out.one_group[tid] = tid ? nk / k : 0;
    const int busy = __syncthreads_count(tid < E && cv > 0);
    for (int i = tid; i < out.n_arrivals; i += 64 * NW) out.arrivals[i] = -(busy + (out.one_group ? 1 : 0));
    for (int i = tid; i < out.n_claims; i += 64 * NW) out.claims[i] = 0;
    int* cur = whist[wave];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        if (64 * it >= slice) break;
        const int g = wbase + 64 * it + lane;
        const int e = ev[it];
        const bool ok = e >= 0;
        if (g < nk && !ok) out.pos[g] = -1;    // no sorted row, the combine skips the slot
        uint64_t peers = __ballot(ok);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const bool bit = (e >> b) & 1;
            const uint64_t bal = __ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        const uint64_t below = peers & ((1ull << lane) - 1ull);
        if (ok) {
            const int r = cur[e] + __popcll(below);
            out.perm[r] = g;
            out.pos[g] = r;
            if (out.row_map) out.row_map[r] = g / k;
        }
        if (ok && below == 0) cur[e] += __popcll(peers);
    }
}

// ---- launches behind the layer call (each checks its arguments as the entry point of the same name does) ----
// logits into memory; shared: also its gate and up projection, may be NULL (for kRouterSharedE < E and up to kTailTokens tokens)
constexpr int kRouterSharedE = 32;
// workgroups of the logits launch in front of the shared expert's: a block of 32 experts each, for the one block of tokens and seven
// that find none (workgroups go to the XCDs round robin)
constexpr int router_shared_front(int E) { return 8 * ((E + 31) / 32); }
int router_logits(const void* x, const void* w_gate, const moe_router_params& p, float* logits, const SharedFirst* shared, hipStream_t st);
// routes from them; logits_bf16: also written as bf16 (Mixtral's second result), may be NULL
int router_select(const float* bias, const moe_router_params& p, int32_t* topk_idx, float* topk_w, float* logits,
                  uint16_t* logits_bf16, hipStream_t st);
// the same and the dispatch in one launch, for up to select_dispatch_tokens(E) tokens: one pass of its 16 waves, of which
// each routes 64 / (lanes per token) at once.  (Four passes of DeepSeek-V2-236B's 160 experts, 64 tokens: 24 us, the two
// launches 10.)
constexpr int select_dispatch_tokens(int E) { return SMALL_WAVES * (E <= 16 ? 4 : E <= 32 ? 2 : 1); }
constexpr int kSelectDispatchTokens = 64;
// logits, routing and dispatch in one launch of one workgroup, where its 4 waves route the tokens in one pass (with 64 experts one
// CU fetches the gate no sooner than two launches are done: DeepSeek-V2-Lite, 1 token, 9.7 + 4.4 us and 14.3)
constexpr int router_dispatch_tokens(int E) { return E <= 16 ? 16 : E <= 32 ? 8 : 0; }
int router_dispatch(const void* x, const void* w_gate, const float* bias, const moe_router_params& p, int32_t* topk_idx, float* topk_w,
                    uint16_t* logits_bf16, const DispatchOut& out, hipStream_t st);
int router_select_dispatch(const float* bias, const moe_router_params& p, int32_t* topk_idx, float* topk_w, float* logits,
                           uint16_t* logits_bf16, const DispatchOut& out, hipStream_t st);
int check_router(const void* x, const void* w_gate, const moe_router_params* params, const int32_t* topk_idx, const float* topk_w);
int dispatch_on_stream(const int32_t* topk_idx, int32_t n_tokens, int32_t top_k, int32_t n_experts, const DispatchOut& out,
                       void* workspace, hipStream_t st);

}  // namespace moe
