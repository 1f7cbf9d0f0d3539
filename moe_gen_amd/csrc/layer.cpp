// A whole MoE-layer call (norm, router, dispatch, expert MLPs, combine) as one host call: the launches of the separate
// entry points with their intermediate buffers carved out of one workspace.  From Python the separate calls cost 5 to
// 15 us of host time each, more than a decode-sized step runs on the GPU.
#include "common.h"
#include "dispatch_small.h"
#include "layer.h"

namespace moe {
namespace {

// byte offsets of the intermediate buffers in the workspace
struct Layout {
    size_t logits, x_norm, offsets, one_group, perm, pos, row_map, segments, arrivals, claims, act, y, act_shared, y_shared, total;
};

Layout layout_of(const moe_layer_args& a) {
    const moe_router_params& p = *a.router;
    const size_t n = p.n_tokens, h = p.hidden, E = p.n_experts, k = p.top_k, nk = n * k;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += (bytes + 255) & ~(size_t)255;
        return here;
    };
    Layout l{};
    l.logits = take(n * E * 4);
    l.x_norm = take(a.norm_weight ? n * h * 2 : 0);
    l.offsets = take((E + 1) * 4);
    l.one_group = take(8);
    l.perm = take(nk * 4);
    l.pos = take(nk * 4);
    l.row_map = take(nk * 4);
    l.segments = take(moe_dispatch_workspace_bytes(p.n_tokens, p.top_k, p.n_experts));
    l.arrivals = take(n <= kTailTokens ? tail_arrivals(p.hidden) * 4 : 0);
    moe_mlp_group routed = *a.routed, shared = a.shared ? *a.shared : moe_mlp_group{};
    routed.n_rows = (int32_t)nk;
    shared.n_rows = (int32_t)n;
    l.claims = take(layer_claims(routed, a.shared ? &shared : nullptr, p.hidden) ? kLayerClaims * 4 : 0);
    l.act = take(nk * (size_t)a.routed->inter * 2);
    l.y = take(nk * h * 2);
    if (a.shared) {
        l.act_shared = take(n * (size_t)a.shared->inter * 2);
        l.y_shared = take(n * h * 2);
    }
    l.total = at;
    return l;
}

int check(const moe_layer_args* a, const char* who) {
    MOE_REQUIRE(a && a->router && a->routed, "%s: NULL arguments", who);
    const moe_router_params& p = *a->router;
    MOE_REQUIRE(p.n_tokens >= 0 && p.hidden > 0 && p.top_k >= 1, "%s: bad sizes", who);
    MOE_REQUIRE((int64_t)p.n_tokens * p.top_k < (int64_t)1 << 31, "%s: n_tokens*top_k does not fit int32", who);
    MOE_REQUIRE(a->routed->n_experts == p.n_experts && a->routed->inter > 0, "%s: router and experts do not match", who);
    MOE_REQUIRE(!a->shared || (a->shared->n_experts == 1 && a->shared->inter > 0), "%s: the shared expert is one MLP", who);
    return MOE_OK;
}

}  // namespace
}  // namespace moe

extern "C" size_t moe_layer_workspace_bytes(const moe_layer_args* args) {
    using namespace moe;
    return check(args, "moe_layer_workspace_bytes") == MOE_OK ? layout_of(*args).total : 0;
}

extern "C" int moe_layer_forward(const moe_layer_args* args, void* stream) {
    using namespace moe;
    const char* who = "moe_layer_forward";
    int rc = check(args, who);
    if (rc != MOE_OK) return rc;
    const moe_layer_args& a = *args;
    const moe_router_params& p = *a.router;
    const int n = p.n_tokens, h = p.hidden, k = p.top_k, E = p.n_experts;
    MOE_REQUIRE(a.counts, "%s: NULL counts", who);
    const Layout l = layout_of(a);
    if (a.workspace == nullptr || a.workspace_bytes < l.total) {
        set_error("%s: workspace %zu bytes, need %zu", who, a.workspace ? a.workspace_bytes : 0, l.total);
        return MOE_ERR_WORKSPACE;
    }
    uint8_t* ws = static_cast<uint8_t*>(a.workspace);
    if (n == 0) return moe_dispatch(nullptr, 0, k, E, a.counts, reinterpret_cast<int32_t*>(ws + l.offsets), nullptr, nullptr, nullptr,
                                    nullptr, 0, nullptr, nullptr, 0, stream);
    MOE_REQUIRE(a.x && a.out, "%s: NULL pointer argument", who);
    const hipStream_t st = as_stream(stream);
    rc = check_router(a.x, a.w_gate, &p, a.topk_idx, a.topk_w);
    if (rc != MOE_OK) return rc;
    const void* x = a.x;
    if (a.norm_weight) {
        rc = moe_rmsnorm(a.x, a.norm_weight, a.norm_eps, n, h, ws + l.x_norm, stream);
        if (rc != MOE_OK) return rc;
        x = ws + l.x_norm;
    }
    float* logits = reinterpret_cast<float*>(ws + l.logits);
    auto ints = [&](size_t off) { return reinterpret_cast<int32_t*>(ws + off); };
    DispatchOut d{a.counts, ints(l.offsets), ints(l.perm), ints(l.pos), ints(l.row_map), a.shared ? ints(l.one_group) : nullptr};
    // Of a few tokens the down projection may combine too (what a separate call would refuse is left to it)
    const void* const y_shared = a.shared ? ws + l.y_shared : nullptr;
    const CombineTail tail{d.pos, a.topk_idx, a.topk_w, static_cast<const uint16_t*>(a.norm_weight ? a.x : nullptr),
                           static_cast<uint16_t*>(a.out), ints(l.arrivals), n, k, a.combine_mode};
    const bool may_combine = n <= kTailTokens && n <= select_dispatch_tokens(E) && a.combine_mode >= MOE_COMBINE_F32 &&
                             a.combine_mode <= MOE_COMBINE_BF16_SEQ && a.out != ws + l.y && a.out != y_shared &&
                             layer_may_combine(E, n * k, a.shared != nullptr, h);
    if (may_combine) {
        d.arrivals = tail.arrivals;
        d.n_arrivals = tail_arrivals(h);
    }
    LayerCall call;
    call.tail = may_combine ? &tail : nullptr;

    moe_mlp_group routed = *a.routed;
    routed.x = x; routed.x_rows = n; routed.n_rows = n * k; routed.row_map = d.row_map; routed.offsets = d.offsets;
    routed.max_rows = n;
    routed.act = ws + l.act; routed.y = ws + l.y;
    routed.workspace = nullptr; routed.workspace_bytes = 0;       // (the caller's fields may hold anything)
    moe_mlp_group shared{};
    if (a.shared) {
        shared = *a.shared;
        shared.x = x; shared.x_rows = shared.n_rows = shared.max_rows = n; shared.row_map = nullptr; shared.offsets = d.one_group;
        shared.act = ws + l.act_shared; shared.y = ws + l.y_shared;
        shared.workspace = nullptr; shared.workspace_bytes = 0;
    }
    const bool join = a.shared && a.join_shared && shared.fp8 == routed.fp8;
    SharedFirst first{};
    if (join && n <= kTailTokens && E > kRouterSharedE && layer_shared_first(routed, shared, h)) {
        first = SharedFirst{shared.w_gate, shared.w_up, shared.s_gate, shared.s_up, static_cast<const uint16_t*>(x),
                            static_cast<uint16_t*>(shared.act), n, h, shared.inter, shared.fp8, 0};
        call.shared_gate_up_done = true;
    }
    if (layer_claims(routed, a.shared && !(join && layer_joins(routed, shared, h)) ? &shared : nullptr, h)) {
        call.claims = d.claims = ints(l.claims);
        d.n_claims = kLayerClaims;
    }
    const SharedFirst* const with = call.shared_gate_up_done ? &first : nullptr;

    uint16_t* logits_bf16 = static_cast<uint16_t*>(a.logits_bf16);
    if (!with && n <= router_dispatch_tokens(E)) {
        rc = router_dispatch(x, a.w_gate, a.bias, p, a.topk_idx, a.topk_w, logits_bf16, d, st);
    } else {
        rc = router_logits(x, a.w_gate, p, logits, with, st);
        if (rc == MOE_OK && n <= select_dispatch_tokens(E)) {
            rc = router_select_dispatch(a.bias, p, a.topk_idx, a.topk_w, logits, logits_bf16, d, st);
        } else if (rc == MOE_OK) {
            rc = router_select(a.bias, p, a.topk_idx, a.topk_w, logits, logits_bf16, st);
            if (rc == MOE_OK) rc = dispatch_on_stream(a.topk_idx, n, k, E, d, ws + l.segments, st);
        }
    }
    if (rc != MOE_OK) return rc;

    if (join || !a.shared) {
        rc = layer_experts(routed, join ? &shared : nullptr, h, routed.fp8, &call, stream);
    } else {
        call.tail = nullptr;
        rc = layer_experts(routed, nullptr, h, routed.fp8, &call, stream);
        if (rc == MOE_OK) rc = layer_experts(shared, nullptr, h, shared.fp8, &call, stream);
    }
    if (rc != MOE_OK || call.combined) return rc;
    if (a.norm_weight)
        return moe_combine_residual(ws + l.y, d.pos, a.topk_idx, a.topk_w, y_shared, a.x, n, k, h, a.combine_mode, a.out, stream);
    return moe_combine(ws + l.y, d.pos, a.topk_idx, a.topk_w, y_shared, n, k, h, a.combine_mode, a.out, stream);
}
