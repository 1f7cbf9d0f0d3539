// MoE router for gfx950: logits, scores, group-limited top-k, renormalisation and routed scaling.
//
// Replaces MoEGate.forward of the reference (modeling_deepseek_v3.py:500-561,
// modeling_deepseek_v2.py:483-533) and the routing lines of transformers-4.42.0
// MixtralSparseMoeBlock.forward.
//
// Logits.  logit[t,e] = sum_k x[t,k] * W[e,k] is evaluated in fp32 in ONE fixed
// order -- acc = fma(x[k], W[k], acc) for k = 0..h-1 -- so that the selected
// expert indices are a pure function of the inputs.  The fp32 matrix core gives exactly that order at twice the rate
// of the vector ALU (router_logits_kernel).
//
// Selection.  A second kernel routes the tokens from the logits in memory, a lane group per token with its lanes
// strided over the experts.  Ties go to the lower expert (group) index and the slot order of the output is the
// selection order (descending score).
#include <type_traits>

#include "common.h"
#include "dispatch_small.h"
#include "moe_math.h"
#include "thin_gemm.h"

namespace moe {
namespace {

// Lanes of a wave work in groups of GW (64, or 16 / 32 when E <= 16 / 32): a group routes one token, its lanes strided
// over the experts (lane g of the group holds experts g, g+GW, ...).

// Value held by the lane's xor-M partner, without going through LDS: cross-row exchanges with
// the gfx950 lane-swap instructions, inside a 16-lane row with DPP.  M = 4 uses a rotation by 4,
// which delivers the xor-4 partner's VALUE whenever the data already agrees between lanes l and
// l^8 -- true in every butterfly below, where the step for 8 precedes the step for 4.
template <int M>
__device__ __forceinline__ int partner_bits(int x) {
    const int lane = threadIdx.x & 63;
    if constexpr (M == 32) {
        auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);   // r[0] = low half twice, r[1] = high half twice
        return (lane & 32) ? (int)r[0] : (int)r[1];
    } else if constexpr (M == 16) {
        auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);   // r[0] = even rows twice, r[1] = odd rows twice
        return (lane & 16) ? (int)r[0] : (int)r[1];
    } else if constexpr (M == 8) {
        return __builtin_amdgcn_update_dpp(x, x, 0x128, 0xf, 0xf, false);   // row_ror:8
    } else if constexpr (M == 4) {
        return __builtin_amdgcn_update_dpp(x, x, 0x124, 0xf, 0xf, false);   // row_ror:4
    } else if constexpr (M == 2) {
        return __builtin_amdgcn_update_dpp(x, x, 0x4E, 0xf, 0xf, false);    // quad_perm [2,3,0,1]
    } else {
        return __builtin_amdgcn_update_dpp(x, x, 0xB1, 0xf, 0xf, false);    // quad_perm [1,0,3,2]
    }
}
template <int M>
__device__ __forceinline__ float partner(float v) {
    return __builtin_bit_cast(float, partner_bits<M>(__builtin_bit_cast(int, v)));
}

template <int GW, int M = GW / 2, typename F>
__device__ __forceinline__ void butterfly(F&& step) {
    if constexpr (M >= 1) {
        step(std::integral_constant<int, M>{});
        butterfly<GW, M / 2>(step);
    }
}

template <int GW>
__device__ __forceinline__ float group_max(float v) {
    butterfly<GW>([&](auto m) { v = fmaxf(v, partner<decltype(m)::value>(v)); });
    return v;
}
template <int GW>
__device__ __forceinline__ uint32_t group_max(uint32_t v) {
    butterfly<GW>([&](auto m) { v = max(v, (uint32_t)partner_bits<decltype(m)::value>((int)v)); });
    return v;
}

// The canonical sum over experts: 64 strided partials folded by the butterfly 32,16,8,4,2,1
// (p[l] += p[l^m]; fp32 addition commutes).  With E <= 16 (E <= 32) the partials of lanes 16..63
// (32..63) are +0, the leading steps add +0 to non-negative values, and the remaining steps are the
// 16-lane (32-lane) butterfly.
template <int GW>
__device__ __forceinline__ float group_sum_butterfly(float v) {
    butterfly<GW>([&](auto m) { v = v + partner<decltype(m)::value>(v); });
    return v;
}

constexpr float kNegInf = -__builtin_inff();

// Order of the selections as an unsigned key: by value, +0 and -0 equal, NaN above every number (as torch.topk ranks
// it) and all NaNs equal, so a NaN score is selected first, every lane of a group reaches the same decision and the
// indices written stay inside [0, E); the NaN then travels on through the weights.  0 is below every value's key.
__device__ __forceinline__ uint32_t order_key(float v) {
    const uint32_t u = __float_as_uint(v + 0.0f);
    return v != v ? 0xffffffffu : (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// lowest lane of the lane group that starts at gbase whose `hit` is true, or GW if there is none
template <int GW>
__device__ __forceinline__ int first_lane(bool hit, int gbase) {
    const uint64_t b = __ballot(hit);
    if constexpr (GW == 64) return b ? __builtin_ctzll(b) : 64;
    const uint32_t m = (uint32_t)(b >> gbase) & (GW == 32 ? 0xffffffffu : (1u << GW) - 1u);
    return m ? __builtin_ctz(m) : GW;
}

// Routes one token per lane group; `row` points at the group's logits (E valid entries), `val` at the group's MAX_EJ * GW
// floats of LDS.  `live` is false for groups without a token (they run the same code on a valid row, store nothing).
// A selection is a maximum over order keys (one vector instruction per butterfly step) and a ballot for the lowest
// index that holds it; an expert group's score is gathered from LDS by GW / n_group lanes.  (With (value, index) pairs
// in the butterflies and one butterfly per expert group a token took 4 times as long.)
template <int GW, int MAX_EJ>
__device__ void route_token(const float* row, const float* __restrict__ bias, const moe_router_params& p,
                            int32_t* __restrict__ idx_out, float* __restrict__ w_out,
                            float* logits_out, uint16_t* logits_bf16, float* val, bool live) {
    // MAX_EJ: experts per lane, ceil(padded experts / GW)
    const int lane = threadIdx.x & 63, gl = lane & (GW - 1), gbase = lane - gl;
    const int E = p.n_experts;
    float L[MAX_EJ], s[MAX_EJ], c[MAX_EJ];
    bool valid[MAX_EJ];
#pragma unroll
    for (int j = 0; j < MAX_EJ; ++j) {
        int e = gl + GW * j;
        valid[j] = e < E;
        L[j] = row[valid[j] ? e : 0];
        c[j] = p.method == MOE_TOPK_NOAUX_TC && bias != nullptr ? bias[valid[j] ? e : 0] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < MAX_EJ; ++j) {
        if (!valid[j]) L[j] = 0.0f;
        if (p.logits_bf16) L[j] = round_to_bf16(L[j]);
        if (logits_out && valid[j] && live) logits_out[gl + GW * j] = L[j];
        if (logits_bf16 && valid[j] && live) logits_bf16[gl + GW * j] = (uint16_t)f32_to_bf16_bits(L[j]);
    }
    if (p.scoring == MOE_SCORE_SIGMOID) {
#pragma unroll
        for (int j = 0; j < MAX_EJ; ++j) s[j] = valid[j] ? canon_sigmoidf(L[j]) : 0.0f;
    } else {
        float m = kNegInf;
#pragma unroll
        for (int j = 0; j < MAX_EJ; ++j) m = valid[j] ? fmaxf(m, L[j]) : m;
        m = group_max<GW>(m);
        float part = 0.0f;
#pragma unroll
        for (int j = 0; j < MAX_EJ; ++j) {
            s[j] = valid[j] ? canon_expf(L[j] - m) : 0.0f;
            part = part + s[j];  // adding +0 for absent experts changes nothing
        }
        float sum = group_sum_butterfly<GW>(part);
#pragma unroll
        for (int j = 0; j < MAX_EJ; ++j) s[j] = s[j] / sum;
    }
#pragma unroll
    for (int j = 0; j < MAX_EJ; ++j) c[j] = p.method == MOE_TOPK_NOAUX_TC && bias != nullptr ? s[j] + c[j] : s[j];

    float tmp[MAX_EJ];
#pragma unroll
    for (int j = 0; j < MAX_EJ; ++j) tmp[j] = c[j];
    if (p.method != MOE_TOPK_GREEDY) {
        const int G = p.n_group, per = E / G;
        const int g_log2 = G <= 1 ? 0 : 32 - __builtin_clz(G - 1);
        const int lpg = GW >> g_log2;                       // lanes per expert group (G <= E <= 32 where GW < 64)
#pragma unroll
        for (int j = 0; j < MAX_EJ; ++j) val[gl + GW * j] = c[j];
        __builtin_amdgcn_wave_barrier();
        const int g = gl / lpg, sub = gl - g * lpg;
        float m1 = kNegInf, m2 = kNegInf;
        bool nan = false;
        if (g < G)
            for (int i = sub; i < per; i += lpg) {
                const float v = val[g * per + i];
                nan |= v != v;
                m2 = fmaxf(m2, fminf(m1, v));
                m1 = fmaxf(m1, v);
            }
        __builtin_amdgcn_wave_barrier();
        // fold the lanes of an expert group, nearest first: inside 16 lanes a mirror brings the other half's (already
        // agreed) value
        auto fold = [&](float o1, float o2, int on) {
            m2 = fmaxf(fminf(m1, o1), fmaxf(m2, o2));
            m1 = fmaxf(m1, o1);
            nan |= on != 0;
        };
        auto dpp = [&](auto ctrl) {
            constexpr int C = decltype(ctrl)::value;
            const int n0 = nan;
            fold(__builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, m1), C, 0xf, 0xf, false)),
                 __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, m2), C, 0xf, 0xf, false)),
                 __builtin_amdgcn_update_dpp(0, n0, C, 0xf, 0xf, false));
        };
        if (lpg > 1) dpp(std::integral_constant<int, 0xB1>{});        // xor 1
        if (lpg > 2) dpp(std::integral_constant<int, 0x4E>{});        // xor 2
        if (lpg > 4) dpp(std::integral_constant<int, 0x141>{});       // row_half_mirror
        if (lpg > 8) dpp(std::integral_constant<int, 0x140>{});       // row_mirror
        if (lpg > 16) fold(partner<16>(m1), partner<16>(m2), partner_bits<16>(nan));
        if (GW == 64 && lpg > 32) fold(partner<32>(m1), partner<32>(m2), partner_bits<32>(nan));
        // noaux_tc: sum of the two largest of the group; otherwise its largest
        const float gs = nan ? __builtin_nanf("") : p.method == MOE_TOPK_NOAUX_TC ? m1 + m2 : m1;
        uint32_t gkey = g < G && sub == 0 ? order_key(gs) : 0u;
        uint32_t keep = 0;
        for (int r = 0; r < p.topk_group; ++r) {
            const int best = first_lane<GW>(gkey == group_max<GW>(gkey), gbase);
            if (gl == best) gkey = 0u;
            keep |= 1u << (best / lpg);
        }
        const uint32_t inv = (1u << 20) / (uint32_t)per + 1u;     // e / per = e * inv >> 20 for e < 256
#pragma unroll
        for (int j = 0; j < MAX_EJ; ++j)
            tmp[j] = ((keep >> (((uint32_t)(gl + GW * j) * inv >> 20) & 31u)) & 1u) ? c[j] : 0.0f;  // masked_fill(~mask, 0.0)
    }
    // the values a winner's weight is read from: V3 gathers the unbiased score, V2 / Mixtral keep the selected value
#pragma unroll
    for (int j = 0; j < MAX_EJ; ++j) val[gl + GW * j] = p.method == MOE_TOPK_NOAUX_TC ? s[j] : tmp[j];

    // top-k by repeated maximum; lane r of the group keeps slot r
    uint32_t key[MAX_EJ];
#pragma unroll
    for (int j = 0; j < MAX_EJ; ++j) key[j] = valid[j] ? order_key(tmp[j]) : 0u;
    int my_idx = 0;
    for (int r = 0; r < p.top_k; ++r) {
        uint32_t m = key[0];
#pragma unroll
        for (int j = 1; j < MAX_EJ; ++j) m = max(m, key[j]);
        m = group_max<GW>(m);
        int best = 0;
#pragma unroll
        for (int j = MAX_EJ - 1; j >= 0; --j) {
            const int l = first_lane<GW>(key[j] == m, gbase);
            best = l < GW ? l + GW * j : best;
        }
#pragma unroll
        for (int j = 0; j < MAX_EJ; ++j) key[j] = best == gl + GW * j ? 0u : key[j];
        my_idx = gl == r ? best : my_idx;
    }
    __builtin_amdgcn_wave_barrier();
    float my_w = val[my_idx];
    if (p.top_k > 1 && p.norm_topk_prob) {
        float sum = 0.0f;
        for (int r = 0; r < p.top_k; ++r) sum = sum + __shfl(my_w, gbase + r);
        float den = sum + p.norm_eps;
        my_w = my_w / den;
        if (p.scale_mode == MOE_SCALE_ALWAYS) my_w = my_w * p.routed_scaling_factor;
    } else if (p.scale_mode >= MOE_SCALE_IF_NOT_NORM) {
        my_w = my_w * p.routed_scaling_factor;
    }
    if (p.weights_bf16) my_w = round_to_bf16(my_w);
    if (live && gl < p.top_k) {
        idx_out[gl] = my_idx;
        w_out[gl] = my_w;
    }
    __builtin_amdgcn_wave_barrier();                              // (the next token of the wave overwrites val)
}

// The logit engine.  v_mfma_f32_16x16x4_f32 adds its four products one after the other, each as one fused
// multiply-add in fp32 (lane group q of the operands holds k = 4j + q, and the accumulation runs q = 0 .. 3):
// exactly the canonical chain, four k per instruction.  (Checked bit for bit against fma chains on 14.7 million
// outputs: normal, wide-range, cancelling, subnormal and signed-zero operands.)  It issues every 32 cycles whether or
// not it depends on the one before, 8 cycles per k of a chain: the 4x4x1 form takes 12.7 per dependent k, a v_fmac_f32
// chain 9.2, and 16 x 16 outputs in 32 cycles per 4 k are the full fp32 matrix rate.  So ONE wave with ONE accumulator
// tile already runs its SIMD's matrix core without a gap, and few tokens and many are the same engine.
//  * Tile: WT waves along tokens x WE along experts, each TT x TE tiles of 16 tokens x 16 experts.  Few tokens take one
//    tile per wave (a chain of h / 4 instructions) and as many CUs as there are
//    there are tiles; many tokens 2 x 2 tiles per wave (half the operand reads).
//  * The fp32 matrix instructions run on the vector ALU's lanes: ONE vector instruction between two of them costs 13
//    cycles, more of them 5 each, while LDS reads, DMA and scalar instructions issue beside them for nothing (a CU
//    serves one LDS read of up to 4 bytes a lane every 4 cycles).  So the k loop holds no vector instruction: a lane
//    needs ONE bf16 of its row per instruction, in the upper half of a register whose lower half stays zero, and
//    ds_read_u16_d16_hi is that load and the conversion to fp32 in one; every address is a base register of the stage
//    plus a constant.  The reads run DEPTH steps ahead in a ring of registers (as far as the 4-bit counter of
//    outstanding LDS reads allows).
//  * Operands reach LDS as bf16 by DMA, 128 k of each row per stage, S stages in a ring, one barrier per stage.  A DMA
//    instruction brings four rows as 16 chunks of 4 x 16 bytes, and blocks of four rows lie 1088 bytes apart: the 16
//    rows of a read fall on 64 different banks and the next k are at a constant distance.
//  * The last stage of a hidden size that is no multiple of 128 stops after its h / 4 steps: nothing is padded.
// Measured (DeepSeek-V3, h = 7168, logits and selection in a loop on the same rows): 1 ... 256 tokens 35 ... 37 us (the chain
// alone at 32 cycles per step and 2.4 GHz: 24), 1024: 37, 65536: 1716 = 140 TFLOP/s (between the other kernels of a layer 1807 + 80).  Without the LDS reads the 65536-token logits take 1587,
// without the DMA 1674, with both 1645.  (Before, on the 4x4x1 and 32x32x1 forms, which take one k per instruction:
// 92 ... 96, 96 and 2133 us.)
// FUSED == false: the logits of the tile go to `logits` [n, E] in memory, router_select_kernel routes the tokens.
// FUSED == true (a caller without a logits buffer): the workgroup walks the expert blocks of its tokens one after the
// other, keeps the logits in LDS and routes the tokens itself.  Where that leaves most CUs without tokens
// router_tokens_kernel takes the call.
// DISPATCH (with FUSED, one workgroup): it sorts the tokens' experts too, for a few tokens of up to 32 experts.
// Mixtral-8x7B, 1 token, us: two launches 17.4 + 4.9, this 20.9.
// SHARED (1 bf16, 2 fp8 weights): workgroups behind the router's bring the shared expert's gate and up projection (SharedFirst).

constexpr int kStageBytes = 256, kStepsPerStage = 32;    // 128 k of a row per stage, 4 k per step
constexpr int kBlock = 1024 + 64;                        // four rows of a stage in LDS

constexpr int ring_depth(int reads) { return 15 / reads > 7 ? 7 : 15 / reads; }

// f(0), f(1), ... f(N - 1) with the index as a constant
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

// two bytes of LDS into the upper half of a register, whose lower half stays as it is: a bf16 as fp32
template <int OFF>
__device__ __forceinline__ void read_bf16_as_f32(float& v, uint32_t addr) {
    asm volatile("ds_read_u16_d16_hi %0, %1 offset:%2" : "+v"(v) : "v"(addr), "n"(OFF));
}

template <int WT, int WE, int TT, int TE, int S, bool FUSED, int GW, int EJ, bool DISPATCH = false, int SHARED = 0>   // (GW, EJ: route_token; read where FUSED)
__global__ __launch_bounds__(64 * WT * WE, 1) void router_logits_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ wg, const float* __restrict__ bias,
    moe_router_params p, int32_t* topk_idx, float* __restrict__ topk_w, float* __restrict__ logits, uint16_t* __restrict__ logits_bf16,
    DispatchOut out, SharedFirst shared) {
    static_assert(FUSED || !DISPATCH, "the tokens of one workgroup");
    static_assert(TT == TE && TT <= 2, "one tile per wave or 2 x 2");
    constexpr int NW = WT * WE, BT = 16 * TT * WT, BE = 16 * TE * WE;
    constexpr int NX = BT / (4 * NW), NE = BE / (4 * NW), NI = NX + NE;   // DMA instructions (4 rows each) per wave and stage
    constexpr int SB = (BT + BE) / 4 * kBlock;                  // bytes of a stage, token rows first
    constexpr int R = TT + TE, DEPTH = ring_depth(R), RING = DEPTH > 3 ? 8 : 4;
    static_assert((TT == 1 ? RING == 8 : RING == 4) && NI <= 10 && DEPTH < RING && DEPTH >= 2 && S >= 3 && (S - 2) * NI < 64, "counters");
    constexpr int LG = GW == 64 ? 64 * EJ : BE;                 // row of the logits kept in LDS: whole expert blocks
    static_assert(LG % BE == 0, "expert blocks");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[S * SB];
    __shared__ float lg[FUSED ? BT * LG : 1];
    constexpr bool VAL_IN_STAGES = S == 3;                      // the selection's values in the stage buffers: two workgroups per CU then fit
    static_assert(NW * 64 * EJ * 4 <= S * SB, "selection");
    __shared__ float val_own[FUSED && !VAL_IN_STAGES ? NW * 64 * EJ : 1];
    if constexpr (SHARED != 0) {
        // one wave of the workgroup, whose LDS is its ring: the launch has no more workgroups than CUs (layer_shared_first)
        constexpr bool W8 = SHARED == 2;
        constexpr int STAGES = W8 ? 8 : 11;                     // as many as the counter of outstanding loads allows
        static_assert(STAGES * thin_stage_bytes<W8, 2> <= S * SB, "ring");
        if ((int)blockIdx.x >= shared.first_block) {
            if (threadIdx.x < 64)
                thin_columns<true, W8, 2, false, STAGES>(ThinUnit{shared.w_gate[0], shared.w_up[0], W8 ? shared.s_gate[0] : nullptr,
                                                                  W8 ? shared.s_up[0] : nullptr, shared.x, nullptr, 0, 0, shared.act, shared.hidden,
                                                                  shared.inter, 0, shared.rows}, 16 * ((int)blockIdx.x - shared.first_block), lds);
            return;
        }
    }

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wt = wave / WE, we = wave % WE;
    const int n = p.n_tokens, h = p.hidden, E = p.n_experts;
    // expert blocks of one token block on one XCD (workgroups go to the XCDs round robin): its rows are fetched once
    const int neb = (E + BE - 1) / BE;
    const int local = blockIdx.x >> 3;
    const int t0 = FUSED ? blockIdx.x * BT : ((local / neb) * 8 + (blockIdx.x & 7)) * BT;
    int e0 = FUSED ? 0 : (local % neb) * BE;
    if (t0 >= n) return;
    do {                                                        // (FUSED: once per expert block)

        // DMA: instruction i of this wave brings block wave + NW i of the stage, lane l chunk l / 4 of row l % 4; rows past
        // the end re-read the last one, chunks past h (last stage) fetch what follows in memory, or zeros past the end of
        // the buffer: neither is multiplied
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)(x + (size_t)t0 * h), 0, min(BT, n - t0) * h * 2, 0x00020000);
        const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)(wg + (size_t)e0 * h), 0, min(BE, E - e0) * h * 2, 0x00020000);
        int voff[10];                                               // (NI <= 10 are used)
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int g = 4 * (wave + NW * i) + (lane & 3);         // row of the stage
            const int row = i < NX ? min(g, n - 1 - t0) : min(g - BT, E - 1 - e0);
            voff[i] = row * h * 2 + ((lane >> 2) << 4);
        }
        auto dma = [&](auto index, int buf, int st) {
            constexpr int i = decltype(index)::value;
            uint8_t* const d = lds + buf * SB + (wave + NW * i) * kBlock;
            const uint32_t soff = (uint32_t)(st * kStageBytes);
            if constexpr (i < NX) __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_u8)d, 16, voff[i], soff, 0, 0);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_u8)d, 16, voff[i], soff, 0, 0);
        };

        // step j of a stage reads chunk j / 2 of the lane's rows, bytes (j & 1) * 8 + 2 q of it
        const int r = lane & 15, q = lane >> 4;
        const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_u8)lds + (r >> 2) * kBlock + (r & 3) * 16 + q * 2;
        const uint32_t xa = lds0 + wt * TT * 4 * kBlock, wa = lds0 + (BT + we * TE * 16) / 4 * kBlock;
        float a[RING][TT], b[RING][TE];
#pragma unroll
        for (int i = 0; i < RING; ++i) {
#pragma unroll
            for (int j = 0; j < TT; ++j) a[i][j] = 0.0f;
#pragma unroll
            for (int j = 0; j < TE; ++j) b[i][j] = 0.0f;
        }
        auto read_step = [&](auto step, uint32_t xbase, uint32_t wbase, auto ring_slot) {
            constexpr int OFF = (decltype(step)::value >> 1) * 64 + (decltype(step)::value & 1) * 8, SLOT = decltype(ring_slot)::value;
            static_for<TT>([&](auto i) { read_bf16_as_f32<i * 4 * kBlock + OFF>(a[SLOT][i], xbase); });
            static_for<TE>([&](auto i) { read_bf16_as_f32<i * 4 * kBlock + OFF>(b[SLOT][i], wbase); });
        };
        f32x4 acc[TT][TE];
#pragma unroll
        for (int i = 0; i < TT; ++i)
#pragma unroll
            for (int j = 0; j < TE; ++j) acc[i][j] = f32x4{0, 0, 0, 0};
        auto multiply_step = [&](auto ring_slot, auto outstanding) {    // waits until at most that many reads are outstanding
            constexpr int slot = decltype(ring_slot)::value, N = decltype(outstanding)::value;
            if constexpr (TT == 1 && TE == 1) asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(a[slot][0]), "+v"(b[slot][0]) : "n"(N));
            else
                asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(a[slot][0]), "+v"(a[slot][1]), "+v"(b[slot][0]), "+v"(b[slot][1]) : "n"(N));
#pragma unroll
            for (int i = 0; i < TT; ++i)
#pragma unroll
                for (int j = 0; j < TE; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[slot][i], b[slot][j], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);                      // the reads that refill these registers stay behind
        };

        // Waits for every read.  All ring registers are its operands: a read that nothing uses any more (the last ones run
        // past the end) still writes its register, which the compiler must not give to anything else before that.
        auto drain = [&] {
            if constexpr (TT == 1)
                asm volatile("s_waitcnt lgkmcnt(0)"
                             : "+v"(a[0][0]), "+v"(a[1][0]), "+v"(a[2][0]), "+v"(a[3][0]), "+v"(a[4][0]), "+v"(a[5][0]),
                               "+v"(a[6][0]), "+v"(a[7][0]), "+v"(b[0][0]), "+v"(b[1][0]), "+v"(b[2][0]), "+v"(b[3][0]),
                               "+v"(b[4][0]), "+v"(b[5][0]), "+v"(b[6][0]), "+v"(b[7][0]));
            else
                asm volatile("s_waitcnt lgkmcnt(0)"
                             : "+v"(a[0][0]), "+v"(a[1][0]), "+v"(a[2][0]), "+v"(a[3][0]), "+v"(a[0][1]), "+v"(a[1][1]),
                               "+v"(a[2][1]), "+v"(a[3][1]), "+v"(b[0][0]), "+v"(b[1][0]), "+v"(b[2][0]), "+v"(b[3][0]),
                               "+v"(b[0][1]), "+v"(b[1][1]), "+v"(b[2][1]), "+v"(b[3][1]));
        };

        const int steps = h / 4, nfull = steps / kStepsPerStage, rem = steps % kStepsPerStage;
        const int nstage = nfull + (rem ? 1 : 0);
        static_for<S - 2>([&](auto st) { static_for<NI>([&](auto i) { dma(i, st, min((int)st, nstage - 1)); }); });
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 3) * NI) : "memory");
        __builtin_amdgcn_s_barrier();
        static_for<DEPTH>([&](auto j) { read_step(j, xa, wa, j); });
        using outstanding_t = std::integral_constant<int, (DEPTH - 1) * R>;
        uint32_t xc = xa, wc = wa;                                  // the stage that is read
        int buf = 0;
        for (int st = 0; st < nfull; ++st) {
            const int next = buf + 1 == S ? 0 : buf + 1;
            const uint32_t xb = xc, wb = wc;
            static_for<kStepsPerStage>([&](auto step) {
                constexpr int j = decltype(step)::value, ahead = (j + DEPTH) % kStepsPerStage;
                multiply_step(std::integral_constant<int, j % RING>{}, outstanding_t{});
                // The DMA of stage st + S - 2, one instruction every few steps (a burst of them blocks the wave's issue, and
                // with it the matrix core), into the buffer that the barrier of the stage before set free.
                static_for<NI>([&](auto i) {
                    if constexpr (j == i * (kStepsPerStage - DEPTH) / NI) dma(i, buf < 2 ? buf + S - 2 : buf - 2, min(st + S - 2, nstage - 1));
                });
                if constexpr (j == kStepsPerStage - DEPTH) {
                    // The reads below are the first of stage st + 1: every wave's part of it has to be there.  The barrier
                    // also says that no wave reads stage st - 1 any more.
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 3) * NI) : "memory");
                    __builtin_amdgcn_s_barrier();
                    xc = xa + next * SB;
                    wc = wa + next * SB;
                }
                constexpr bool same = j + DEPTH < kStepsPerStage;
                read_step(std::integral_constant<int, ahead>{}, same ? xb : xc, same ? wb : wc, std::integral_constant<int, ahead % RING>{});
            });
            buf = next;
        }
        drain();                                                    // the reads ahead of the last whole stage
        if (rem) {
            const uint32_t xb = xa + buf * SB, wb = wa + buf * SB;
            static_for<DEPTH>([&](auto j) { read_step(j, xb, wb, j); });
            static_for<kStepsPerStage - 2>([&](auto step) {
                constexpr int j = decltype(step)::value, ahead = j + DEPTH;
                if (j >= rem) return;
                multiply_step(std::integral_constant<int, j % RING>{},
                              std::integral_constant<int, ahead <= kStepsPerStage ? outstanding_t::value : 0>{});
                if constexpr (ahead < kStepsPerStage)
                    read_step(std::integral_constant<int, ahead>{}, xb, wb, std::integral_constant<int, ahead % RING>{});
            });
            drain();
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");            // no DMA may land in LDS after the workgroup has gone

        // register i of lane l: token 4 q + i, expert r of the tile
#pragma unroll
        for (int ti = 0; ti < TT; ++ti)
#pragma unroll
            for (int te = 0; te < TE; ++te)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int tl = (wt * TT + ti) * 16 + 4 * q + i, e = e0 + (we * TE + te) * 16 + r;
                    if constexpr (FUSED) lg[tl * LG + e] = acc[ti][te][i];
                    else if (t0 + tl < n && e < E) logits[(size_t)(t0 + tl) * E + e] = acc[ti][te][i];
                }
        if constexpr (FUSED) __syncthreads();                   // the logits are there; no wave reads a stage buffer any more
        e0 += BE;
    } while (FUSED && e0 < E);
    if constexpr (FUSED) {
        float* const val = VAL_IN_STAGES ? reinterpret_cast<float*>(lds) : val_own;       // (behind the barrier above)
        constexpr int TPW = 64 / GW;
        for (int tb = wave * TPW; tb < BT; tb += NW * TPW) {
            if (t0 + tb >= n) break;
            const int tl = tb + lane / GW, t = t0 + tl;
            const bool live = t < n;
            const int tr = live ? t : n - 1, tlr = live ? tl : tb;
            route_token<GW, EJ>(lg + tlr * LG, bias, p, topk_idx + (size_t)tr * p.top_k, topk_w + (size_t)tr * p.top_k,
                                nullptr, DISPATCH && logits_bf16 ? logits_bf16 + (size_t)tr * E : nullptr,
                                val + wave * 64 * EJ + lane / GW * (EJ * GW), live);
        }
    }
    if constexpr (DISPATCH) {
        __threadfence_block();
        __syncthreads();                                            // the other waves' indices are in memory
        const volatile int32_t* idx = topk_idx;
        dispatch_one_workgroup<1, NW>(n * p.top_k, E, out, p.top_k, [&](int i) { return idx[i]; });
    }
}

// Logits and selection in one launch for more than 128 experts and up to 1024 tokens whose caller has no logits buffer.
// Sixteen tokens per workgroup, as above, are 64 CUs at most, each with four blocks of experts one after the other
// (DeepSeek-V3's gate, 64 tokens: 143 us).  Here a workgroup takes 4 tokens and a wave 64 experts, in the 4 x 64 layout
// of the 4x4 MFMA: lane l of a wave the expert 64 wave + l.
//  * The 128-byte lines of a wave's 64 gate rows reach its own LDS region as bf16 by DMA (8 instructions per 64 k; chunk c
//    of row r in 16-byte slot c ^ g(r), so that the 16 lanes the LDS serves together -- rows 8i .. 8i+7 and
//    32+8i .. 39+8i -- fall on 16 different bank groups); a lane reads the 8 weights of its expert with one
//    ds_read_b128 and widens them to fp32 between the MFMAs (a shift or a mask each).
//  * The token values never touch LDS: the MFMA broadcasts the A operand of one block to all 16, so a register that
//    holds the 4 tokens' values of 16 consecutive k (one 2-byte load per lane) feeds 16 instructions.
//  * One wave's LDS reads execute in order and its DMA is ordered by vmcnt, so the k loop has no barrier.
// Each logit is the same chain of one fused multiply-add per k as in the engine above.  Per k a wave issues one
// MFMA, one conversion and an eighth of a 16-byte LDS read: 11.9 ns; 9.7 ns without the conversion and 8.3 ns without
// the LDS read either, which is the MFMA chain itself.
__device__ __forceinline__ int thin_slot(int r) { return ((r >> 1) & 3) | (((r >> 5) & 1) << 2); }

// The A operand of block B is broadcast to all 16 blocks of the instruction (cbsz = 4, abid = B), so ONE register holds
// the token values of 16 consecutive k: lanes 4b .. 4b+3 the 4 tokens at k0 + b.  The B operand of lane l is expert l
// of the wave's 64.
template <int B>
__device__ __forceinline__ f32x4 mfma_4_tokens(float a, float b, f32x4 acc) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, acc, 4, B, 0);
}

template <int WE>
__global__ __launch_bounds__(64 * WE, 1) void router_tokens_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ wg, const float* __restrict__ bias,
    moe_router_params p, int32_t* __restrict__ topk_idx, float* __restrict__ topk_w) {
    constexpr int KC = 64, BT = 4, EP = 64 * WE, WBYTES = 64 * 128;
    // (one workgroup per CU) one array per weight buffer: a read of one then never waits for the DMA in flight into another
    __shared__ __attribute__((aligned(1024))) uint8_t wb0[WE * WBYTES];           // written by DMA only
    __shared__ __attribute__((aligned(1024))) uint8_t wb1[WE * WBYTES];
    __shared__ __attribute__((aligned(1024))) uint8_t wb2[WE * WBYTES];
    __shared__ __attribute__((aligned(16))) float lg[BT * EP];
    __shared__ float val[WE * EP];                                                // selection: EP per wave
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = p.n_tokens, h = p.hidden, E = p.n_experts;
    const int t0 = blockIdx.x * BT;
    const int nfull = h / KC, rem8 = (h % KC) / 8, nstage = nfull + (rem8 ? 1 : 0);

    // weight DMA: instruction i brings rows 8i .. 8i+7 of the wave's 64, a lane the chunk that belongs in its slot
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)wg, 0, E * h * 2, 0x00020000);
    int w_voff[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int r = 8 * i + (lane >> 3), c = (lane & 7) ^ thin_slot(r);
        w_voff[i] = (min(64 * wave + r, E - 1) * h + c * 8) * 2;
    }
    auto dma_w = [&](uint8_t* buf, int st) {
        uint8_t* dst = buf + wave * WBYTES;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_u8)(dst + i * 1024), 16, w_voff[i], (uint32_t)(st * (KC * 2)), 0, 0);
    };
    // token values straight from memory into the broadcast layout: register g of a stage holds, in lanes
    // 4b .. 4b+3, element 16 g + b of the 4 tokens (one 2-byte load per lane and 16 k), widened when its 16 k come up
    const uint16_t* const xrow = x + (size_t)min(t0 + (lane & 3), n - 1) * h;
    uint32_t xr[2][4];
    auto load_x = [&](int set, int st) {       // (elements past h are never multiplied: any address inside the row will do)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int k = st * KC + 16 * g + (lane >> 2);
            xr[set][g] = xrow[k < h ? k : 0];
        }
    };

    f32x4 acc = {0, 0, 0, 0};                  // register i: token i, expert 64 wave + lane
    int w_roff[8];                             // chunk c of the lane's row inside a buffer
#pragma unroll
    for (int c = 0; c < 8; ++c) w_roff[c] = wave * WBYTES + lane * 128 + ((c ^ thin_slot(lane)) << 4);

    auto wf = [](const u32x4& v, int j) {      // element j of 8 bf16 as fp32
        return __uint_as_float((j & 1) ? (v[j >> 1] & 0xffff0000u) : (v[j >> 1] << 16));
    };
    // Stage st; the register set st & 1 and the buffers are literals at every call site.  The DMA of stage
    // st + 2 leaves first, then the wait for the DMA of stage st.  Its count is the DMA instructions issued
    // since -- 8 per stage ahead -- and nothing else: the token loads sit behind the wait in program order, but the
    // compiler may place a register load on either side of it, and every one that is in the window only makes the
    // wait stricter (the oldest operations in the window are token loads of a stage ago, long complete).
    auto stage = [&](int st, int set, const uint8_t* wb, uint8_t* wb_refill, int nch) {
        uint32_t xs[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) xs[g] = xr[set][g];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the reads of stage st - 1, a stage old, before their buffer is refilled
        dma_w(wb_refill, min(st + 2, nstage - 1));
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * 8) : "memory");
        load_x(set, min(st + 2, nstage - 1));            // (tokens of stage st + 2 into the set that held stage st)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (2 * g >= nch) break;
            const u32x4 w0 = *reinterpret_cast<const u32x4*>(wb + w_roff[2 * g]);
            const u32x4 w1 = *reinterpret_cast<const u32x4*>(wb + w_roff[2 * g + 1]);
            const float xa = __uint_as_float(xs[g] << 16);
#define MOE_THIN_K(B) \
    if (2 * g + ((B) >> 3) < nch) acc = mfma_4_tokens<B>(xa, wf((B) < 8 ? w0 : w1, (B) & 7), acc);
            MOE_THIN_K(0) MOE_THIN_K(1) MOE_THIN_K(2) MOE_THIN_K(3) MOE_THIN_K(4) MOE_THIN_K(5) MOE_THIN_K(6) MOE_THIN_K(7)
            MOE_THIN_K(8) MOE_THIN_K(9) MOE_THIN_K(10) MOE_THIN_K(11) MOE_THIN_K(12) MOE_THIN_K(13) MOE_THIN_K(14) MOE_THIN_K(15)
#undef MOE_THIN_K
        }
    };

    int st = 0;
    load_x(0, 0);
    load_x(1, min(1, nstage - 1));
    dma_w(wb0, 0);
    dma_w(wb1, min(1, nstage - 1));
    for (; st + 6 <= nfull; st += 6) {
        stage(st, 0, wb0, wb2, 8);
        stage(st + 1, 1, wb1, wb0, 8);
        stage(st + 2, 0, wb2, wb1, 8);
        stage(st + 3, 1, wb0, wb2, 8);
        stage(st + 4, 0, wb1, wb0, 8);
        stage(st + 5, 1, wb2, wb1, 8);
    }
    // up to 5 whole stages and one of fewer than 64 k are left; stage st + i has the literals of i
    const int left = nfull - st;
    if (left > 0) stage(st, 0, wb0, wb2, 8);
    if (left > 1) stage(st + 1, 1, wb1, wb0, 8);
    if (left > 2) stage(st + 2, 0, wb2, wb1, 8);
    if (left > 3) stage(st + 3, 1, wb0, wb2, 8);
    if (left > 4) stage(st + 4, 0, wb1, wb0, 8);
    if (rem8) {
        if (left == 0) stage(st, 0, wb0, wb2, rem8);
        else if (left == 1) stage(st + 1, 1, wb1, wb0, rem8);
        else if (left == 2) stage(st + 2, 0, wb2, wb1, rem8);
        else if (left == 3) stage(st + 3, 1, wb0, wb2, rem8);
        else if (left == 4) stage(st + 4, 0, wb1, wb0, rem8);
        else stage(st + 5, 1, wb2, wb1, rem8);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // no DMA may land in LDS after the workgroup has gone

#pragma unroll
    for (int i = 0; i < 4; ++i) lg[i * EP + 64 * wave + lane] = acc[i];
    __syncthreads();
    for (int tb = wave; tb < BT; tb += WE) {
        if (t0 + tb >= n) break;
        const int t = t0 + tb;
        route_token<64, WE>(lg + tb * EP, bias, p, topk_idx + (size_t)t * p.top_k, topk_w + (size_t)t * p.top_k, nullptr, nullptr,
                            val + wave * EP, true);
    }
}


// Routes the tokens of a logits matrix in memory, a lane group per token (the group width follows from the expert count
// alone: it fixes the order of the softmax sum).  logits_bf16 (Mixtral): the rounded values are written back.
template <int GW, int EJ>
__device__ __forceinline__ void select_tokens(int tb, const float* bias, const moe_router_params& p, int32_t* topk_idx, float* topk_w,
                                              float* logits, uint16_t* logits_bf16, float* val) {
    const int lane = threadIdx.x & 63, t = tb + lane / GW;
    const bool live = t < p.n_tokens;
    const int tr = live ? t : p.n_tokens - 1;
    float* row = logits + (size_t)tr * p.n_experts;
    route_token<GW, EJ>(row, bias, p, topk_idx + (size_t)tr * p.top_k, topk_w + (size_t)tr * p.top_k,
                        p.logits_bf16 ? row : nullptr, logits_bf16 ? logits_bf16 + (size_t)tr * p.n_experts : nullptr,
                        val + lane / GW * (EJ * GW), live);
}

template <int GW, int EJ>
__global__ __launch_bounds__(256) void router_select_kernel(const float* __restrict__ bias, moe_router_params p,
                                                            int32_t* __restrict__ topk_idx, float* __restrict__ topk_w,
                                                            float* logits, uint16_t* logits_bf16) {
    const int wave = threadIdx.x >> 6;
    __shared__ float val[4][64 * EJ];
    const int tb = (blockIdx.x * 4 + wave) * (64 / GW);
    if (tb < p.n_tokens) select_tokens<GW, EJ>(tb, bias, p, topk_idx, topk_w, logits, logits_bf16, val[wave]);
}

// Selection and dispatch of a few tokens by one workgroup: its 16 waves route them, then it sorts the indices (5 tokens of
// 256 experts: 8.3 us; the two launches 5.8 + 4.8 and the gap between them).
template <int GW, int EJ>
__global__ __launch_bounds__(64 * SMALL_WAVES) void router_select_dispatch_kernel(const float* __restrict__ bias, moe_router_params p,
                                                                                  int32_t* topk_idx, float* topk_w, float* logits,
                                                                                  uint16_t* logits_bf16, DispatchOut out) {
    const int wave = threadIdx.x >> 6;
    __shared__ float val[SMALL_WAVES][64 * EJ];
    for (int tb = wave * (64 / GW); tb < p.n_tokens; tb += SMALL_WAVES * (64 / GW))
        select_tokens<GW, EJ>(tb, bias, p, topk_idx, topk_w, logits, logits_bf16, val[wave]);
    __threadfence_block();
    __syncthreads();                                            // the other waves' indices are in memory
    const volatile int32_t* idx = topk_idx;
    constexpr int IT = kSelectDispatchTokens * 16 / (SMALL_WAVES * 64);   // (top_k <= 16)
    dispatch_one_workgroup<IT>(p.n_tokens * p.top_k, p.n_experts, out, p.top_k, [&](int i) { return idx[i]; });
}

// The launch's workgroups for the shared expert, if there is one, follow the router's
SharedFirst behind(const SharedFirst* shared, int blocks) {
    SharedFirst s = shared ? *shared : SharedFirst{};
    s.first_block = blocks;
    return s;
}
int more_blocks(const SharedFirst* shared) { return shared ? shared_first_blocks(shared->inter) : 0; }

template <int WT, int WE, int TT, int TE, int S, int SHARED = 0>
void launch_logits(const void* x, const void* w, const moe_router_params& p, float* logits, const SharedFirst* shared, hipStream_t st) {
    constexpr int BT = 16 * TT * WT, BE = 16 * TE * WE;
    const int ntb = (p.n_tokens + BT - 1) / BT, neb = (p.n_experts + BE - 1) / BE, blocks = (ntb + 7) / 8 * 8 * neb;
    hipLaunchKernelGGL((router_logits_kernel<WT, WE, TT, TE, S, false, 64, 2, false, SHARED>), dim3(blocks + more_blocks(shared)),
                       dim3(64 * WT * WE), 0, st, (const uint16_t*)x, (const uint16_t*)w, nullptr, p, nullptr, nullptr, logits, nullptr,
                       DispatchOut{}, behind(shared, blocks));
}
template <int WE>
void launch_tokens(const void* x, const void* w, const float* bias, const moe_router_params& p, int32_t* idx, float* tw, hipStream_t st) {
    hipLaunchKernelGGL((router_tokens_kernel<WE>), dim3((p.n_tokens + 3) / 4), dim3(64 * WE), 0, st, (const uint16_t*)x, (const uint16_t*)w,
                       bias, p, idx, tw);
}
template <int WT, int WE, int TT, int S, int GW, int EJ>
void launch_fused(const void* x, const void* w, const float* bias, const moe_router_params& p, int32_t* idx, float* tw, hipStream_t st) {
    constexpr int BT = 16 * TT * WT;
    hipLaunchKernelGGL((router_logits_kernel<WT, WE, TT, TT, S, true, GW, EJ>), dim3((p.n_tokens + BT - 1) / BT), dim3(64 * WT * WE), 0, st,
                       (const uint16_t*)x, (const uint16_t*)w, bias, p, idx, tw, nullptr, nullptr, DispatchOut{}, SharedFirst{});
}

}  // namespace

// f(GW, EJ) with the lane-group width and the experts per lane that the expert count asks for
template <typename F>
static void for_expert_count(int E, F f) {
    using std::integral_constant;
    if (E <= 16) f(integral_constant<int, 16>{}, integral_constant<int, 1>{});
    else if (E <= 32) f(integral_constant<int, 32>{}, integral_constant<int, 1>{});
    else if (E <= 64) f(integral_constant<int, 64>{}, integral_constant<int, 1>{});
    else if (E <= 128) f(integral_constant<int, 64>{}, integral_constant<int, 2>{});
    else if (E <= 192) f(integral_constant<int, 64>{}, integral_constant<int, 3>{});
    else f(integral_constant<int, 64>{}, integral_constant<int, 4>{});
}

int router_select(const float* bias, const moe_router_params& p, int32_t* topk_idx, float* topk_w, float* logits,
                  uint16_t* logits_bf16, hipStream_t st) {
    for_expert_count(p.n_experts, [&](auto gw, auto ej) {
        constexpr int GW = decltype(gw)::value, EJ = decltype(ej)::value, per_block = 4 * (64 / GW);
        hipLaunchKernelGGL((router_select_kernel<GW, EJ>), dim3((p.n_tokens + per_block - 1) / per_block), dim3(256), 0, st, bias, p,
                           topk_idx, topk_w, logits, logits_bf16);
    });
    MOE_HIP_CHECK(hipGetLastError());
    return MOE_OK;
}

int router_select_dispatch(const float* bias, const moe_router_params& p, int32_t* topk_idx, float* topk_w, float* logits,
                           uint16_t* logits_bf16, const DispatchOut& out, hipStream_t st) {
    for_expert_count(p.n_experts, [&](auto gw, auto ej) {
        constexpr int GW = decltype(gw)::value, EJ = decltype(ej)::value;
        hipLaunchKernelGGL((router_select_dispatch_kernel<GW, EJ>), dim3(1), dim3(64 * SMALL_WAVES), 0, st, bias, p, topk_idx, topk_w,
                           logits, logits_bf16, out);
    });
    MOE_HIP_CHECK(hipGetLastError());
    return MOE_OK;
}

int router_dispatch(const void* x, const void* w_gate, const float* bias, const moe_router_params& p, int32_t* topk_idx, float* topk_w,
                    uint16_t* logits_bf16, const DispatchOut& out, hipStream_t st) {
    static_assert(router_dispatch_tokens(1) * 16 <= 256, "one pass of 4 waves over the indices");
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(1), dim3(256), 0, st, (const uint16_t*)x, (const uint16_t*)w_gate, bias, p, topk_idx, topk_w, nullptr,
                           logits_bf16, out, SharedFirst{});
    };
    if (p.n_experts <= 16) launch(router_logits_kernel<4, 1, 1, 1, 6, true, 16, 1, true>);
    else launch(router_logits_kernel<1, 4, 1, 1, 6, true, 32, 1, true>);
    MOE_HIP_CHECK(hipGetLastError());
    return MOE_OK;
}

int router_logits(const void* x, const void* w_gate, const moe_router_params& p, float* logits, const SharedFirst* shared, hipStream_t st) {
    const int E = p.n_experts, n = p.n_tokens;
    // One tile per wave up to 4096 tokens of 256 experts: the matrix cores of all CUs are then busy for less than about
    // four rounds of it, and smaller workgroups leave less of the last round idle; and where the last block of 64 experts
    // would be half empty (160 experts: 32-expert blocks fit).  Beyond, 2 x 2 tiles per wave, in workgroups of 8 waves
    // where 128-expert blocks fit and there is one for every CU.  Measured, logits alone (us, h = 7168):
    //   256 experts  1024 tokens: one tile 33;  3000: 86;  4096: 121, 2 x 2 in 4 waves 110, in 8 waves 208
    //                8192: 2 x 2 in 4 waves 215, in 8 waves 211;  65536: one tile 1890, 1690, 1645
    //   160 experts  16384 tokens: one tile 264, 2 x 2 with 32-expert blocks 301
    //   8 experts    16384 tokens (h = 6144): 4 waves along the tokens 35, 2 waves 38
    const int64_t work = (int64_t)n * E;
    if (E <= 16) launch_logits<4, 1, 1, 1, 4>(x, w_gate, p, logits, nullptr, st);
    else if (shared && shared->fp8) launch_logits<2, 2, 1, 1, 4, 2>(x, w_gate, p, logits, shared, st);
    else if (shared) launch_logits<2, 2, 1, 1, 4, 1>(x, w_gate, p, logits, shared, st);
    else if (work < (1 << 20) || (E % 64 != 0 && E % 64 <= 32)) launch_logits<2, 2, 1, 1, 4>(x, w_gate, p, logits, nullptr, st);
    else if (work < (1 << 21) || (E % 128 != 0 && E % 128 <= 64)) launch_logits<2, 2, 2, 2, 4>(x, w_gate, p, logits, nullptr, st);
    else launch_logits<2, 4, 2, 2, 3>(x, w_gate, p, logits, nullptr, st);
    MOE_HIP_CHECK(hipGetLastError());
    return MOE_OK;
}

}  // namespace moe

namespace moe {
namespace {
int route(const void* x, const void* w_gate, const float* bias, const moe_router_params* params, int32_t* topk_idx,
          float* topk_w, float* logits_out, void* stream);
}
}  // namespace moe

extern "C" int moe_router(const void* x, const void* w_gate, const float* bias, const moe_router_params* params,
                          int32_t* topk_idx, float* topk_w, float* logits_out, void* stream) {
    return moe::route(x, w_gate, bias, params, topk_idx, topk_w, logits_out, stream);
}

extern "C" int moe_router_rmsnorm(const void* x, const void* norm_weight, float eps, const void* w_gate,
                                  const float* bias, const moe_router_params* params, void* x_norm,
                                  int32_t* topk_idx, float* topk_w, float* logits_out, void* stream) {
    using namespace moe;
    if (params != nullptr && params->n_tokens == 0) return MOE_OK;
    MOE_REQUIRE(norm_weight && x_norm, "moe_router_rmsnorm: NULL norm weight or output");
    MOE_REQUIRE(x_norm != x, "moe_router_rmsnorm: x_norm must not alias x (rows are read twice)");
    MOE_REQUIRE(eps >= 0.0f, "moe_router_rmsnorm: eps %g < 0", (double)eps);
    int rc = check_router(x, w_gate, params, topk_idx, topk_w);       // (a refused call leaves x_norm as it was)
    if (rc != MOE_OK) return rc;
    // The norm as a kernel of its own: the logit engine takes its operands by DMA and has no place to normalise them.
    rc = moe_rmsnorm(x, norm_weight, eps, params->n_tokens, params->hidden, x_norm, stream);
    if (rc != MOE_OK) return rc;
    return route(x_norm, w_gate, bias, params, topk_idx, topk_w, logits_out, stream);
}

namespace moe {
int check_router(const void* x, const void* w_gate, const moe_router_params* params, const int32_t* topk_idx, const float* topk_w) {
    MOE_REQUIRE(params != nullptr, "moe_router: params is NULL");
    const moe_router_params& p = *params;
    MOE_REQUIRE(p.n_tokens >= 0, "moe_router: n_tokens %d < 0", p.n_tokens);
    if (p.n_tokens == 0) return MOE_OK;
    MOE_REQUIRE(x && w_gate && topk_idx && topk_w, "moe_router: NULL tensor pointer");
    MOE_REQUIRE(p.hidden > 0 && p.hidden % 8 == 0, "moe_router: hidden %d must be a positive multiple of 8", p.hidden);
    MOE_REQUIRE(p.n_experts >= 1 && p.n_experts <= 256, "moe_router: n_experts %d outside [1,256]", p.n_experts);
    MOE_REQUIRE(p.top_k >= 1 && p.top_k <= 16 && p.top_k <= p.n_experts, "moe_router: top_k %d outside [1,min(16,E)]",
                p.top_k);
    MOE_REQUIRE(p.scoring == MOE_SCORE_SOFTMAX || p.scoring == MOE_SCORE_SIGMOID,
                "moe_router: insupportable scoring function %d", p.scoring);
    MOE_REQUIRE(p.method >= MOE_TOPK_GREEDY && p.method <= MOE_TOPK_NOAUX_TC, "moe_router: insupportable TopK method %d",
                p.method);
    MOE_REQUIRE(p.scale_mode >= MOE_SCALE_NEVER && p.scale_mode <= MOE_SCALE_ALWAYS, "moe_router: bad scale_mode %d",
                p.scale_mode);
    if (p.method != MOE_TOPK_GREEDY) {
        MOE_REQUIRE(p.n_group >= 1 && p.n_group <= 32 && p.n_experts % p.n_group == 0,
                    "moe_router: n_group %d must divide n_experts %d and be <= 32", p.n_group, p.n_experts);
        MOE_REQUIRE(p.topk_group >= 1 && p.topk_group <= p.n_group, "moe_router: topk_group %d outside [1,n_group]",
                    p.topk_group);
        MOE_REQUIRE(p.method != MOE_TOPK_NOAUX_TC || p.n_experts / p.n_group >= 2,
                    "moe_router: noaux_tc needs at least 2 experts per group");
    }
    MOE_REQUIRE(p.hidden < 1 << 22, "moe_router: hidden %d: 256 rows have to lie within 2 GiB", p.hidden);
    return MOE_OK;
}
}  // namespace moe

namespace moe {
namespace {
int route(const void* x, const void* w_gate, const float* bias, const moe_router_params* params, int32_t* topk_idx,
          float* topk_w, float* logits_out, void* stream) {
    const int ok = check_router(x, w_gate, params, topk_idx, topk_w);
    if (ok != MOE_OK || params->n_tokens == 0) return ok;
    const moe_router_params& p = *params;
    hipStream_t st = as_stream(stream);
    const int E = p.n_experts;
    if (logits_out == nullptr) {
        // 4 tokens per workgroup while 16 leave most CUs without any, where that beats three or four expert blocks one
        // after the other; a ring of 4 stages while every CU has one block of 16 tokens; then two workgroups per CU, so that
        // one selects while the other multiplies; and 2 x 2 tiles per wave where 128-expert blocks fit and there are many
        // rounds.  Measured (us, h = 7168 / 5120 / 4096 / 2048 for 256 / 160 / 128 / 64 experts; the engines that took
        // one k per instruction -> this):
        //   64 tokens     256 experts 94 -> 84 (16 tokens per workgroup 143), 160: 77 -> 64 (81), 128: 57 -> 48
        //   4096          235 -> 145, 136 -> 81, 76 -> 49, 41 -> 19      8192: ring of 4 288, of 3 267
        //   16384         635 -> 530, 427 -> 287, 248 -> 167, 82 -> 54
        //   65536         2127 -> 2106 (one tile per wave 2161), 1174 -> 1172, 678 -> 682, 260 -> 214
        for_expert_count(E, [&](auto gw, auto ej) {
            constexpr int GW = decltype(gw)::value, EJ = decltype(ej)::value;
            const int n = p.n_tokens;
            if constexpr (GW == 16) {
                launch_fused<2, 1, 1, 4, GW, EJ>(x, w_gate, bias, p, topk_idx, topk_w, st);
            } else {
                if constexpr (EJ > 2)
                    if (n <= 1024) return launch_tokens<EJ>(x, w_gate, bias, p, topk_idx, topk_w, st);
                if constexpr (EJ % 2 == 0)
                    if (n > 32768) return launch_fused<1, 4, 2, 3, GW, EJ>(x, w_gate, bias, p, topk_idx, topk_w, st);
                if (n <= 4096) launch_fused<1, 4, 1, 4, GW, EJ>(x, w_gate, bias, p, topk_idx, topk_w, st);
                else launch_fused<1, 4, 1, 3, GW, EJ>(x, w_gate, bias, p, topk_idx, topk_w, st);
            }
        });
        MOE_HIP_CHECK(hipGetLastError());
        return MOE_OK;
    }
    const int rc = router_logits(x, w_gate, p, logits_out, nullptr, st);
    return rc != MOE_OK ? rc : router_select(bias, p, topk_idx, topk_w, logits_out, nullptr, st);
}
}  // namespace
}  // namespace moe
