// The weighted sum of a token's expert outputs, 8 columns (16 bytes) of a row at a time: shared by the combine kernel and by the
// down projection of a few tokens, which combines what it has just written.
#pragma once
#include "common.h"

namespace moe {

constexpr int kCombineMaxK = 16;

// adds a source row in its place of the summation order
template <int MODE>
__device__ __forceinline__ void combine_add(float (&acc)[8], const u32x4& v, float w) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float lo = __uint_as_float(v[i] << 16), hi = __uint_as_float(v[i] & 0xffff0000u);
        if (MODE == MOE_COMBINE_F32) {
            acc[2 * i] = acc[2 * i] + lo * w;
            acc[2 * i + 1] = acc[2 * i + 1] + hi * w;
        } else {
            acc[2 * i] = acc[2 * i] + round_to_bf16(lo * w);
            acc[2 * i + 1] = acc[2 * i + 1] + round_to_bf16(hi * w);
            if (MODE == MOE_COMBINE_BF16_SEQ) {
                acc[2 * i] = round_to_bf16(acc[2 * i]);
                acc[2 * i + 1] = round_to_bf16(acc[2 * i + 1]);
            }
        }
    }
}

// the sum rounded, then bf16 + bf16 -> bf16 with the shared expert's row and with the residual, as torch adds two bf16 tensors
__device__ __forceinline__ u32x4 combine_finish(const float (&acc)[8], bool has_shared, const u32x4& sh, bool has_residual, const u32x4& res) {
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t lo = f32_to_bf16_bits(acc[2 * i]), hi = f32_to_bf16_bits(acc[2 * i + 1]);
        if (has_shared) {
            lo = f32_to_bf16_bits(bf16_bits_to_f32(lo) + __uint_as_float(sh[i] << 16));
            hi = f32_to_bf16_bits(bf16_bits_to_f32(hi) + __uint_as_float(sh[i] & 0xffff0000u));
        }
        if (has_residual) {
            lo = f32_to_bf16_bits(__uint_as_float(res[i] << 16) + bf16_bits_to_f32(lo));
            hi = f32_to_bf16_bits(__uint_as_float(res[i] & 0xffff0000u) + bf16_bits_to_f32(hi));
        }
        o[i] = lo | (hi << 16);
    }
    return o;
}

// the weight of a slot as the mode multiplies it
template <int MODE>
__device__ __forceinline__ float combine_weight(float w) { return MODE == MOE_COMBINE_F32 ? w : round_to_bf16(w); }

}  // namespace moe
