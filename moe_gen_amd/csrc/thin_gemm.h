// One wave's share of a product with few token rows: the body of the thin kernel (grouped_gemm.hip), which the router's launch also
// runs for the shared expert's gate and up projection; and the pieces it shares with the other GEMM bodies.
#pragma once
#include "common.h"

namespace moe {
namespace {

// LDS rows are 128 bytes = 8 chunks of 16 bytes; chunk c of row r is stored at chunk c ^ swz(r).
// swz makes any 8 consecutive rows hit 8 different chunks (32 banks x 4 B = one 128-byte row per
// cycle) AND any 16 consecutive rows hit 16 different (row parity, chunk) slots (64 banks =
// two rows per cycle), so 16-byte operand reads by 32 consecutive rows never collide.
__device__ __forceinline__ int swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }

// global-address-space views: expert pointers come out of a pointer table in memory, and
// without the address space the compiler must emit flat loads, whose completion is tracked
// by the same counter as the LDS reads of the MFMA operands
typedef const __attribute__((address_space(1))) u32x4* gptr_u32x4;
typedef const __attribute__((address_space(1))) float* gptr_f32;
typedef const __attribute__((address_space(1))) int32_t* gptr_i32;
typedef __attribute__((address_space(3))) uint8_t* lds_u8;

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ const uint8_t* uni_ptr(const void* p) {
    uint64_t u = (uint64_t)(uintptr_t)p;
    uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u), hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
    return reinterpret_cast<const uint8_t*>((uintptr_t)(((uint64_t)hi << 32) | lo));
}

__device__ __forceinline__ float bf16r(float a) { return __uint_as_float(pack_bf16(a, 0.0f) << 16); }

// 8 fp8 weights (two dwords) -> 8 bf16: bf16(f32(q) * s), the reference's dequantisation
__device__ __forceinline__ u32x4 dequant8(uint32_t q0, uint32_t q1, float sc) {
    const f32x2 c0 = __builtin_amdgcn_cvt_pk_f32_fp8(q0, false), c1 = __builtin_amdgcn_cvt_pk_f32_fp8(q0, true);
    const f32x2 c2 = __builtin_amdgcn_cvt_pk_f32_fp8(q1, false), c3 = __builtin_amdgcn_cvt_pk_f32_fp8(q1, true);
    return u32x4{pack_bf16(c0[0] * sc, c0[1] * sc), pack_bf16(c1[0] * sc, c1[1] * sc),
                 pack_bf16(c2[0] * sc, c2[1] * sc), pack_bf16(c3[0] * sc, c3[1] * sc)};
}

// Epilogue values of one lane for one pair of accumulators: 4 consecutive output columns of one row.
// SWIGLU: act = bf16(bf16(silu(bf16(g))) * bf16(u)), the rounding points of the reference's bf16
// Linear / SiLU / mul modules (silu through the hardware exp and reciprocal); else bf16(acc).
template <bool SWIGLU>
__device__ __forceinline__ u32x2 epilogue_pack(const f32x4& a, const f32x4& up) {
    if (SWIGLU) {
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float gv = bf16r(a[i]);
            const float uv = bf16r(up[i]);
            const float sg = bf16r(gv * __builtin_amdgcn_rcpf(1.0f + __expf(-gv)));
            o[i] = sg * uv;
        }
        return u32x2{pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3])};
    }
    return u32x2{pack_bf16(a[0], a[1]), pack_bf16(a[2], a[3])};
}

// LDS keys of the fp8 forms that read 16 weights of a row at once (stream8_tile): part c of weight row r at c ^ wsw(r), chunk c of a
// 128-k token row at c ^ tsw(r)
__device__ __forceinline__ int wsw(int r) { return ((r >> 1) & 1) | (((r >> 2) & 1) << 2); }
__device__ __forceinline__ int tsw(int r) { return (r & 3) | ((r & 4) << 1); }

// The expert that a wave works on: its matrices and scales, the rows of the call (row_map: gathered from `a`) and the output
struct ThinUnit {
    const void *b0, *b1;         // gate and up, or down
    const float *s0, *s1;        // fp8: their block scales
    const uint16_t* a;
    const int32_t* row_map;
    size_t a_bytes;
    int a_rows;
    uint16_t* c;
    int K, N, row0, row_end;
};

// 8 bytes past the L2 of an XCD (a relaxed atomic at agent scope), for a wave on another one
__device__ __forceinline__ void store_shared_8(uint16_t* p, const u32x2& v) {
    __hip_atomic_store(reinterpret_cast<uint64_t*>(p), __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Bytes of LDS of a stage
template <bool W8, int NF>
constexpr int thin_stage_bytes = NF * 2048 + (W8 ? 4096 : 2048);

// Columns n0 .. of the unit by one wave; lds: NB stages of its own.  NF: 16-row fragments of weights (gate and up: one of either).
// AGENT: the outputs are read in the same launch.
template <bool SWIGLU, bool W8, int NF, bool AGENT, int NB>
__device__ __forceinline__ void thin_columns(const ThinUnit& u, int n0, uint8_t* lds) {
    static_assert(!SWIGLU || NF == 2, "gate and up: a fragment of either");
    constexpr int WBYTES = NF * 2048, TBYTES = W8 ? 4096 : 2048;       // weights and 16 token rows of a stage
    constexpr int NDW = 2 * NF, NDT = TBYTES / 1024, NI = NDW + NDT;   // DMA instructions per stage
    constexpr int SB = thin_stage_bytes<W8, NF>;
    static_assert(NB >= 3 && (NB - 1) * NI < 64, "stages");
    const int lane = threadIdx.x & 63, K = u.K, N = u.N, row0 = u.row0, row_end = u.row_end;
    const int nk = K / (W8 ? 128 : 64);
    const int rot = (n0 / (SWIGLU ? 128 : 256)) % nk;      // the k rotation of the N tile these columns belong to
    auto stage_at = [&](int k) { const int s = min(k, nk - 1) + rot; return s >= nk ? s - nk : s; };

    const uint8_t* bm0 = uni_ptr(u.b0);
    const uint8_t* bm1 = SWIGLU ? uni_ptr(u.b1) : bm0;
    gptr_f32 sc0 = nullptr, sc1 = nullptr;                 // scales of the 128 rows the wave's columns lie in
    if (W8) {
        sc0 = (gptr_f32)(uintptr_t)uni_ptr(u.s0) + (n0 >> 7) * nk;
        sc1 = SWIGLU ? (gptr_f32)(uintptr_t)uni_ptr(u.s1) + (n0 >> 7) * nk : sc0;
    }
    // DMA: weights, instruction i: fragment i / 2 (gate / up, or the two halves of the 32 down rows), rows 8 (i & 1) +
    // lane / 8; tokens, instruction i: 8 (fp8: 4) rows; chunks swizzled as in the streamers
    const int lr = lane >> 3, pp = lane & 7;
    const uint32_t row_bytes = (uint32_t)K * (W8 ? 1 : 2);
    uint32_t w_voff[4], t_voff[4];                         // (NDW and NDT are used)
#pragma unroll
    for (int i = 0; i < NDW; ++i) {
        const int fr = 8 * (i & 1) + lr;
        w_voff[i] = (uint32_t)min(n0 + (SWIGLU ? 0 : 16 * (i >> 1)) + fr, N - 1) * row_bytes + (uint32_t)((pp ^ (W8 ? wsw(fr) : swz(fr))) << 4);
    }
    const int frow = lane & 15, q = lane >> 4;
    const int fq = ((q & 1) << 1) | (q >> 1);
    const uint32_t w_rd = (uint32_t)(frow * 128), wkey = (uint32_t)(W8 ? wsw(frow) : swz(frow));
    const uint32_t t_rd = (uint32_t)WBYTES + (uint32_t)(frow * (W8 ? 256 : 128)), tkey = (uint32_t)(W8 ? tsw(frow) : swz(frow));

    for (int r0 = row0; r0 < row_end; r0 += 16) {          // (more than once only if a caller's row bound was wrong)
        const uint8_t* a_base = reinterpret_cast<const uint8_t*>(u.a) + (u.row_map ? (size_t)0 : (size_t)r0 * K * 2);
        const int a_records = u.row_map ? (int)(uint32_t)u.a_bytes : min(16, row_end - r0) * K * 2;
#pragma unroll
        for (int i = 0; i < NDT; ++i) {
            const int tr = W8 ? 4 * i + (lane >> 4) : 8 * i + lr;
            const int r = min(r0 + tr, row_end - 1);
            const int src = u.row_map ? ((gptr_i32)(uintptr_t)u.row_map)[r] : r - r0;
            t_voff[i] = (uint32_t)src * (uint32_t)(K * 2) + (uint32_t)((W8 ? (lane & 15) ^ tsw(tr) : pp ^ swz(tr)) << 4);
            if (r0 + tr >= row_end || (u.row_map && (unsigned)src >= (unsigned)u.a_rows)) t_voff[i] = 0xfffffff0u;
        }
        auto dma = [&](int k, int buf) __attribute__((always_inline)) {
            const int live = uni(k < nk ? -1 : 0);         // past the end: empty descriptors, the instructions still count
            uint8_t* d = lds + buf * SB;
            const uint32_t so = (uint32_t)stage_at(k) * 128u;
            const __amdgpu_buffer_rsrc_t r0d = __builtin_amdgcn_make_buffer_rsrc((void*)bm0, 0, live, 0x00020000);
            const __amdgpu_buffer_rsrc_t r1d = __builtin_amdgcn_make_buffer_rsrc((void*)bm1, 0, live, 0x00020000);
            const __amdgpu_buffer_rsrc_t rad = __builtin_amdgcn_make_buffer_rsrc((void*)a_base, 0, live & a_records, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r0d, (lds_u8)d, 16, w_voff[0], so, 0, 2);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r0d, (lds_u8)(d + 1024), 16, w_voff[1], so, 0, 2);
            if constexpr (NF == 2) {
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r1d, (lds_u8)(d + 2048), 16, w_voff[2], so, 0, 2);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r1d, (lds_u8)(d + 3072), 16, w_voff[3], so, 0, 2);
            }
#pragma unroll
            for (int i = 0; i < NDT; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rad, (lds_u8)(d + WBYTES + i * 1024), 16, t_voff[i], W8 ? 2 * so : so, 0, 0);
        };
        f32x4 acc[NF];
#pragma unroll
        for (int j = 0; j < NF; ++j) acc[j] = f32x4{0};
        float v0 = 0.0f, v1 = 0.0f;                        // fp8: lane l holds the scales of stage 64 i + l
        if (W8) { v0 = sc0[stage_at(lane)]; v1 = sc1[stage_at(lane)]; }
        for (int i = 0; i < NB - 1; ++i) dma(i, i);
        // (waits by hand: the compiler's own, in front of the readlane below, would cover the DMA of the next stage too.  The
        // scales were requested before the DMA; where the compiler moves them behind some of it, it waits for them here itself)
        if (W8) asm volatile("s_waitcnt vmcnt(%2)" : "+v"(v0), "+v"(v1) : "n"((NB - 1) * NI));
        int buf = 0;
        for (int k = 0; k < nk; ++k) {
            // this wave's DMA of stage k has landed and its reads of stage k - 1, whose buffer is refilled, have returned
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((NB - 2) * NI) : "memory");
            if (W8 && (k & 63) == 0 && k > 0) {
                v0 = sc0[stage_at(k + lane)];
                v1 = sc1[stage_at(k + lane)];
                asm volatile("s_waitcnt vmcnt(0)" : "+v"(v0), "+v"(v1));
            }
            dma(k + NB - 1, buf == 0 ? NB - 1 : buf - 1);
            const uint8_t* b = lds + buf * SB;
            if (W8) {
                const float c[2] = {__builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v0), k & 63)),
                                    __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v1), k & 63))};
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    u32x4 raw[NF];
#pragma unroll
                    for (int j = 0; j < NF; ++j) raw[j] = *reinterpret_cast<const u32x4*>(b + j * 2048 + w_rd + (((4 * h + fq) ^ wkey) << 4));
#pragma unroll
                    for (int s2 = 0; s2 < 2; ++s2) {
                        const bf16x8 tf = *reinterpret_cast<const bf16x8*>(b + t_rd + (((8 * h + 2 * fq + s2) ^ tkey) << 4));
#pragma unroll
                        for (int j = 0; j < NF; ++j)
                            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                __builtin_bit_cast(bf16x8, dequant8(raw[j][2 * s2], raw[j][2 * s2 + 1], c[j])), tf, acc[j], 0, 0, 0);
                    }
                }
            } else {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const uint32_t coff = (uint32_t)((4 * s + fq) ^ wkey) << 4;      // (wkey == tkey)
                    const bf16x8 tf = *reinterpret_cast<const bf16x8*>(b + t_rd + coff);
#pragma unroll
                    for (int j = 0; j < NF; ++j)
                        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(b + j * 2048 + w_rd + coff), tf, acc[j], 0, 0, 0);
                }
            }
            buf = buf + 1 == NB ? 0 : buf + 1;
        }
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // no DMA may land in LDS after the workgroup has gone
        const int r = r0 + frow;
        if (r < row_end) {
#pragma unroll
            for (int j = 0; j < (SWIGLU ? 1 : NF); ++j) {
                const int col = n0 + 16 * j + 4 * q;
                if (col >= N) continue;
                const u32x2 o = epilogue_pack<SWIGLU>(acc[j], acc[SWIGLU ? 1 : j]);
                if constexpr (AGENT) store_shared_8(u.c + (size_t)r * N + col, o);
                else *reinterpret_cast<u32x2*>(u.c + (size_t)r * N + col) = o;
            }
        }
    }
}

}  // namespace
}  // namespace moe
