// Grouped SwiGLU expert GEMMs for gfx950 on bf16 MFMA, with a W8A16 variant that
// dequantises fp8-e4m3fn weights (one fp32 scale per 128x128 block) in registers on the
// way from HBM to LDS.
//
// Replaces the expert loop of moe_infer (modeling_deepseek_v3.py:675-691), the body of
// Expert_Wrapper.forward (Wrapper.py:470-530: fetch, dequantise, run the MLP in chunks,
// synchronise) and DeepseekV3MLP.forward (:463-467) for all experts with two launches:
//   launch 1 (SWIGLU): act = bf16( bf16(silu(bf16(X Wg^T))) * bf16(X Wu^T) )
//   launch 2         : Y   = bf16( act Wd^T )
// Rounding points are those of the reference's bf16 nn.Linear / SiLU / mul modules; the
// dequantisation is deepseek_v3_dequantization (Wrapper.py:109-138) element for element:
// w = bf16(f32(q) * scale[i/128, j/128]).
//
// Work decomposition.  Sorted rows of expert e are [offsets[e], offsets[e+1]).  Each
// expert is cut into M tiles (the last one partial); an M tile times an N tile of the
// weight matrix is one unit of work.  Every workgroup rebuilds the (tiny) M-tile prefix
// over experts in LDS from offsets[], so a launch needs neither a host sync nor a tile table.
// Two kinds of tiles; which kind an expert's rows are follows its own count, which every workgroup reads from offsets[]
// (both_kernels, launch_mt):
//  * persistent tiles (persistent_body): experts above one small tile, with fp8 weights the full 256-row tiles of every expert.  256
//    rows, one workgroup per CU; groups of 32 consecutive tiles go round-robin to the XCDs (workgroup ids are dealt to the 8 XCDs
//    one by one by the hardware; the tiles of a group share their A and B panels through that XCD's L2), and a workgroup's k
//    pipeline runs on from one of its tiles into the next.
//  * tiles of one workgroup each: experts of up to 192 rows, and with fp8 weights what an expert's full 256-row tiles leave over if that
//    is at most 192 rows, a single MLP's where a padded persistent tile is not the shorter way; work that mostly streams weights.  The
//    grid is an upper bound on the tile count, surplus workgroups exit at once; the tile height (16 ... 192 rows in steps of 16)
//    follows the expert.  They run through the weight streamers (stream16_tile, stream8x_tile, stream8_tile): weights AND token
//    rows reach LDS by DMA, three weight buffers, one barrier per stage.
// Kernels: grouped_gemm_both_kernel has both kinds in one launch, the persistent workgroups first (calls of many rows per
// expert: both_kinds); grouped_gemm_kernel one-workgroup tiles alone (fewer rows, and what the persistent body cannot address);
// grouped_gemm_half_kernel halves of those (bf16 down projections of few tiles); grouped_gemm_thin_kernel waves of 16 columns (up to
// 16 rows per expert); gate_up_few_rows_kernel a tile per CU of one wide fp8 MLP; the split kernels slices of k of one.
//
// Workgroup = 8 waves, two per SIMD.  v_mfma_f32_16x16x32_bf16 throughout: on real (non-zero) data this
// chip is power-limited under MFMA load; the 16x16x32 shape moves a third less accumulator data per flop
// than 32x32x16 and sustains ~13 % more (1.95 vs 1.73 PFLOP/s in a registers-only loop with random
// operands), which is worth ~6 % here.  The persistent body's waves are 2 along M x 4 along N, 8 x 4 MFMA
// tiles each (128x64 outputs, 128 fp32 accumulators).  K advances 64 at a time through two LDS stages; rows
// are 128 bytes with a 16-byte-chunk XOR swizzle so that both the 16-byte stores and the 16-byte MFMA
// operand reads are bank-conflict free.  Token rows and bf16 weights come into LDS by DMA
// (buffer_load ... lds); fp8 weights of the persistent body go through registers, converted on the way,
// two k-stages ahead, every wave interleaving its share of that with its MFMAs, one piece per group of
// MFMAs, between the two barriers per k-stage.  gemm_tile, the register-staged body of one-workgroup tiles,
// remains for calls that gather from 4 GiB of rows or more (the DMA paths address them with 32 bits).
//
// The MFMA is issued with the WEIGHT fragment as srcA and the TOKEN fragment as srcB, so
// a lane ends up holding 4 consecutive output columns of one token row per accumulator;
// the epilogues put them together, between lanes or through LDS, into 16-byte stores of row segments.

#include <cmath>
#include <type_traits>

#include "combine_math.h"
#include "common.h"
#include "dispatch_small.h"
#include "layer.h"
#include "thin_gemm.h"

namespace moe {
namespace {

constexpr int BK = 64;           // k per stage (bf16 elements); 128 bytes per LDS row
constexpr int ROW_B = 128;       // bytes per LDS row
constexpr int BN_ROWS = 256;     // weight rows per workgroup (128 gate + 128 up when SWIGLU)
constexpr int MAX_E = 1024;
constexpr int PAIR_LO = 257, PAIR_HI = 384;   // bf16: rows of an expert that runs as two tiles of the 192-row body

// 16 fp8 bytes -> 16 bf16 (two 16-byte chunks): bf16(f32(q) * s)
__device__ __forceinline__ void dequant16(u32x4 q, float s, u32x4& lo, u32x4& hi) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f32x2 a = __builtin_amdgcn_cvt_pk_f32_fp8(q[i], false);
        f32x2 b = __builtin_amdgcn_cvt_pk_f32_fp8(q[i], true);
        uint32_t p0 = pack_bf16(a[0] * s, a[1] * s), p1 = pack_bf16(b[0] * s, b[1] * s);
        if (i < 2) { lo[2 * i] = p0; lo[2 * i + 1] = p1; }
        else       { hi[2 * (i - 2)] = p0; hi[2 * (i - 2) + 1] = p1; }
    }
}

struct GemmArgs {
    const uint16_t* a;          // activations, row stride K
    const int32_t* row_map;     // optional: sorted row -> row of a
    size_t a_bytes;             // size of a when rows are gathered through row_map
    int a_rows;                 // rows of a when rows are gathered through row_map
    const void* const* b0;      // per-expert weight matrix [N, K] (gate when SWIGLU, else down)
    const void* const* b1;      // per-expert up matrix [N, K] (SWIGLU only)
    const float* const* s0;     // per-expert block scales of b0 (W8 only)
    const float* const* s1;     // per-expert block scales of b1 (W8, SWIGLU only)
    const int32_t* offsets;     // [E+1]
    uint16_t* c;                // output, row stride N, sorted-row order
    int E, K, N;
    int n_tiles_n;              // ceil(N / (SWIGLU ? 128 : 256))
    // a call of both kinds of tiles (grouped_gemm_both_kernel):
    int cold_max;               // experts of up to this many rows are tiles of one workgroup each, the others tiles of the
                                // persistent workgroups (0: all are)
    int rem_split;              // 1: the rule applies to what an expert's full 256-row tiles leave over (count % 256)
                                // instead of to its count: the full tiles are persistent ones, and so is the
                                // last, ragged one if it holds more than cold_max rows
    int pair_rows;              // 1: experts of PAIR_LO .. PAIR_HI rows are tiles of one workgroup each too
    int alone;                  // 1 (fp8): no persistent tile's sums have to be matched: k_rotation, and the stage order of
                                // stream8_tile for tiles of up to 64 rows
    int tail_cus;               // > 0: the persistent workgroups run whole rounds of this many tiles (one per CU); what
                                // is left goes to workgroups of one piece of a tile each if that pays (tail_of)
    int cut_cus;                // > 0 (bf16, tiles of one workgroup alone): the CUs, see cut_prefix_scan
};

// What a launch works on: the routed experts and a second problem of one expert with matrices, sizes and buffers of its own,
// the layer's shared expert.  A launch pair for the shared expert alone has a tile for a fraction of the CUs at small batches
// (DeepSeek-V2-236B, 64 tokens: 24 and 20 tiles, 70 + 44 us for 94 MB) and rounds of its own that end part-filled at larger ones.
// The host knows a bound of its rows, the kernels its rows (offsets[], like every expert's):
//  * a call of one kind of tiles: `shared_tiles` workgroups in front of the routed experts' are the shared expert's; those past
//    its rows return at once.
//  * a call of both: `shared_rows` > 0 bounds its rows, and its tiles are counted as any expert's (persistent ones in front of the
//    routed experts'; one-workgroup tiles behind them, in front of the pieces of last tiles).
struct GemmPair {
    GemmArgs p[2];              // routed, shared
    int shared_tiles, shared_rows;
    int32_t* claims;            // kClaimInts zeros, or NULL (see Claims)
};

// Stage at which a tile of N tile n_tile starts its walk over k.  Workgroups that run side by side mostly differ in
// their N tile; started at the same stage, their requests in flight would share the low address bits (rows of the weight
// matrices are K elements apart) and crowd the same memory channels: with the start spread over the stages a launch
// that streams weights gains about a tenth (Mixtral-8x22B shapes, 8 experts x 16 ... 120 rows: 6.1 -> 6.8, 5.4 -> 6.1
// TB/s; 128 / 160 / 192 rows next to persistent tiles: gate/up 0.63 / 0.64 / 0.66 -> 0.55 / 0.58 / 0.62 ms).
// bf16 weights: every path uses this rule, so which kernel or tile computes a row does not change the order its products are
// added in (the persistent body itself runs within 0.5 % either way).  fp8 weights (a scale per 128 k: pairs of stages stay
// together): only in calls of one-workgroup tiles alone (and not for a large shared expert in them, joint_alone); the persistent
// body loses 1.6 % of the DeepSeek-V3 step to a rotated walk, so calls with persistent tiles start every tile at stage 0.
template <bool W8>
__device__ __forceinline__ int k_rotation(int n_tile, int nk) { return (W8 ? 2 * n_tile : n_tile) % nk; }

__device__ __forceinline__ u32x4 gload16(const void* p) { return *(gptr_u32x4)(uintptr_t)p; }
// Weights of one-workgroup tiles are streamed: a tile of them is used by one workgroup (two
// or more for an expert above 256 rows) and never again in the launch, so those loads are non-temporal
// (Mixtral-8x22B, 256 tokens: down projection 0.325 -> 0.302 ms).  In the persistent body the panels are
// shared through L2 and stay plain.
template <bool STREAM>
__device__ __forceinline__ u32x4 gload16_w(const void* p) {
    return STREAM ? __builtin_nontemporal_load((gptr_u32x4)(uintptr_t)p) : *(gptr_u32x4)(uintptr_t)p;
}


// A barrier behind this wave's LDS operations that leaves loads and stores to memory in flight
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// ---- which workgroup computes which tile of one workgroup ----
//
// Tiles are dealt to the XCDs in groups of 4 consecutive ones (the M tiles of one N tile first), round robin: those that read the
// same weights share them through one XCD's L2, and small groups keep the XCDs even whatever the number of tiles and however much
// one expert's tiles cost more than another's.  (Workgroup ids are dealt to the XCDs one by one by the hardware.)
__device__ __forceinline__ int dealt_tile(int xcd, int i) { return (((i >> 2) << 3) + xcd) * 4 + (i & 3); }
// The i-th tile of an XCD goes to the i-th workgroup of the XCD, in a grid that the host bounds without knowing the counts (OneTile);
// or, in calls of both kinds that bring counters (zeros: a layer call, whose dispatch sets them), to its i-th claim: a workgroup per
// CU, the persistent ones among them when they are done, claims tiles until none is left, and an XCD that is done goes on with
// the others'.  That spares a tile its launch and the scan over the experts, and the CUs the surplus workgroups of such a grid, which
// take 3 us each: DeepSeek-V2-236B, 4000 tokens, 4100 of them in the down projection, the layer 2165 -> 2108 us.  (Calls of tiles of one
// workgroup alone stay with the launches: with claims 1 % faster where many experts have no rows, DeepSeek-V2-236B 32 and 64 tokens,
// 2 to 3 % slower at few tiles a CU, DeepSeek-V2-Lite 32 ... 256 and DeepSeek-V3 1000.)
struct OneTile {
    __device__ __forceinline__ void ask() {}
};
struct Claims {
    int32_t* counters;           // one per XCD, kClaimStride apart; NULL: the workgroup has one tile
    int xcd, limit;              // the tiles are those below limit
    int next;                    // what ask() found (the first lane's)
    __device__ __forceinline__ int count(int from) const {
        return __hip_atomic_fetch_add(counters + from * kClaimStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // in front of a tile's epilogue: the answer takes about 2 us
    __device__ __forceinline__ void ask() {
        if (counters && threadIdx.x == 0) next = count(xcd);
    }
    // The workgroup's next tile, -1 if there is none.  All threads; told: LDS.  (Bare barriers: a fence would wait for the stores of
    // the epilogue.)
    __device__ __forceinline__ int take(int* told) const {
        if (!counters) return -1;
        int v = -1;
        if (threadIdx.x < 64) {
            const int lane = threadIdx.x;
            v = dealt_tile(xcd, uni(next));
            while (v >= limit) {
                v = -1;
                const int seen = lane < 8 ? __hip_atomic_load(counters + lane * kClaimStride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
                const uint64_t left = __ballot(lane < 8 && dealt_tile(lane, seen) < limit);
                if (left == 0) break;
                const int from = (int)__builtin_ctzll(left);
                int i = 0;
                if (lane == 0) i = count(from);
                v = dealt_tile(from, uni(i));
            }
        }
        lds_barrier();                           // every wave has left the tile before, and read its number
        if (threadIdx.x == 0) *told = v;
        lds_barrier();
        return uni(*told);
    }
};

// ---- pieces shared by one-workgroup tiles and the persistent body ----

// Position of the expert's `local`-th tile.  Inside an expert, tiles are visited in groups of about
// GM consecutive M tiles (the expert's M tiles split as evenly as possible); within a group the M
// tile varies fastest.  The ~32 workgroups an XCD runs at once then cover ~GM M tiles x 32/GM N
// tiles and share those panels through the XCD's L2: an A panel is fetched once per 32/GM N tiles
// and a B panel once per group.  GM = 4 (4 x 8 tiles) balances the two re-fetch factors; measured on
// 64 experts x 2048 rows (7168 -> 2048, fp8) it fetches 7.0 GiB against 8.75 GiB for GM = 8 or 16.
__device__ __forceinline__ void tile_in_expert(int local, int mt_e, int n_tiles_n, int& m_tile, int& n_tile) {
    constexpr int GM = 4;
    const int ng = max(1, (mt_e + GM / 2) / GM);
    const int base = mt_e / ng, extra = mt_e - base * ng;      // `extra` groups hold base+1 tiles
    const int big = (base + 1) * n_tiles_n, cut = extra * big;
    int gm, m0, rem;
    if (local < cut) {
        const int gi = local / big;
        rem = local - gi * big; gm = base + 1; m0 = gi * (base + 1);
    } else {
        const int l2 = local - cut, sz = base * n_tiles_n, gi = l2 / sz;
        rem = l2 - gi * sz; gm = base; m0 = extra * (base + 1) + gi * base;
    }
    n_tile = rem / gm;
    m_tile = m0 + (rem - n_tile * gm);
}

// A lane's 4 columns (8 bytes) of two neighbouring 16-column fragments of one row -> 16 consecutive bytes of that row: lane
// group q gets columns 8 (q / 2) .. + 7 of fragment q % 2, so the four groups write 64 consecutive bytes of a row.
__device__ __forceinline__ u32x4 pair_columns(u32x2 p0, u32x2 p1) {
    const auto lo = __builtin_amdgcn_permlane16_swap(p0[0], p1[0], false, false);   // odd groups of p0 <-> even groups of p1
    const auto hi = __builtin_amdgcn_permlane16_swap(p0[1], p1[1], false, false);
    return u32x4{lo[0], hi[0], lo[1], hi[1]};
}

// 16 bytes to base + offset; an offset of 2 GiB or more stores nothing, and the instruction still counts.  AUX 2: non-temporal
template <int AUX>
__device__ __forceinline__ void store16(u32x4 v, const uint8_t* base, uint32_t offset) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0x7fffffff, 0x00020000);
    __builtin_amdgcn_raw_buffer_store_b128(v, r, offset, 0, AUX);
}

// Exclusive scan of the experts' M-tile counts, tiles_of(count), by the whole workgroup: s_pref[e] = number of
// M tiles in front of expert e (the caller adds s_pref[E] if it needs it).  Returns the total; the thread that
// handled expert tid in the LAST pass keeps that expert's prefix, tile count and row range in `mine`
// (experts beyond NT take further passes), and per_expert(e, first_row, end_row) runs once per expert.
struct ExpertOfThread { int start, mt, o0, o1; };
template <int NT, typename T, typename F>
__device__ __forceinline__ int mtile_prefix_scan(const GemmArgs& g, int tid, int* s_pref, int* s_wtot,
                                                 ExpertOfThread& mine, T tiles_of, F per_expert) {
    const int lane = tid & 63, wave = tid >> 6;
    int run = 0;
    mine = ExpertOfThread{0, 0, 0, 0};
    for (int e0 = 0; e0 < g.E; e0 += NT) {
        const int e = e0 + tid;
        int mt = 0;
        if (e < g.E) {
            mine.o0 = g.offsets[e];
            mine.o1 = g.offsets[e + 1];
            mt = tiles_of(mine.o1 - mine.o0);
            per_expert(e, mine.o0, mine.o1);
        }
        int inc = mt;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            int o = __shfl_up(inc, d);
            if (lane >= d) inc += o;
        }
        if (lane == 63) s_wtot[wave] = inc;
        __syncthreads();
        int pre = run, tot = 0;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) {
            if (w < wave) pre += s_wtot[w];
            tot += s_wtot[w];
        }
        mine.start = pre + inc - mt;
        mine.mt = mt;
        if (e < g.E) s_pref[e] = mine.start;
        run += tot;
        if (g.E > NT) __syncthreads();   // s_wtot is rewritten by the next pass
    }
    return run;
}

// LDS row offsets of a wave's MFMA operand fragments (v_mfma_f32_16x16x32_bf16): fragment row = base + lane%16,
// bases multiples of 16.  Tokens: the wave's 32*MT rows; weights: TN fragments of 16 rows, for SWIGLU the first
// half from the gate rows (0..127 of the tile) and the second half from the matching up rows (128..255).
template <int MT, int TN, bool SWIGLU>
__device__ __forceinline__ void fragment_rows(int wm, int wn, int frow, uint32_t (&tok_off)[2 * MT], uint32_t (&w_off)[TN]) {
#pragma unroll
    for (int mi = 0; mi < 2 * MT; ++mi) tok_off[mi] = (uint32_t)((wm * 32 * MT + 16 * mi + frow) * ROW_B);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int r = SWIGLU ? ((j < TN / 2 ? 0 : 128) + wn * (8 * TN) + 16 * (j % (TN / 2))) : (wn * (16 * TN) + 16 * j);
        w_off[j] = (uint32_t)((r + frow) * ROW_B);
    }
}

// Epilogue of one wave.  acc[mi][j][i]: token row = 16*mi + lane%16 of the wave's M range; output column
// = 16*j + 4*(lane/16) + i of the wave's N range, i.e. a lane holds 4 consecutive columns (8 bytes) of one row per
// accumulator.  Storing those directly would issue 8-byte writes to 16 different rows per instruction; instead
// the wave transposes its outputs RPW rows at a time through `ep` (its own RPW * row-bytes of idle LDS) and writes
// 16 bytes per lane, whole 64/128-byte row segments per 4/8 lanes.  `out` points at the wave's first row and
// column, rows_here rows of it are valid and cols_here columns (a ragged last N tile).
template <int MT, int TN, bool SWIGLU, int RPW, bool STREAM>
__device__ __forceinline__ void store_wave_outputs(const f32x4 (&acc)[2 * MT][TN], uint8_t* ep, int lane, uint16_t* out,
                                                   int N, int rows_here, int cols_here) {
    constexpr int CW = SWIGLU ? 8 * TN : 16 * TN;    // output columns of a wave
    constexpr int RBW = CW * 2;                      // bytes per output row of a wave
    constexpr int CPR = RBW / 16;                    // 16-byte chunks per row (4 or 8)
    constexpr int KSH = CPR == 8 ? 0 : 1;            // swizzle key = (row >> KSH) & (CPR-1)
    constexpr int RPP = 64 / CPR;                    // rows per read-back instruction
    const int frow = lane & 15, fquad = lane >> 4, rr = lane / CPR, cc = lane % CPR;
#pragma unroll
    for (int pass = 0; pass < 32 * MT / RPW; ++pass) {
#pragma unroll
        for (int ml = 0; ml < RPW / 16; ++ml) {
            const int mi = pass * (RPW / 16) + ml;
            const int r = 16 * ml + frow;
            uint8_t* erow = ep + r * RBW + (fquad & 1) * 8;
            const int key = (r >> KSH) & (CPR - 1);
#pragma unroll
            for (int jj = 0; jj < (SWIGLU ? TN / 2 : TN); ++jj) {
                const u32x2 pk = epilogue_pack<SWIGLU>(acc[mi][jj], acc[mi][SWIGLU ? jj + TN / 2 : jj]);
                *reinterpret_cast<u32x2*>(erow + (((2 * jj + (fquad >> 1)) ^ key) << 4)) = pk;
            }
        }
#pragma unroll
        for (int ps = 0; ps < RPW / RPP; ++ps) {
            const int r = rr + RPP * ps;
            const u32x4 v = *reinterpret_cast<const u32x4*>(ep + r * RBW + ((cc ^ ((r >> KSH) & (CPR - 1))) << 4));
            if (pass * RPW + r < rows_here && cc * 8 < cols_here) {
                u32x4* dst = reinterpret_cast<u32x4*>(out + (size_t)(pass * RPW + r) * N + cc * 8);
                // whole 128-byte lines per 8 lanes can be written non-temporally (the pipeline's next load waits also
                // cover these stores); half lines per wave stay plain stores, so that L2 merges the halves
                if (STREAM) __builtin_nontemporal_store(v, dst); else *dst = v;
            }
        }
    }
}

// One one-workgroup tile: rows [row0, min(row0 + 64 MT, row_end)) of expert e times N tile n_tile.
// MT: 32-row units per wave along M (tile rows BM = 64*MT, 2 waves along M)
// WN: waves along N; 4 -> 8 waves of up to 128x64 outputs, two per SIMD; every wave interleaves
//     its share of the load / dequantise / LDS-store work with its MFMAs, a piece per MFMA group
// smem0 / smem1: the two LDS stages (two separate arrays: stores into one stage and reads from the other provably
//     do not alias, which lets the scheduler move them past each other)
// STREAM: no other tile reads these weights (the expert has one M tile): non-temporal loads
// One LDS stage of gemm_tile: token rows, weight rows and the start of the region that the epilogue may transpose
// through (the two parts are one array in the bf16 kernel and separate arrays in the fp8 kernel, whose weight
// streamers write them by DMA)
struct Stage {
    uint8_t *a, *b, *ep;
};

template <int MT, int WN, bool SWIGLU, bool W8, bool STREAM>
__device__ __forceinline__ void gemm_tile(const GemmArgs& g, Stage st0, Stage st1, int e, int row0, int row_end,
                                          int n_tile) {
    constexpr int NT = 128 * WN;                // threads
    constexpr int BM = 64 * MT;                 // rows per workgroup
    constexpr int RA = NT / 8;                  // A rows covered by one pass of the workgroup
    constexpr int NA = BM / RA;                 // 16-byte A chunks per thread per stage
    constexpr int RB = NT / 8;                  // B rows per pass of the workgroup (8 lanes per 128-byte row)
    constexpr int NB = BN_ROWS / RB;            // 16-byte global B chunks per thread per stage (fp8: per pair of stages)
    constexpr int NBLK = SWIGLU ? 128 : 256;    // output columns per workgroup
    constexpr int NJ = 8 / WN;                  // 32-row units of the weight tile per wave
    static_assert(MT <= 3 && NA >= 1 && NB == 4, "tile/thread mismatch");

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = (wave >> 1) % WN;
    const int n0 = n_tile * NBLK;
    const int K = g.K, N = g.N;
    const int nk = K / BK;
    // (fp8 weights under tiles below 256 rows are fetched 128 k at a time, see PAIR8 below: k_rotation keeps their
    // pairs of stages together)
    constexpr bool PAIR8 = W8;
    const int rot = (W8 && !g.alone) ? 0 : k_rotation<W8>(n_tile, nk);
    auto stage_at = [&](int kt) { const int kp = kt + rot; return kp >= nk ? kp - nk : kp; };

    // ---- per-thread load coordinates ----
    const int lrow = tid >> 3, lchunk = tid & 7;          // bf16 tiles: row tid/8 (+RA i), chunk tid%8
    int a_src[NA];
    bool a_ok[NA];                                        // a row_map entry outside x stands for a row of zeros
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        int r = min(row0 + lrow + RA * i, row_end - 1);
        a_src[i] = g.row_map ? ((gptr_i32)(uintptr_t)g.row_map)[r] : r;
        a_ok[i] = !g.row_map || (unsigned)a_src[i] < (unsigned)g.a_rows;
        if (!a_ok[i]) a_src[i] = 0;
    }
    const uint32_t a_lds = (uint32_t)(lrow * ROW_B + ((lchunk ^ swz(lrow)) << 4));

    const uint8_t* bmat0 = uni_ptr(g.b0[e]);
    const uint8_t* bmat1 = SWIGLU ? uni_ptr(g.b1[e]) : bmat0;
    gptr_f32 sc0 = W8 ? (gptr_f32)(uintptr_t)uni_ptr(g.s0[e]) : nullptr;
    gptr_f32 sc1 = (W8 && SWIGLU) ? (gptr_f32)(uintptr_t)uni_ptr(g.s1[e]) : sc0;
    // weight rows: thread (row tid/8 + 64 i of the tile, 16-byte chunk tid%8 of a 128-byte piece of the row: one
    // k-stage of bf16 weights, a pair of k-stages of fp8 weights)
    const int brow = tid >> 3, bcol_b = (tid & 7) << 4;
    int b_n[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        int r = brow + RB * i;                            // row inside the 256-row B tile
        int n = SWIGLU ? (n0 + (r & 127)) : (n0 + r);
        b_n[i] = min(n, N - 1);
    }
    const uint32_t b_lds = (uint32_t)(brow * ROW_B + (((tid & 7) ^ swz(brow)) << 4));   // (bf16 weights)
    // block-scale rows (W8): first / second 128 rows of the B tile
    int srow0 = 0, srow1 = 0;
    const int KB = K >> 7;
    if (W8) {
        if (SWIGLU) { srow0 = (n0 >> 7) * KB; srow1 = srow0; }
        else        { srow0 = (n0 >> 7) * KB; srow1 = min((n0 >> 7) + 1, (N >> 7) - 1) * KB; }
    }

    // PF register sets: global loads run PF tiles ahead of the LDS stores.  One set when the
    // workgroup is compute bound (BM = 256, which has no registers to spare); two for the smaller
    // tiles, which mostly stream weights (decode) and where bytes in flight per CU are what
    // limits the HBM rate.
    constexpr int PF = (MT <= 2) ? 2 : 1;
    u32x4 ra[PF][NA], rb[PF][NB];

    // PAIR8.  A 64-k stage of fp8 weights is 64 bytes of a row, half a cache line: fetched stage by stage, every
    // row costs two half-line requests, and a CU can only keep so many requests in flight whatever their size
    // (DeepSeek-V3 shapes, 8 rows per expert: 3.6 TB/s of weights against 5-6.5 with bf16 weights).  So the
    // weights of TWO stages are requested together, 8 lanes x 16 bytes = one whole line per row: thread (row
    // tid/8 + 64 i, i < 4; 16-byte chunk c = tid%8) gets 16 weights of stage c/4 of the pair.  Lanes c and c^4
    // then swap their second 8 bytes, after which every lane holds 8 weights of either stage (one 16-byte LDS
    // store each, the unit of work of a data item): chunk 2 (c%4) + (c/4 ^ stage) of the stage's LDS row.  Two
    // register sets of pairs; a set is refilled while the second stage of its pair is stored, three
    // iterations before it is needed again.
    const int pq = tid & 3, phb = (tid >> 2) & 1;
    u32x4 rp[2][4];
    float rps[2][2];
    uint32_t p_lds[2];
#pragma unroll
    for (int st = 0; st < 2; ++st) p_lds[st] = (uint32_t)(brow * ROW_B + (((2 * pq + (phb ^ st)) ^ swz(brow)) << 4));
    const int npair = nk >> 1, prot = rot >> 1;
    auto pair_load = [&](int pr_pipe, int ps, int i) {      // chunk i of pair pr_pipe (pipeline order) into set ps
        const bool past = pr_pipe >= npair;                  // nobody reads it: not from the weights
        int pr = min(pr_pipe, npair - 1) + prot;
        pr = pr >= npair ? pr - npair : pr;
        const uint8_t* m = (SWIGLU && i >= 2) ? bmat1 : bmat0;
        rp[ps][i] = gload16_w<STREAM>(past ? (const uint8_t*)g.a : m + (size_t)b_n[i] * K + (size_t)pr * 128 + bcol_b);
        if (i == 1) rps[ps][0] = sc0[srow0 + pr];
        if (i == 3) rps[ps][1] = sc1[srow1 + pr];
    };
    auto pair_swap = [&](int ps, int i) {                    // lanes c and c^4 swap dwords 2, 3
        const u32x4 own = rp[ps][i];
        u32x4 o;
        // first stage of the pair: c < 4 keeps its dwords 0, 1; c >= 4 takes dwords 2, 3 of lane c-4 (row_shr:4, banks 1, 3)
        o[0] = (uint32_t)__builtin_amdgcn_update_dpp((int)own[0], (int)own[2], 0x114, 0xf, 0xa, false);
        o[1] = (uint32_t)__builtin_amdgcn_update_dpp((int)own[1], (int)own[3], 0x114, 0xf, 0xa, false);
        // second stage: c >= 4 keeps its dwords 0, 1; c < 4 takes dwords 2, 3 of lane c+4 (row_shl:4, banks 0, 2)
        o[2] = (uint32_t)__builtin_amdgcn_update_dpp((int)own[0], (int)own[2], 0x104, 0xf, 0x5, false);
        o[3] = (uint32_t)__builtin_amdgcn_update_dpp((int)own[1], (int)own[3], 0x104, 0xf, 0x5, false);
        rp[ps][i] = o;
    };
    auto pair_store = [&](uint8_t* Bs, int ps, int i, int st) {   // the 8 weights of stage st of the pair -> LDS
        const u32x4 o = dequant8(rp[ps][i][2 * st], rp[ps][i][2 * st + 1], rps[ps][i >> 1]);
        *reinterpret_cast<u32x4*>(Bs + p_lds[st] + i * RB * ROW_B) = o;
    };
    auto gload = [&](int kt_pipe, int set) {
        const int kt = stage_at(kt_pipe);
        const size_t kofs = (size_t)kt * BK;
#pragma unroll
        for (int i = 0; i < NA; ++i) ra[set][i] = gload16(g.a + (size_t)a_src[i] * K + kofs + lchunk * 8);
        if (PAIR8) return;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const uint8_t* m = (SWIGLU && i >= NB / 2) ? bmat1 : bmat0;  // rows >= 128 of the B tile are the up matrix
            rb[set][i] = gload16_w<STREAM>(m + ((size_t)b_n[i] * K + kofs) * 2 + bcol_b);
        }
    };
    auto lds_store = [&](Stage S, int set) {
        uint8_t *As = S.a, *Bs = S.b;
#pragma unroll
        for (int i = 0; i < NA; ++i) *reinterpret_cast<u32x4*>(As + a_lds + i * RA * ROW_B) = a_ok[i] ? ra[set][i] : u32x4{0, 0, 0, 0};
        if (PAIR8) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                pair_swap(0, i);
                pair_store(Bs, 0, i, 0);
            }
        } else {
#pragma unroll
            for (int i = 0; i < NB; ++i) *reinterpret_cast<u32x4*>(Bs + b_lds + i * RB * ROW_B) = rb[set][i];
        }
    };

    // ---- MFMA operand coordinates (v_mfma_f32_16x16x32_bf16) ----
    // fragment row = base + lane%16 (bases are multiples of 16); logical chunk = 4*s + lane/16 for
    // the 32-wide k-step s of the stage: lane l supplies k = 8*(l/16) .. +7 of row l%16
    const int frow = lane & 15, fquad = lane >> 4, fkey = swz(frow);
    // The LDS serves a 16-byte read 8 + 8 lanes at a time (lanes 8i.. together with 32+8i..):
    // such a pair of lane groups must read neighbouring chunks of the same rows, which is what the
    // swizzle keeps conflict-free, so lane group q takes chunk 0,2,1,3 of the k-step instead of q
    // (with q the counter SQ_LDS_BANK_CONFLICT reads 22 % of the busy cycles, with this order
    // 0.3 %).  Both operands use the same order, and a dot product does not care in which order
    // k is walked.
    const int fchunk = ((fquad & 1) << 1) | (fquad >> 1);
    constexpr int TM = 2 * MT, TN = 2 * NJ;       // 16-row token tiles / 16-row weight tiles per wave
    uint32_t tok_off[TM], w_off[TN];
    fragment_rows<MT, TN, SWIGLU>(wm, wn, frow, tok_off, w_off);

    f32x4 acc[TM][TN];
#pragma unroll
    for (int mi = 0; mi < TM; ++mi)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[mi][j] = f32x4{0};

    // A stage is multiplied in NU sub-phases: k-step s (32 wide) x token part q (TQ tiles), each
    // TQ x TN MFMAs.  Weight fragments are double-buffered by k-step; token parts ping-pong between
    // two small buffers.  Slot v of an iteration issues the MFMAs of sub-phase v-2 (the last two
    // sub-phases of a stage run in the first two slots of the next iteration, across the workgroup
    // barrier) and then requests the fragments of sub-phase v, whose buffer those MFMAs just freed.
    constexpr int TQ = MT == 3 ? 3 : (MT >= 2) ? MT / 2 : 1;    // token tiles per part (the parts per k-step, 2 MT / TQ, must divide the 4 weight tiles)
    constexpr int NP = TM / TQ;                   // parts per k-step
    constexpr int NU = 2 * NP;                    // sub-phases per stage
    bf16x8 wfr[2][TN], tq[2][TQ];
    // 16-row token groups of this wave that hold rows of the expert (the same for every lane of the wave).  With
    // few rows per expert most groups are empty: a wave whose last group is empty runs the loop in its
    // `part` form, which skips the fragment reads and MFMAs of empty groups behind wave-uniform branches
    // (Mixtral-8x22B, 64 rows per expert under 128-row tiles: gate/up 0.61 -> 0.55 ms; DeepSeek-V3 shapes, 8 rows
    // per expert, fp8: 4.3 -> 5.0 TB/s of weights).  Full waves keep the branch-free form: the branches cost the
    // exact operand waits (128 rows per expert: down projection 0.27 -> 0.30 ms with them).
    bool live[TM];
#pragma unroll
    for (int mi = 0; mi < TM; ++mi) live[mi] = wm * 32 * MT + 16 * mi < row_end - row0;
    auto read_w1 = [&](Stage S, int s, int j, auto part) __attribute__((always_inline)) {
        if (decltype(part)::value && !live[0]) return;
        const uint8_t* Bs = S.b;
        const uint32_t coff = (uint32_t)(((4 * s + fchunk) ^ fkey) << 4);
        wfr[s][j] = *reinterpret_cast<const bf16x8*>(Bs + w_off[j] + coff);
    };
    auto read_tq = [&](Stage S, int u, auto part) __attribute__((always_inline)) {
        const uint8_t* As = S.a;
        const int s = u / NP, q = u % NP;
        const uint32_t coff = (uint32_t)(((4 * s + fchunk) ^ fkey) << 4);
#pragma unroll
        for (int i = 0; i < TQ; ++i)
            if (!decltype(part)::value || live[q * TQ + i])
                tq[u & 1][i] = *reinterpret_cast<const bf16x8*>(As + tok_off[q * TQ + i] + coff);
    };
    auto mfma_sub = [&](int u, auto part) __attribute__((always_inline)) {
        const int s = u / NP, q = u % NP;
#pragma unroll
        for (int i = 0; i < TQ; ++i)
            if (!decltype(part)::value || live[q * TQ + i])
#pragma unroll
            for (int jx = 0; jx < TN; ++jx) {
                // snake order over the weight fragments: every instruction differs from the one before in
                // ONE operand (fewer input toggles per MFMA on a power-limited chip; +0.4 % measured)
                const int j = ((i + u) & 1) ? TN - 1 - jx : jx;
                acc[q * TQ + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wfr[s][j], tq[u & 1][i], acc[q * TQ + i][j], 0, 0, 0);
            }
    };
    // ---- main loop ----
    // On entry to iteration kt: LDS stage kt&1 holds tile kt and the registers hold tiles kt+1 ..
    // kt+PF (possibly still in flight).  The iteration moves tile kt+1 into the other LDS stage,
    // refills that register set with tile kt+1+PF and multiplies tile kt.
    gload(0, 0);
    if (PAIR8) {
#pragma unroll
        for (int i = 0; i < 4; ++i) pair_load(0, 0, i);
#pragma unroll
        for (int i = 0; i < 4; ++i) pair_load(1, 1, i);
    }
    lds_store(st0, 0);
    // No load or store of the pipeline sits under a branch or in a region that only some waves
    // execute (past the end the last tile is loaded again and stored where nobody reads it): with
    // straight-line code the compiler counts the outstanding loads exactly, so a store waits only
    // for the chunk it stores.  Under a branch it must assume the load may never have been issued
    // and waits for ALL outstanding loads, which serialises the whole pipeline.
#pragma unroll
    for (int d = 0; d < PF; ++d) gload(min(1 + d, nk - 1), d);
    __syncthreads();
    // One data item = one LDS store's worth of this thread's staged chunks (a 16-byte token chunk,
    // a 16-byte bf16 weight chunk, or half of a 16-byte fp8 weight chunk -> 8 bf16): store it to the
    // other stage and, once a chunk's last item is stored, refill its registers with the chunk of
    // tile kt+1+PF.  The items are spread over the iteration, one per group of MFMAs, so LDS, the
    // vector-memory pipe and the matrix core see a steady mix instead of bursts; with exact load
    // waits each item stalls only until its own chunk (requested PF iterations earlier) is there.
    constexpr int NI = NA + NB;
    // par = kt & 1 and ps, the register set of the pair that stage kt+1 belongs to, are literals at the call sites
    auto data_item = [&](int i, Stage S, int kt, int set, int par, int ps) __attribute__((always_inline)) {
        uint8_t *As = S.a, *Bs = S.b;
        const int kn = stage_at(min(kt + 1 + PF, nk - 1));
        const size_t kofs = (size_t)kn * BK;
        // past the end nobody reads what is loaded: streamed weights would come from HBM once more
        // (PF + 1 stages per tile), so those loads take the first 16 bytes of the activations instead
        const bool past = kt + 1 + PF >= nk;
        if (i < NA) {
            *reinterpret_cast<u32x4*>(As + a_lds + i * RA * ROW_B) = a_ok[i] ? ra[set][i] : u32x4{0, 0, 0, 0};
            ra[set][i] = gload16(g.a + (size_t)a_src[i] * K + kofs + lchunk * 8);
        } else if (PAIR8) {
            const int b = i - NA;
            if (par) {                      // stage kt+1 opens a pair
                pair_swap(ps, b);
                pair_store(Bs, ps, b, 0);
            } else {                        // it closes one: the set is free for the pair after the next
                pair_store(Bs, ps, b, 1);
                pair_load((kt >> 1) + 2, ps, b);
            }
        } else {
            const int b = i - NA;
            const uint8_t* m = (SWIGLU && b >= NB / 2) ? bmat1 : bmat0;
            *reinterpret_cast<u32x4*>(Bs + b_lds + b * RB * ROW_B) = rb[set][b];
            rb[set][b] = gload16_w<STREAM>(past ? (const uint8_t*)g.a : m + ((size_t)b_n[b] * K + kofs) * 2 + bcol_b);
        }
    };
    constexpr int NG = NU;                        // one group of MFMAs per slot
    constexpr int WPS = TN / NP;                  // weight fragments of the second k-step read per slot
    auto iteration = [&](int kt, int set, int par, int ps, auto part) __attribute__((always_inline)) {   // par == kt & 1
        const Stage rd = par ? st1 : st0;
        const Stage wr = par ? st0 : st1;
#pragma unroll
        for (int v = 0; v < NU; ++v) {
            // group v takes items [v*NI/NG, (v+1)*NI/NG): in order, so the two halves of an fp8
            // chunk are stored before its registers are refilled
#pragma unroll
            for (int i0 = v * NI / NG; i0 < (v + 1) * NI / NG; ++i0) {
                data_item(i0, wr, kt, set, par, ps);
            }
            if (!W8) __builtin_amdgcn_sched_barrier(0);
            if (v >= 2) mfma_sub(v - 2, part);
            else if (kt > 0) mfma_sub(NU - 2 + v, part);
            read_tq(rd, v, part);
            if (v == 0) {
#pragma unroll
                for (int j = 0; j < TN; ++j) read_w1(rd, 0, j, part);
            } else if (v >= 2 && v < 2 + NP) {
#pragma unroll
                for (int j = (v - 2) * WPS; j < (v - 1) * WPS; ++j) read_w1(rd, 1, j, part);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();   // (waits for this wave's LDS reads and writes, then for the other waves)
    };
    // Unrolled by two, the stage parity is a literal and every LDS address is a register plus an
    // immediate (about 20 vector and 12 scalar instructions less per iteration; headline -2 %).  The
    // bf16 kernel with BM = 256 has no registers for the longer live ranges (it would spill) and
    // keeps the rolled loop.
    auto k_loop = [&](auto part) __attribute__((always_inline)) {
        if (PAIR8) {
            // stage kt+1 belongs to pair (kt+1)/2, whose register set alternates: by four, every index is a literal
            int kt = 0;
            for (; kt + 4 <= nk; kt += 4) {
                iteration(kt, 0, 0, 0, part);
                iteration(kt + 1, 1, 1, 1, part);
                iteration(kt + 2, 0, 0, 1, part);
                iteration(kt + 3, 1, 1, 0, part);
            }
            if (kt < nk) {                       // (an even number of stages: fp8 scales come per 128 k)
                iteration(kt, 0, 0, 0, part);
                iteration(kt + 1, 1, 1, 1, part);
            }
        } else if (W8 || PF == 2) {
            int kt = 0;
            for (; kt + 2 <= nk; kt += 2) {
                iteration(kt, 0, 0, 0, part);
                iteration(kt + 1, PF - 1, 1, 0, part);
            }
            if (kt < nk) iteration(kt, 0, 0, 0, part);
        } else {
            for (int kt = 0; kt < nk; ++kt) iteration(kt, 0, kt & 1, 0, part);
        }
        mfma_sub(NU - 2, part);
        mfma_sub(NU - 1, part);
    };
    // (both forms pass the same barriers, so the waves of a workgroup may differ in theirs)
    if (!live[TM - 1]) k_loop(std::true_type{});
    else k_loop(std::false_type{});

    // ---- epilogue ----
    // All waves passed the loop's last barrier, so no one reads the stages: each wave transposes through its own
    // slice of them.
    constexpr int CW = SWIGLU ? 8 * TN : 16 * TN;    // output columns of this wave
    uint8_t* ep = ((wave < 4) ? st0.ep : st1.ep) + (wave & 3) * (32 * MT * CW * 2);
    const int ncol0 = n0 + wn * CW;
    store_wave_outputs<MT, TN, SWIGLU, 32 * MT, false>(acc, ep, lane, g.c + (size_t)(row0 + wm * 32 * MT) * N + ncol0, N,
                                                       min(BM, row_end - row0) - wm * 32 * MT, N - ncol0);
}

// ---- fp8 weight streamer: experts of up to 64 rows in calls of one-workgroup tiles alone ----
//
// With a handful of rows per expert a launch reads every weight once (Expert_Wrapper.forward in its decoding use,
// Wrapper.py:470-530) and is bound by how fast a CU can take fp8 weights in.  Through gemm_tile a 64-k stage of 256
// weight rows costs 16 KiB of global loads into registers, the conversion, 32 KiB of LDS stores, a barrier and
// 64 KiB of fragment reads, and streams at 4-5 TB/s.  Here
//  * the workgroup's 8 waves split the tile's WEIGHT rows (32 each: a 16-row gate fragment and the matching up
//    fragment, or two fragments of the down matrix) and every wave multiplies all token rows, so a weight is
//    converted once, by the wave that feeds it to the matrix core;
//  * weights reach LDS as fp8 by DMA (buffer_load ... lds), 8 lanes x 16 bytes per row = whole 128-byte lines per
//    request, 128 k at a time, into the wave's own 4 KiB of a buffer: no staging registers, no LDS stores, half the
//    bytes, and three buffers keep two 128-k blocks in flight per CU;
//  * a lane reads 16 consecutive fp8 weights of its fragment row (one ds_read_b128), which after conversion are its
//    A operands of BOTH 32-wide k-steps of a 64-k half: lane group q holds k = 16 f(q) + 8 s + (0..7) in step s
//    (f = 0, 2, 1, 3), and the token operand reads the chunk that holds those k.  A dot product does not care in which order k is walked,
//    and the order depends on nothing but the column: a row's result does not depend on its tile or its neighbours.
// LDS layouts (the DMA lets every lane fetch what belongs at its place, so swizzles are free):
//  weights: 128-byte rows, 16-byte part c of fragment row r at part c ^ wsw(r); tokens: 256-byte rows (128 k), chunk
//  c of row r at chunk c ^ tsw(r).  The LDS serves lanes 8 i .. 8 i + 7 together with lanes 32 + 8 i .. (the same 8
//  rows, lane groups q and q + 2, whose chunks f(q) and f(q + 2) = f(q) + 1 are neighbours): with these keys their 16
//  reads fall on 16 different bank groups.  (Measured with 8 waves reading back to back: 32 cycles per wave and
//  ds_read_b128 for both layouts, 55 with lane group q on chunk q.)
constexpr int S8_WBYTES = 32 * 1024;              // weight region of a buffer: 8 waves x 32 rows x 128 fp8
constexpr int S8_TROWS = 64;                      // token rows staged

// A buffer of the weight streamers: the weight region and the token region are separate LDS arrays, so that a read of
// one never has to wait for a DMA into the other
struct SBuf {
    uint8_t *w, *t;
};

// LDS of a workgroup of the tile kernel or of the split kernel, an array each: three weight buffers of 32 KiB, token buffers of
// 16, 24 (split kernel: 16) and 16 KiB
struct TileLds {
    uint8_t *w0, *w1, *w2, *t0, *t1, *t2;
};

// Whether a call of a group has tiles of both kinds (where the persistent body can address its rows): from a mean of 128 rows per expert
// on; sums of fp8 weights start elsewhere in calls of one kind (k_rotation).  Sums of bf16 weights do not depend on it: with many
// experts some hold most of the rows well below that mean (and would be 128-row tiles that fetch their weights again and again), and all
// gain by the other rounds.  Both kinds cost a call 7 to 10 us in front of the first tiles, against a gain that grows with the weights and
// with the mean: below 128 rows the call has to be long enough for the one, and its rows enough for the other.  Layers, us, one kind ->
// both.  Above the line: 160 experts, DeepSeek-V2-236B, 900 / 1500 / 2500 tokens (means of 33 to 93 rows) skewed 1403 / 1591 / 1911 -> 1357 / 1491 /
// 1693, even 1405 / 1518 / 1704 -> 1336 / 1467 / 1644; 64, DeepSeek-V2-Lite, 920 / 1100 / 1300 skewed 284 / 310 / 340 -> 277 / 301 / 332, even the
// same; 96 of 5120 x 1536 (hidden x intermediate size), 689 / 961 (43 / 60 rows) skewed 914 / 1025 -> 878 / 980, even 916 / 970 -> 847 / 908.  Below it:
// 64 experts, 2048 x 1024, 939 tokens 225 -> 241, 1024 x 1024 119 -> 142, 2048 x 768, 1259 202 -> 211; 128,
// 2048 x 512, 726 149 -> 156; 256, 1024 x 384, 1451 107 -> 117.  32 experts, above it too: 2048 x 4096, 470 / 630 415 / 461 -> 442 / 470.  138 calls of
// 64 to 256 experts, even and skewed: above it both kinds are 3.9 per cent faster in the mean, 1.6 slower at most; below it 1.8 slower.
template <bool W8>
inline bool both_kinds(long n_rows, int E, int K, int N) {
    const long mean = E > 0 ? n_rows / E : 0;
    const double weights = (double)E * K * N;      // of one matrix
    return mean >= 128 || (!W8 && E >= 64 && mean >= 32 && weights >= 1.6e8 && weights * mean * mean >= 1.33e12);
}

// How the down projection of one MLP is cut when its k is: row tiles of `rows` (256: on the persistent body, else on the split
// kernel), k into `slices` of up to `blocks` blocks of 128.  part: where the fp32 sums go, [slices][n_rows][N].
struct SplitPlan {
    int m_tiles, rows, slices, blocks;
};
struct SplitArgs {
    SplitPlan plan;
    int n_rows;
    float* part;
};

// A slice of k for a tile whose sums other workgroups share (split kernel): blocks first .. first + count - 1 of 128 k, and
// where the fp32 sums go: part[(row - row_base) * N + column]
struct KSlice {
    int first, count, row_base;
    float* part;
};

template <int TG, bool SWIGLU, bool SPLIT = false, typename C>   // TG: 16-row token groups multiplied (the expert has at most 16 TG <= 64 rows)
__device__ __forceinline__ void stream8_tile(const GemmArgs& g, SBuf buf0, SBuf buf1, SBuf buf2, int e, int row0,
                                             int row_end, int n_tile, C& claims, KSlice ks = {}) {
    constexpr int NBLK = SWIGLU ? 128 : 256;
    constexpr int NDW = 4, NDT = 2;               // DMA instructions per wave and 128-k block: weights, tokens
    // Operations that may stay in flight at the wait for a block: the DMA of the next block, NDW + NDT instructions
    // (the counter retires in issue order).  The next block's two scale loads are issued before its DMA and are
    // older still: not counting them costs at most a wait for two small loads that hit in L2, and keeps the count
    // right for the first block, which has no scale loads of a block before it behind its DMA.
    constexpr int VM_BLOCK = NDW + NDT;
    static_assert(!(SPLIT && SWIGLU), "slices of k: the down projection");
    static_assert(TG >= 1 && 16 * TG <= S8_TROWS, "token rows staged");
    const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
    const int n0 = n_tile * NBLK;
    const int K = g.K, N = g.N;
    const int npair = SPLIT ? ks.count : K >> 7;             // blocks of 128 k multiplied
    const int kfirst = SPLIT ? ks.first : 0;
    // N tile t walks k from 128-k block t (mod the number of blocks), so that the requests in flight on the chip do
    // not share their low address bits (weight rows are K bytes apart); a column's order depends on its tile alone
    const int prot = n_tile % npair;

    // ---- DMA coordinates ----
    // weights, instruction i: rows 8 i + lane / 8 of the wave's 32 (fragment i / 2, fragment row 8 (i & 1) + lane / 8)
    const int lr = lane >> 3, pp = lane & 7;
    uint32_t w_voff[NDW];
    const uint8_t* bmat[2];
    gptr_f32 sc[2];
    int srow[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        bmat[j] = uni_ptr((SWIGLU && j == 1) ? g.b1[e] : g.b0[e]);
        sc[j] = (gptr_f32)(uintptr_t)uni_ptr((SWIGLU && j == 1) ? g.s1[e] : g.s0[e]);
        srow[j] = min((n0 + (SWIGLU ? 0 : 32 * wave)) >> 7, (N >> 7) - 1) * (K >> 7) + kfirst;
    }
#pragma unroll
    for (int i = 0; i < NDW; ++i) {
        const int fr = 8 * (i & 1) + lr;
        const int rt = SWIGLU ? 16 * wave + fr : 32 * wave + 16 * (i >> 1) + fr;      // row of the tile's N range
        w_voff[i] = (uint32_t)min(n0 + rt, N - 1) * (uint32_t)K + (uint32_t)((pp ^ wsw(fr)) << 4);
    }
    // tokens, instruction i: rows 8 wave + 4 i + lane / 16 of the 64 staged, chunk lane % 16.  Gathered rows go through
    // one descriptor over x (a row_map entry outside x reads zeros), sorted rows through one that holds the tile's rows
    // and nothing else.  Rows past the expert's last get an offset past either descriptor: zeros arrive in LDS
    // without a request to memory (nobody uses the products of those rows; the instruction still counts).
    uint32_t t_voff[NDT];
    const uint8_t* a_base = reinterpret_cast<const uint8_t*>(g.a) + (g.row_map ? (size_t)0 : (size_t)row0 * K * 2);
    const int a_records = g.row_map ? (int)(uint32_t)g.a_bytes : (row_end - row0) * K * 2;
#pragma unroll
    for (int i = 0; i < NDT; ++i) {
        const int tr = 8 * wave + 4 * i + (lane >> 4);
        const int r = min(row0 + tr, row_end - 1);
        const int src = g.row_map ? ((gptr_i32)(uintptr_t)g.row_map)[r] : r - row0;
        t_voff[i] = (uint32_t)src * (uint32_t)(K * 2) + (uint32_t)(((lane & 15) ^ tsw(tr)) << 4);
        if (row0 + tr >= row_end || (g.row_map && (unsigned)src >= (unsigned)g.a_rows)) t_voff[i] = 0xfffffff0u;
    }
    float rsc[2][2];                              // block scales of the block being multiplied / of the next one
    auto scales = [&](int p_pipe, int set) {
        int pr = min(p_pipe, npair - 1) + prot;
        pr = pr >= npair ? pr - npair : pr;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)sc[j], 0, -1, 0x00020000);
            rsc[set][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, 0, (srow[j] + pr) * 4, 0));
        }
    };
    // DMA instruction i of a block: 0 .. NDW-1 weights (read once: non-temporal, which is worth 5 % of the stream),
    // NDW .. NDW+NDT-1 tokens
    auto dma_one = [&](int p_pipe, SBuf buf, int i) __attribute__((always_inline)) {
        // past the end of k nobody reads what arrives: an empty descriptor returns zeros without touching memory,
        // and the instruction still counts
        const int live = uni(p_pipe < npair ? -1 : 0);   // (a scalar, or the descriptor ends up in vector registers)
        int pr = min(p_pipe, npair - 1) + prot;
        pr = pr >= npair ? pr - npair : pr;
        if (i < NDW) {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)bmat[i >> 1], 0, live, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_u8)(buf.w + wave * 4096 + i * 1024), 16, w_voff[i], (uint32_t)((pr + kfirst) * 128), 0, 2);
        } else {
            const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)a_base, 0, live & a_records, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_u8)(buf.t + wave * 2048 + (i - NDW) * 1024), 16, t_voff[i - NDW],
                                                     (uint32_t)((pr + kfirst) * 256), 0, 0);
        }
    };
    auto dma = [&](int p_pipe, SBuf buf) {
#pragma unroll
        for (int i = 0; i < NDW + NDT; ++i) dma_one(p_pipe, buf, i);
    };

    const int frow = lane & 15, q = lane >> 4;
    const int fq = ((q & 1) << 1) | (q >> 1);
    const uint32_t w_rd = (uint32_t)(wave * 4096 + frow * 128), wkey = (uint32_t)wsw(frow);
    const uint32_t t_rd = (uint32_t)(frow * 256), tkey = (uint32_t)tsw(frow);   // (group bases are multiples of 16)
    f32x4 acc[TG][2];
#pragma unroll
    for (int t = 0; t < TG; ++t) { acc[t][0] = f32x4{0}; acc[t][1] = f32x4{0}; }

    // Iteration p multiplies block p out of buffer p % 3.  Before it: this wave's DMA of block p has landed (at most the
    // DMA of block p + 1 is outstanding) and its LDS reads have returned, then everybody's (a bare s_barrier: a fence
    // would make the compiler wait for ALL outstanding DMA).  After the barrier every wave has left block p - 1,
    // whose buffer takes block p + 2 (its DMA is spread over the iteration).  The scale loads come BEFORE the DMA: the
    // compiler's own wait for a scale counts everything issued after it as allowed to be in flight.
    auto iteration = [&](int p, SBuf rd, SBuf refill, int sset) __attribute__((always_inline)) {
        // (lgkmcnt: this wave's LDS reads of block p - 1 have returned -- its last matrix instructions may be scheduled
        // behind the barrier, and the buffer they read is refilled right after it)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(VM_BLOCK) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        scales(p + 1, sset ^ 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            bf16x8 wa[2][2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const u32x4 raw = *reinterpret_cast<const u32x4*>(rd.w + w_rd + j * 2048 + (((4 * h + fq) ^ wkey) << 4));
                wa[j][0] = __builtin_bit_cast(bf16x8, dequant8(raw[0], raw[1], rsc[sset][j]));
                wa[j][1] = __builtin_bit_cast(bf16x8, dequant8(raw[2], raw[3], rsc[sset][j]));
            }
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2) {
                const uint32_t coff = (uint32_t)(((8 * h + 2 * fq + s2) ^ tkey) << 4);
#pragma unroll
                for (int t = 0; t < TG; ++t) {
                    const bf16x8 tf = *reinterpret_cast<const bf16x8*>(rd.t + t_rd + t * 16 * 256 + coff);
                    acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[0][s2], tf, acc[t][0], 0, 0, 0);
                    acc[t][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[1][s2], tf, acc[t][1], 0, 0, 0);
                }
                // the refill of the freed buffer goes out between the four groups of matrix instructions (2, 2, 1, 1
                // DMA instructions): a wave that issues all six first stands in the memory pipeline's queue while its
                // matrix instructions wait behind them (3 % at 40-64 rows)
                const int st = 2 * h + s2;
                __builtin_amdgcn_sched_barrier(0);
                dma_one(p + 2, refill, st < 2 ? 2 * st : st + 2);
                if (st < 2) dma_one(p + 2, refill, 2 * st + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    scales(0, 0);
    dma(0, buf0);
    dma(1, buf1);
    int p = 0;
    for (; p + 3 <= npair; p += 3) {
        iteration(p, buf0, buf2, 0);
        iteration(p + 1, buf1, buf0, 1);
        iteration(p + 2, buf2, buf1, 0);
        // (three iterations flip the scale set: swap so that the loop body keeps literal indices)
        const float t0 = rsc[0][0], t1 = rsc[0][1];
        rsc[0][0] = rsc[1][0]; rsc[0][1] = rsc[1][1];
        rsc[1][0] = t0; rsc[1][1] = t1;
    }
    if (p < npair) {
        iteration(p, buf0, buf2, 0);
        if (p + 1 < npair) iteration(p + 1, buf1, buf0, 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no DMA may land in LDS after the workgroup has gone
    claims.ask();

    // ---- epilogue: a lane holds 4 consecutive columns of one row per accumulator and stores them itself ----
#pragma unroll
    for (int t = 0; t < TG; ++t) {
        const int r = row0 + 16 * t + frow;
        if (r >= row_end) continue;
        if (SWIGLU) {
            const int col = n0 + 16 * wave + 4 * q;
            if (col < N) *reinterpret_cast<u32x2*>(g.c + (size_t)r * N + col) = epilogue_pack<true>(acc[t][0], acc[t][1]);
        } else {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int col = n0 + 32 * wave + 16 * j + 4 * q;
                if (col >= N) continue;
                if (SPLIT) *reinterpret_cast<f32x4*>(ks.part + (size_t)(r - ks.row_base) * N + col) = acc[t][j];
                else *reinterpret_cast<u32x2*>(g.c + (size_t)r * N + col) = epilogue_pack<false>(acc[t][j], acc[t][j]);
            }
        }
    }
}


// ---- fp8 weight streamer in the persistent body's summation order: tiles of up to 192 rows ----
//
// The same division of labour as stream8_tile (8 waves x 32 weight rows, fp8 weights by DMA in whole lines, every wave
// multiplies all token rows, a weight is converted once, by the wave that multiplies it), for tiles whose rows another
// kernel might have computed: what an fp8 expert's full 256-row tiles leave over, the pieces of the persistent body's last
// tiles, and in calls that this kernel serves alone the experts (or 128-row slices of experts) above 64 rows.  A row's bits
// must then not depend on who computes it, so every matrix instruction gets the k values the persistent body gives it,
// in the same lanes: lane group q holds k = 32 s + 8 f(q) + (0..7) of k-step s, f = 0, 2, 1, 3.  Those are the 16-byte token
// chunk 4 s + f(q) of a 64-k half, and 8 consecutive fp8 weights, one half of the 16-byte part 2 s + (q & 1): lane groups q and
// q + 2 use the two halves of one part.  So lane group q reads part q, the lower half of the wave those of step 0 and the upper
// those of step 1, and one v_permlane32_swap per pair of dwords gives every lane its 8 weights of either step: every weight
// leaves LDS once.
//
// Weights travel in blocks of 128 k through three buffers, token rows in halves of 64 k with one barrier per half: up to 128
// rows through three buffers of 16 KiB, two halves ahead, above through two of 24 KiB (one is two arrays), one half ahead.
// A wave brings and reads its own weight rows, so only token rows need the barrier.
//
// The k loop is a pipeline of slots, one per k-step of 32 and part of at most 4 token groups.  Slot n requests the token operands of
// part n, multiplies part n - 1 and converts its share of the weights of the step after the one that is multiplied, so the LDS
// latency and the conversion stand beside matrix instructions instead of in front of them.  Slots run on across the barriers; in
// front of the first one operands and accumulators are zero.
//
// What bounds it: power.  DeepSeek-V3 shapes, 256 experts of 96 rows, gate and up 1833 us; with operands of zero, the same
// instructions and bytes, 1447 (5.2 TB/s of weights), at 176 rows 2519 and 1792; without any load 1201 and 1652, weights alone
// 1312.  Behind that come the instruction slots of a SIMD: a matrix instruction takes 8 of its 16 cycles from the vector ALU, a
// vector instruction 4, an LDS read about 6, which at 96 rows adds up to 1200 cycles a half, 600 of them the conversion.
// Against reads at the end of a slot, which the next slot waited for, two LDS reads a fragment and half, and the compiler's order of
// products and conversion, same box, us: 96 rows each 1863 -> 1828 (gate and up), 1067 -> 1045 (down), 176 rows 2569 -> 2525 and
// 1460 -> 1442.
// weights in LDS: 16-byte part c of fragment row r at part c ^ wsx(r).  A 16-byte read serves lanes 0-3, 12-15, 20-27 together, then
// 4-11, 16-19, 28-31, and the same of the upper half-wave: with lane group q on part q their 16 reads fall on 16 different bank
// groups (wsw gives two on each)
__device__ __forceinline__ int wsx(int r) { return (r & 2) | ((r >> 1) & 4); }
template <int TG, bool SWIGLU, bool SPLIT = false, typename C>   // TG: 16-row token groups multiplied (1 .. 12)
__device__ __forceinline__ void stream8x_tile(const GemmArgs& g, const TileLds& lds, int e, int row0, int row_end, int n_tile,
                                              bool rotate, C& claims, KSlice ks = {}) {
    constexpr int NBLK = SWIGLU ? 128 : 256;
    constexpr bool WIDE = TG > 8;                 // two token buffers
    constexpr int NP = (TG + 3) / 4;              // parts of a k-step
    constexpr int V = 2 * NP;                     // slots of a half
    constexpr int NDT = (2 * TG + 7) / 8;         // token DMA instructions per wave and half (8 rows each)
    constexpr int NS = SWIGLU ? 2 : 1;            // block scales of a wave's columns
    // Order of issue in half h of block p: the tokens two halves ahead (above 128 rows: one), h = 0: the scales of block p + 1, and
    // the weights of block p + 2 (all four instructions in h = 0; above 128 rows two in either half).  VM: DMA operations that may
    // stay in flight at the barrier of a half, those issued after its tokens.  (The scales do not count: nothing holds their
    // place among the DMA, see the persistent body)
    constexpr int VM = WIDE ? 2 : 4 + NDT;
    static_assert(!(SPLIT && SWIGLU), "slices of k: the down projection");
    static_assert(TG >= 1 && TG <= 12, "token rows staged");
    const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
    const int n0 = n_tile * NBLK;
    const int K = g.K, N = g.N;
    const int npair = SPLIT ? ks.count : K >> 7;             // blocks of 128 k multiplied
    const int kfirst = SPLIT ? ks.first : 0;
    const int prot = rotate ? n_tile % npair : 0;             // k_rotation in blocks of 128 k
    auto block_of = [&](int p_pipe) { const int pr = min(p_pipe, npair - 1) + prot; return pr >= npair ? pr - npair : pr; };

    // ---- DMA coordinates ----
    // weights, instruction i (0..3): rows 8 i + lane / 8 of the wave's 32 (fragment i / 2, fragment row 8 (i & 1) + lane / 8);
    // 16-byte part c of fragment row r at part c ^ wsx(r)
    const int lr = lane >> 3, pp = lane & 7;
    uint32_t w_voff[4], t_voff[3];                // (NDT of the latter are used)
    const uint8_t* bmat[2];
    const uint8_t* sc[2];
    int srow = 0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        bmat[j] = uni_ptr((SWIGLU && j == 1) ? g.b1[e] : g.b0[e]);
        sc[j] = uni_ptr((SWIGLU && j == 1) ? g.s1[e] : g.s0[e]);
    }
    srow = min((n0 + (SWIGLU ? 0 : 32 * wave)) >> 7, (N >> 7) - 1) * (K >> 7) + kfirst;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int fr = 8 * (i & 1) + lr;
        const int rt = SWIGLU ? 16 * wave + fr : 32 * wave + 16 * (i >> 1) + fr;      // row of the tile's N range
        w_voff[i] = (uint32_t)min(n0 + rt, N - 1) * (uint32_t)K + (uint32_t)((pp ^ wsx(fr)) << 4);
    }
    // tokens, instruction i: rows 64 i + 8 wave + lane / 8, 16-byte chunk c of row r at chunk c ^ swz(r) (the persistent
    // kernel's layout of a 64-k stage).  Rows past the tile's last: zeros, no request.
    const uint8_t* a_base = reinterpret_cast<const uint8_t*>(g.a) + (g.row_map ? (size_t)0 : (size_t)row0 * K * 2);
    const int a_records = g.row_map ? (int)(uint32_t)g.a_bytes : (row_end - row0) * K * 2;
#pragma unroll
    for (int i = 0; i < NDT; ++i) {
        const int tr = 64 * i + 8 * wave + lr;
        const int r = min(row0 + tr, row_end - 1);
        const int src = g.row_map ? ((gptr_i32)(uintptr_t)g.row_map)[r] : r - row0;
        t_voff[i] = (uint32_t)src * (uint32_t)(K * 2) + (uint32_t)((pp ^ swz(tr)) << 4);
        if (row0 + tr >= row_end || (g.row_map && (unsigned)src >= (unsigned)g.a_rows)) t_voff[i] = 0xfffffff0u;
    }
    float rsc[3][2];                              // block scales, block p in set p % 3
    auto scales = [&](int p_pipe, int set) __attribute__((always_inline)) {   // (buffer loads: scalar ones share a counter with the operand reads)
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)sc[j], 0, -1, 0x00020000);
            rsc[set][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, 0, (srow + block_of(p_pipe)) * 4, 0));
        }
    };
    // weight DMA instruction i of block p_pipe (pipeline order) / token DMA instruction i of half-block hb_pipe, into token
    // buffer tb
    auto dma_w = [&](int p_pipe, uint8_t* wb, int i) __attribute__((always_inline)) {
        const int live = uni(p_pipe < npair ? -1 : 0);   // past the end: an empty descriptor, zeros without a request
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)bmat[i >> 1], 0, live, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_u8)(wb + wave * 4096 + i * 1024), 16, w_voff[i],
                                                 (uint32_t)((block_of(p_pipe) + kfirst) * 128), 0, 2);
    };
    auto dma_t = [&](int hb_pipe, int tb, int i) __attribute__((always_inline)) {
        const int live = uni(hb_pipe < 2 * npair ? -1 : 0);
        const int hb = min(hb_pipe, 2 * npair - 1);
        uint8_t* d = WIDE ? (tb == 0 ? lds.t1 + i * 8192 : i < 2 ? lds.t0 + i * 8192 : lds.t2)
                          : (tb == 0 ? lds.t0 : tb == 1 ? lds.t1 : lds.t2) + i * 8192;
        const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)a_base, 0, live & a_records, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_u8)(d + wave * 1024), 16, t_voff[i],
                                                 (uint32_t)((block_of(hb >> 1) + kfirst) * 256 + (hb & 1) * 128), 0, 0);
    };

    // ---- operands ----
    const int frow = lane & 15, q4 = lane >> 4;
    const int fq = ((q4 & 1) << 1) | (q4 >> 1);
    const uint32_t w_rd = (uint32_t)(wave * 4096 + frow * 128), wkey = (uint32_t)wsx(frow);
    const uint32_t t_rd = (uint32_t)(frow * 128), tkey = (uint32_t)swz(frow);   // (group bases are multiples of 16 rows)
    f32x4 acc[TG][2];
    bf16x8 tf[2][4], wa[2][2];
    u32x4 raw[2][2];                              // [half & 1][fragment]
#pragma unroll
    for (int t = 0; t < TG; ++t) { acc[t][0] = f32x4{0}; acc[t][1] = f32x4{0}; }
#pragma unroll
    for (int t = 0; t < 4; ++t) tf[0][t] = tf[1][t] = __builtin_bit_cast(bf16x8, u32x4{0});
#pragma unroll
    for (int j = 0; j < 2; ++j) wa[0][j] = wa[1][j] = __builtin_bit_cast(bf16x8, u32x4{0});
    auto part_lo = [](int q) { return q * TG / NP; };
    auto read_tokens = [&](int tb, int v) __attribute__((always_inline)) {      // part v % NP of step v / NP
        const int s = v / NP, q = v % NP;
        const uint32_t coff = (uint32_t)(((4 * s + fq) ^ tkey) << 4);
#pragma unroll
        for (int t = part_lo(q); t < part_lo(q + 1); ++t) {
            const uint8_t* b = WIDE ? (tb == 0 ? lds.t1 + t * 2048 : t < 8 ? lds.t0 + t * 2048 : lds.t2 + (t - 8) * 2048)
                                    : (tb == 0 ? lds.t0 : tb == 1 ? lds.t1 : lds.t2) + t * 2048;
            tf[v & 1][t - part_lo(q)] = *reinterpret_cast<const bf16x8*>(b + t_rd + coff);
        }
    };
    auto read_weights = [&](const uint8_t* wb, int h) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
            raw[h][j] = *reinterpret_cast<const u32x4*>(wb + w_rd + j * 2048 + (((4 * h + q4) ^ wkey) << 4));
    };
    // dwords 0 and 1: step 0's weights of this lane, 2 and 3: step 1's
    auto sort_weights = [&](int h, int j) __attribute__((always_inline)) {
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const auto r = __builtin_amdgcn_permlane32_swap(raw[h][j][d], raw[h][j][2 + d], false, false);
            raw[h][j][d] = r[0];
            raw[h][j][2 + d] = r[1];
        }
    };
    auto convert = [&](int h, int s, int part, int set) __attribute__((always_inline)) {   // share `part` of NP of raw[h] -> wa[s]
#pragma unroll
        for (int u = part * 4 / NP; u < (part + 1) * 4 / NP; ++u) {              // 4 weights of fragment u / 2
            const int j = u >> 1, d = u & 1;
            const float scale = rsc[set][SWIGLU ? j : 0];
            if (s == 0 && d == 0) sort_weights(h, j);
            const uint32_t qv = raw[h][j][2 * s + d];
            const f32x2 c0 = __builtin_amdgcn_cvt_pk_f32_fp8(qv, false), c1 = __builtin_amdgcn_cvt_pk_f32_fp8(qv, true);
            u32x4 o = __builtin_bit_cast(u32x4, wa[s][j]);
            o[2 * d] = pack_bf16(c0[0] * scale, c0[1] * scale);
            o[2 * d + 1] = pack_bf16(c1[0] * scale, c1[1] * scale);
            wa[s][j] = __builtin_bit_cast(bf16x8, o);
        }
    };
    auto multiply = [&](int v) __attribute__((always_inline)) {                  // part v % NP of step v / NP
        const int s = v / NP, q = v % NP;
#pragma unroll
        for (int t = part_lo(q); t < part_lo(q + 1); ++t) {
            acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[s][0], tf[v & 1][t - part_lo(q)], acc[t][0], 0, 0, 0);
            acc[t][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[s][1], tf[v & 1][t - part_lo(q)], acc[t][1], 0, 0, 0);
        }
    };

    // Half h of block p: weights out of wb (block p; the next block's out of w_next), tokens out of buffer tb.  Before it: this
    // wave's DMA of its tokens and of everything older has landed and its LDS reads have returned, then everybody's (a
    // bare s_barrier).  After the barrier every wave has left the half before, whose token buffer is t_refill, and (h == 0) this
    // wave block p - 1, whose weight buffer is w_refill.
    auto half = [&](int p, int h, const uint8_t* wb, const uint8_t* w_next, uint8_t* w_refill, int tb, int t_refill, int set) __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(VM) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int v = 0; v < V; ++v) {
            read_tokens(tb, v);
            if (v == NP) read_weights(h == 0 ? wb : w_next, h ^ 1);
            __builtin_amdgcn_sched_barrier(0);
            if (v == 0) {
#pragma unroll
                for (int i = 0; i < NDT; ++i) dma_t(2 * p + h + (WIDE ? 1 : 2), t_refill, i);
                if (h == 0) scales(p + 1, (set + 1) % 3);
                __builtin_amdgcn_sched_barrier(0);
            }
            // the weights of block p + 2: behind the first slots of the half
            if (!WIDE && h == 0) {
                if (V == 2) { dma_w(p + 2, w_refill, 2 * v); dma_w(p + 2, w_refill, 2 * v + 1); }
                else dma_w(p + 2, w_refill, v);
            }
            if (WIDE && v < 2) dma_w(p + 2, w_refill, 2 * h + v);
            multiply((v + V - 1) % V);
            // the step after the one that is multiplied: its share of the conversion
            const int share = (v + V - 1) % NP;
            if (v == 0) convert(h, 0, share, set);
            else if (v <= NP) convert(h, 1, share, set);
            else convert(h ^ 1, 0, share, h == 0 ? set : (set + 1) % 3);
            // two vector instructions are free beside a matrix instruction of 16 cycles, the third costs 4
            const int nm = 2 * (part_lo((v + V - 1) % NP + 1) - part_lo((v + V - 1) % NP));
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (i < nm) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // Prologue: what the halves before the first would have issued, in their order
    if (WIDE) scales(0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) dma_w(0, lds.w0, i);
    __builtin_amdgcn_sched_barrier(0);
    if (WIDE) {
        dma_w(1, lds.w1, 0); dma_w(1, lds.w1, 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NDT; ++i) dma_t(0, 0, i);
        __builtin_amdgcn_sched_barrier(0);
        dma_w(1, lds.w1, 2); dma_w(1, lds.w1, 3);
    } else {
#pragma unroll
        for (int i = 0; i < NDT; ++i) dma_t(0, 0, i);
        __builtin_amdgcn_sched_barrier(0);
        scales(0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) dma_w(1, lds.w1, i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NDT; ++i) dma_t(1, 1, i);
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(VM) : "memory");         // this wave's weights of block 0
    read_weights(lds.w0, 0);
#pragma unroll
    for (int part = 0; part < NP - 1; ++part) convert(0, 0, part, 0);
    // Six halves = three blocks bring the rotations back to where they started: literal buffers in the loop body.
    uint8_t *const w0 = lds.w0, *const w1 = lds.w1, *const w2 = lds.w2;
    constexpr int T1 = 1, T2 = WIDE ? 0 : 2, T3 = WIDE ? 1 : 0, T4 = WIDE ? 0 : 1, T5 = WIDE ? 1 : 2;   // token buffers of halves 1 .. 5
    auto refill = [](int b) { return WIDE ? b ^ 1 : (b + 2) % 3; };
    int p = 0;
    for (; p + 3 <= npair; p += 3) {
        half(p, 0, w0, w1, w2, 0, refill(0), 0);
        half(p, 1, w0, w1, w2, T1, refill(T1), 0);
        half(p + 1, 0, w1, w2, w0, T2, refill(T2), 1);
        half(p + 1, 1, w1, w2, w0, T3, refill(T3), 1);
        half(p + 2, 0, w2, w0, w1, T4, refill(T4), 2);
        half(p + 2, 1, w2, w0, w1, T5, refill(T5), 2);
    }
    if (p < npair) {
        half(p, 0, w0, w1, w2, 0, refill(0), 0);
        half(p, 1, w0, w1, w2, T1, refill(T1), 0);
        if (p + 1 < npair) {
            half(p + 1, 0, w1, w2, w0, T2, refill(T2), 1);
            half(p + 1, 1, w1, w2, w0, T3, refill(T3), 1);
        }
    }
    multiply(V - 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no DMA may land in LDS after the workgroup has gone
    claims.ask();

    // ---- epilogue: a lane holds 4 consecutive columns of one row per accumulator and stores them itself ----
#pragma unroll
    for (int t = 0; t < TG; ++t) {
        const int r = row0 + 16 * t + frow;
        if (r >= row_end) continue;
        if (SWIGLU) {
            const int col = n0 + 16 * wave + 4 * q4;
            if (col < N) *reinterpret_cast<u32x2*>(g.c + (size_t)r * N + col) = epilogue_pack<true>(acc[t][0], acc[t][1]);
        } else {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int col = n0 + 32 * wave + 16 * j + 4 * q4;
                if (col >= N) continue;
                if (SPLIT) *reinterpret_cast<f32x4*>(ks.part + (size_t)(r - ks.row_base) * N + col) = acc[t][j];
                else *reinterpret_cast<u32x2*>(g.c + (size_t)r * N + col) = epilogue_pack<false>(acc[t][j], acc[t][j]);
            }
        }
    }
}

// One-workgroup tiles of an expert with `count` rows: one tile of up to 192 rows if that
// holds them all, else tiles of 128.  The height follows the EXPERT, not the launch: a tile taller
// than its expert stages and multiplies rows that do not exist, and an expert cut into several tiles reads its
// weights once per tile and adds workgroups (the hot expert of a skewed decode batch: 9 x 128 tiles are 4.5 rounds
// of 256 CUs and cost 5).  The tiles of an expert that is cut (above 192 rows) run side by side on one XCD and take
// the weights with plain loads, so that all but the first read of a line come out of that XCD's L2.
// (tiles_of, own_tiles; persistent_tiles: 256-row tiles of such an expert.)  is_cold: whether all its rows are one-workgroup tiles (no
// rem_split)
__host__ __device__ __forceinline__ bool is_cold(const GemmArgs& g, int count) {
    return count <= g.cold_max || (g.pair_rows && count >= PAIR_LO && count <= PAIR_HI);
}
__host__ __device__ __forceinline__ int persistent_tiles(const GemmArgs& g, int count) {
    if (g.rem_split) return (count >> 8) + ((count & 255) > g.cold_max ? 1 : 0);
    return is_cold(g, count) ? 0 : (count + 255) >> 8;
}
// How the CUs are shared between the two kinds of tiles.  Persistent workgroups are bound by the matrix cores, tiles of one workgroup
// mostly by the weights they stream: with every CU at the one kind and then at the other, the memory idles first and the matrix
// cores behind it.  So `full` rounds run on every persistent workgroup, and in the rounds behind those `width` of them go on while
// the CUs of the others fall to the tiles of one workgroup (persistent_plan).  Rounds: as many as the tiles of both kinds take
// together, one of the others counted kStreamCost hundredths (of 36 us beside persistent tiles and 50 among its like, where a persistent
// one takes 60: DeepSeek-V2-Lite, 4096 tokens, gate and up), rounded down: what is left of the others then runs on every CU, in
// small pieces.  The places that the persistent tiles leave free in those rounds are taken in the longest stretch of the narrowest
// strip that holds nearly all of them, of whole 32 CUs: the tiles that an XCD has at a time then stay whole blocks of 4 M tiles,
// which share their panels.
// A last round of a few tiles costs as much as a full one.  Where the others do not fill the CUs that it leaves over, or fill them up
// to twice with tall ones among them (two of which, one behind the other, take longer than a persistent tile), and cut into pieces its
// tiles make the sum of both kinds' rounds shorter, it goes to workgroups of one tile: as 128-row halves, or, where no others share the
// round, in as many as three or four pieces that fit in it (next to others, which take as long as a half, they end no sooner).  Every
// workgroup evaluates all this on the same offsets[].
// Layers, us, every CU at the persistent tiles first and one workgroup launched per tile of the others -> this (and Claims): DeepSeek-V2-Lite
// 1400 / 2400 / 4096 tokens 379 / 483 / 662 -> 342 / 458 / 635, DeepSeek-V2-236B 1500 / 4000 / 8000 1594 / 2238 / 3384 -> 1479 / 2054 / 3150, DeepSeek-V3
// 6000 5296 -> 5195.  Mixtral-8x22B, 8 experts, goes by how the rounds fall out: 640 / 760 / 850 1121 / 1266 / 1300 -> 1042 / 1130 / 1161, 820 / 920 / 1100 /
// 1200 1323 / 1353 / 1451 / 1561 -> 1304 / 1356 / 1453 / 1561; there the down projection has 96 to 144 tiles of 256 rows and 144 to 192
// others, and without the count of tall ones (kTwoTall) it was 22 to 39 us longer: 1336 / 1393 / 1491 / 1598.
constexpr int kStreamCost = 50, kTwoTall = 150, kMostAside = 128;
struct RoundCost { int keep, move, pieces; };       // hundredths of a round, with the last one persistent / in so many pieces a tile
__host__ __device__ __forceinline__ RoundCost round_cost(int total, int own, bool tall, int cus) {
    const int whole = 100 * ((total + cus - 1) / cus), shared = (100 * total + kStreamCost * own) / cus, tail = total % cus;
    RoundCost c{whole > shared ? whole : shared, 72 * ((own + 2 * tail + cus - 1) / cus), 2};
    if (tall && total < cus && own > cus - total && own <= 2 * (cus - total)) c.keep = kTwoTall;
    if (own == 0 && 3 * tail <= cus) { c.move = 54; c.pieces = 3; }
    if (own == 0 && 4 * tail <= cus) { c.move = 44; c.pieces = 4; }
    c.move += 100 * (total / cus);
    return c;
}
__host__ __device__ __forceinline__ int piece_rows(int pieces) { return pieces == 2 ? 128 : pieces == 3 ? 96 : 64; }
struct Tail { int tiles, pieces; };
__device__ __forceinline__ Tail tail_of(const GemmArgs& g, int total, int own, bool tall) {
    if (g.tail_cus <= 0) return Tail{0, 2};
    const int tail = total % g.tail_cus;
    if (tail == 0) return Tail{0, 2};
    const RoundCost c = round_cost(total, own, tall, g.tail_cus);
    return Tail{c.move < c.keep ? tail : 0, c.pieces};
}
struct PersistentPlan { int full, width; };
// of `grid` persistent workgroups with `total` tiles.  (Less than a round of tiles: an eighth of them on each XCD; all of an XCD's places
// in a row, as in whole rounds, left the memory paths of the others idle: Mixtral-8x22B, 512 tokens, 1012 us with that and 988 with this.)
__device__ __forceinline__ PersistentPlan persistent_plan(const GemmArgs& g, int total, int own, int grid) {
    if (total <= grid) return PersistentPlan{0, (total + 7) / 8 * 8};
    PersistentPlan p{0, grid};
    if (own == 0 || grid < g.tail_cus) return p;
    const int rounds = max((total + grid - 1) / grid, (total + own * kStreamCost / 100) / grid), spare = rounds * grid - total;
    int most = 0;
#pragma unroll
    for (int c = kMostAside; c >= 32; c -= 32) {
        const int b = min(rounds, spare / c);
        if (c * b >= max(most, 1) && c < grid) {
            most = c * b;
            p = PersistentPlan{rounds - b, grid - c};
        }
    }
    return p;
}

template <bool PAIR>   // whether an expert of PAIR_LO .. PAIR_HI rows is cut in the middle (bf16 weights)
__host__ __device__ __forceinline__ int tiles_of(int count) {
    constexpr int SINGLE = 192;   // rows that one tile may hold
    if (count <= SINGLE) return count > 0 ? 1 : 0;
    // bf16 weights: an expert of 257 to 384 rows is cut in the middle, into two tiles of the 192-row body that run
    // side by side on one XCD and share the weights through its L2: 320 rows are 2 x 160 rows of MFMA work, where
    // two 256-row tiles of the persistent body multiply 512 and three 128-row tiles read the weights three times.
    // Mixtral-8x22B shapes, 8 experts of 288 / 320 / 384 rows: gate/up 1.31 / 1.29 / 1.30 -> 1.07 / 1.13 / 1.17 ms,
    // down projection within 4 % either way; up to 256 rows one tile of the persistent body stays better (224
    // rows: 0.82 against 1.01 ms).
    if (PAIR && count > PAIR_LO - 1 && count <= PAIR_HI) return 2;
    return (count + 127) >> 7;
}
// rows of either tile of such a pair (the first tile holds whole 16-row groups)
__device__ __forceinline__ int half_rows(int count) { return ((count + 1) / 2 + 15) & ~15; }

// One-workgroup tiles of an expert with `count` rows in a call of both kinds
template <bool W8>
__host__ __device__ __forceinline__ int own_tiles(const GemmArgs& g, int c) {
    if (g.rem_split) c &= 255;      // the rows the persistent body's full tiles leave over
    return (g.rem_split ? c > g.cold_max : !is_cold(g, c)) ? 0 : tiles_of<!W8>(c);
}

// Whether the tallest of them has more than kTallRows: two in a row then outlast a persistent tile by so much that its halves in front of or
// behind one are the shorter way (round_cost).  DeepSeek-V3's dense MLP, fp8, one such tile a column: 400 / 420 / 440 tokens (144 / 164 / 184 rows)
// with the persistent tiles kept 354 / 375 / 391 us, in halves 363 / 373 / 382.
constexpr int kTallRows = 150;
template <bool W8>
__device__ __forceinline__ bool has_tall_tile(const GemmArgs& g, int c) {
    const int tiles = own_tiles<W8>(g, c), rows = g.rem_split ? c & 255 : c;
    return tiles == 1 ? rows > kTallRows : !W8 && tiles == 2 && rows >= PAIR_LO && half_rows(rows) > kTallRows;
}

// The shared expert's rows and its tiles of either kind in a call of both, all 0 without one
struct SharedTiles { int first, end, own, persistent; bool tall; };
template <bool W8>
__host__ __device__ __forceinline__ SharedTiles shared_tiles_of(const GemmArgs& g, int first, int end) {
    return SharedTiles{first, end, own_tiles<W8>(g, end - first) * g.n_tiles_n, persistent_tiles(g, end - first) * g.n_tiles_n,
                       has_tall_tile<W8>(g, end - first)};
}
// The most tiles of each kind that up to `rows` rows can have (fewer rows can have more: 200 rows one 256-row tile, 300 none)
template <bool W8>
inline SharedTiles shared_tiles_bound(const GemmArgs& g, int rows) {
    return SharedTiles{0, rows, (!W8 && rows >= PAIR_LO ? 2 : 1) * g.n_tiles_n, rows > g.cold_max ? ((rows + 255) >> 8) * g.n_tiles_n : 0, false};
}

// sum over the experts of f(count) (every thread gets it; two barriers)
template <int NT, typename F>
__device__ __forceinline__ int sum_over_experts(const GemmArgs& g, int tid, int* s_wtot, F f) {
    int v = 0;
    for (int e = tid; e < g.E; e += NT) v += f(g.offsets[e + 1] - g.offsets[e]);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
    __syncthreads();                 // whoever read s_wtot before has done so
    if ((tid & 63) == 0) s_wtot[tid >> 6] = v;
    __syncthreads();
    int tot = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) tot += s_wtot[w];
    return tot;
}

// ---- bf16 weight streamer in the persistent body's summation order: tiles of up to 192 rows ----
//
// The fp8 streamers' way of moving data for bf16 weights: weights and token rows reach LDS by DMA in the persistent
// kernel's layout of a 64-k stage (128-byte rows, chunk c of row r at c ^ swz(r)), and every matrix instruction gets
// the k values the persistent body gives it, in the same lanes, so a row's bits do not depend on who computes it.
// No staging registers and no LDS stores, so every operand of a stage can be requested up front.  Up to 64 rows the 8
// waves split the tile's 256 weight rows and each multiplies all token rows; above, two sets of 4 waves take half of
// the token groups each (4 + TG / 2 operand reads per k-step for 2 TG matrix instructions, where 8 x 1 waves need
// 2 + TG for as many).  Three weight buffers of 32 KiB keep two stages of weights in flight; token rows (up to
// 24 KiB per stage, out of L2) have two buffers and travel one stage ahead, issued first in a stage so that the wait
// before the next stage's barrier leaves only the 4 weight instructions behind them in flight.
// Weight row R of a stage (LDS row R, brought by wave R / 32): column n0 + R; gate and up: gate column n0 + R,
// R < 128, up column n0 + R - 128 above.  k starts at stage 0 unless the kernel has the call to itself.
// NW waves: 8, or 4 with half the weight rows (down projection, up to 64 rows)
template <int TG, bool SWIGLU, bool SHARED, typename C, int NW = 8>   // TG: 16-row token groups multiplied (1 .. 12); SHARED: another tile reads these weights
__device__ __forceinline__ void stream16_tile(const GemmArgs& g, uint8_t* w0, uint8_t* w1, uint8_t* w2, uint8_t* t0, uint8_t* t1,
                                              int e, int row0, int row_end, int n_tile, C& claims) {
    constexpr int NBLK = SWIGLU ? 128 : 32 * NW;
    constexpr int WM = TG >= 5 ? 2 : 1;           // sets of waves across the token groups
    constexpr int TH = (TG + WM - 1) / WM;        // token groups per wave (an odd TG: the second set's last group is padding)
    constexpr int NF = 2 * WM;                    // 16-row weight fragments per wave
    constexpr int NDW = 4;                        // weight DMA instructions per wave and stage
    constexpr int NDT = (2 * TG + NW - 1) / NW;   // token DMA instructions per wave and stage (8 rows each; 8 NW rows per round of the waves)
    static_assert(NW == 8 || (NW == 4 && !SWIGLU && TG <= 4), "halves");
    static_assert(TG >= 1 && TG <= 12, "token rows staged");
    const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
    const int wm = WM == 2 ? wave >> 2 : 0, wn = WM == 2 ? wave & 3 : wave;
    const int n0 = n_tile * NBLK;
    const int K = g.K, N = g.N;
    const int nk = K / BK;
    const int prot = k_rotation<false>(n0 / (SWIGLU ? 128 : 256), nk);

    // ---- DMA coordinates: lane l supplies row +l/8 of an instruction's 8 rows and the 16 bytes that belong at physical chunk l%8 ----
    const int lr = lane >> 3, pp = lane & 7;
    uint32_t w_voff[NDW], t_voff[NDT];
    const uint8_t* bmat = uni_ptr((SWIGLU && wave >= 4) ? g.b1[e] : g.b0[e]);
#pragma unroll
    for (int i = 0; i < NDW; ++i) {               // LDS rows 32 wave + 8 i + lr
        const int R = 32 * wave + 8 * i + lr;
        w_voff[i] = (uint32_t)min(n0 + (SWIGLU ? R & 127 : R), N - 1) * (uint32_t)(K * 2) + (uint32_t)((pp ^ swz(R)) << 4);
    }
    const uint8_t* a_base = reinterpret_cast<const uint8_t*>(g.a) + (g.row_map ? (size_t)0 : (size_t)row0 * K * 2);
    const int a_records = g.row_map ? (int)(uint32_t)g.a_bytes : (row_end - row0) * K * 2;
#pragma unroll
    for (int i = 0; i < NDT; ++i) {               // token rows 8 NW i + 8 wave + lr; rows past the tile's last: zeros, no request
        const int tr = 8 * NW * i + 8 * wave + lr;
        const int r = min(row0 + tr, row_end - 1);
        const int src = g.row_map ? ((gptr_i32)(uintptr_t)g.row_map)[r] : r - row0;
        t_voff[i] = (uint32_t)src * (uint32_t)(K * 2) + (uint32_t)((pp ^ swz(tr)) << 4);
        if (row0 + tr >= row_end || (g.row_map && (unsigned)src >= (unsigned)g.a_rows)) t_voff[i] = 0xfffffff0u;
    }
    auto stage_off = [&](int kt_pipe) {           // byte offset of pipeline stage kt_pipe in a row (the last one again past the end)
        int kt = min(kt_pipe, nk - 1) + prot;
        kt = kt >= nk ? kt - nk : kt;
        return (uint32_t)(kt * BK * 2);
    };
    auto dma_w = [&](int kt_pipe, uint8_t* wb, int i) __attribute__((always_inline)) {
        const int live = uni(kt_pipe < nk ? -1 : 0);   // past the end: an empty descriptor, zeros without a request
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)bmat, 0, live, 0x00020000);
        // (non-temporal unless a neighbour on this XCD reads the same lines and should find them in its L2)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_u8)(wb + wave * 4096 + i * 1024), 16, w_voff[i], stage_off(kt_pipe), 0, SHARED ? 0 : 2);
    };
    auto dma_t = [&](int kt_pipe, uint8_t* tb, int i) __attribute__((always_inline)) {
        const int live = uni(kt_pipe < nk ? -1 : 0);
        const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)a_base, 0, live & a_records, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_u8)(tb + (8 * NW * i + 8 * wave) * ROW_B), 16, t_voff[i], stage_off(kt_pipe), 0, 0);
    };

    // ---- operand coordinates: fragment j of the wave is LDS rows wrow(j) .. + 15 ----
    const int frow = lane & 15, q = lane >> 4;
    const int fq = ((q & 1) << 1) | (q >> 1);
    const uint32_t fkey = (uint32_t)swz(frow);
    auto wrow = [&](int j) { return SWIGLU ? (j / WM) * 128 + 16 * WM * wn + 16 * (j % WM) : 32 * WM * wn + 16 * j; };
    const uint32_t w_rd = (uint32_t)((wrow(0) + frow) * ROW_B), t_rd = (uint32_t)((16 * TH * wm + frow) * ROW_B);
    f32x4 acc[TH][NF];
#pragma unroll
    for (int t = 0; t < TH; ++t)
#pragma unroll
        for (int j = 0; j < NF; ++j) acc[t][j] = f32x4{0};

    // Stage kt is multiplied out of weight buffer kt % 3 and token buffer kt % 2.  Before it: this wave's DMA of its
    // tokens (issued first in the stage before) and of everything older has landed, its LDS reads have returned, then
    // everybody's (a bare s_barrier).  After the barrier every wave has left stage kt - 1: its token buffer takes
    // stage kt + 1, its weight buffer stage kt + 2.
    // Every operand of the stage is requested up front (4 + TG / 2 or 2 + TG reads per k-step): the matrix instructions
    // then run behind the LDS pipeline instead of waiting out its latency one token group at a time.
    bf16x8 wa0[NF], tf0[TH], wa1[NF], tf1[TH];
    auto read_step = [&](const uint8_t* wb, const uint8_t* tb, int s, bf16x8 (&wa)[NF], bf16x8 (&tf)[TH]) __attribute__((always_inline)) {
        const uint32_t coff = (uint32_t)(((4 * s + fq) ^ fkey) << 4);
#pragma unroll
        for (int j = 0; j < NF; ++j) wa[j] = *reinterpret_cast<const bf16x8*>(wb + w_rd + (wrow(j) - wrow(0)) * ROW_B + coff);
#pragma unroll
        for (int t = 0; t < TH; ++t) tf[t] = *reinterpret_cast<const bf16x8*>(tb + t_rd + t * 16 * ROW_B + coff);
    };
    // (with 2 of the 4 instructions of the weight DMA after the first token group)
    auto mfma_step = [&](const bf16x8 (&wa)[NF], const bf16x8 (&tf)[TH], int kt_dma, uint8_t* w_refill, int i0) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TH; ++t) {
#pragma unroll
            for (int j = 0; j < NF; ++j) acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[j], tf[t], acc[t][j], 0, 0, 0);
            if (t == 0) { dma_w(kt_dma, w_refill, i0); dma_w(kt_dma, w_refill, i0 + 1); }
        }
    };
    auto stage = [&](int kt, const uint8_t* wb, const uint8_t* tb, uint8_t* w_refill, uint8_t* t_refill) __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(NDW) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < NDT; ++i) dma_t(kt + 1, t_refill, i);
        __builtin_amdgcn_sched_barrier(0);
        read_step(wb, tb, 0, wa0, tf0);
        read_step(wb, tb, 1, wa1, tf1);
        __builtin_amdgcn_sched_barrier(0);
        mfma_step(wa0, tf0, kt + 2, w_refill, 0);
        mfma_step(wa1, tf1, kt + 2, w_refill, 2);
        __builtin_amdgcn_sched_barrier(0);      // (or the matrix instructions sink below the next stage's barrier, behind its reads)
    };
    // Prologue: the tokens of stage 0 between the weights of stages 0 and 1, so that the first wait (all but the 4
    // youngest instructions) covers what stage 0 reads, as in the steady state.
#pragma unroll
    for (int i = 0; i < NDW; ++i) dma_w(0, w0, i);
#pragma unroll
    for (int i = 0; i < NDT; ++i) dma_t(0, t0, i);
#pragma unroll
    for (int i = 0; i < NDW; ++i) dma_w(1, w1, i);
    // Six stages bring both rotations back to where they started: literal buffers in the loop body.
    int kt = 0;
    for (; kt + 6 <= nk; kt += 6) {
        stage(kt, w0, t0, w2, t1);
        stage(kt + 1, w1, t1, w0, t0);
        stage(kt + 2, w2, t0, w1, t1);
        stage(kt + 3, w0, t1, w2, t0);
        stage(kt + 4, w1, t0, w0, t1);
        stage(kt + 5, w2, t1, w1, t0);
    }
    if (kt < nk) stage(kt, w0, t0, w2, t1);
    if (kt + 1 < nk) stage(kt + 1, w1, t1, w0, t0);
    if (kt + 2 < nk) stage(kt + 2, w2, t0, w1, t1);
    if (kt + 3 < nk) stage(kt + 3, w0, t1, w2, t0);
    if (kt + 4 < nk) stage(kt + 4, w1, t0, w0, t1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no DMA may land in LDS after the workgroup has gone
    claims.ask();

    // ---- epilogue: a lane holds 4 consecutive columns of one row per accumulator and stores them itself ----
#pragma unroll
    for (int t = 0; t < TH; ++t) {
        const int r = row0 + 16 * (TH * wm + t) + frow;
        if (r >= row_end) continue;
#pragma unroll
        for (int j = 0; j < (SWIGLU ? WM : NF); ++j) {
            const int col = n0 + wrow(j) + 4 * q;
            if (col < N) *reinterpret_cast<u32x2*>(g.c + (size_t)r * N + col) = epilogue_pack<SWIGLU>(acc[t][j], acc[t][SWIGLU ? WM + j : j]);
        }
    }
}

template <bool SWIGLU, bool SHARED, typename C>
__device__ __forceinline__ void stream16(const GemmArgs& g, uint8_t* w0, uint8_t* w1, uint8_t* w2, uint8_t* t0, uint8_t* t1, int e,
                                         int row0, int row_end, int n_tile, C& claims) {
    const int tg = (row_end - row0 + 15) >> 4;
    switch (tg) {
#define MOE_S16_CASE(n) case n: stream16_tile<n, SWIGLU, SHARED>(g, w0, w1, w2, t0, t1, e, row0, row_end, n_tile, claims); break;
    MOE_S16_CASE(1) MOE_S16_CASE(2) MOE_S16_CASE(3) MOE_S16_CASE(4) MOE_S16_CASE(5) MOE_S16_CASE(6)
    MOE_S16_CASE(7) MOE_S16_CASE(8) MOE_S16_CASE(9) MOE_S16_CASE(10) MOE_S16_CASE(11)
#undef MOE_S16_CASE
    default: stream16_tile<12, SWIGLU, SHARED>(g, w0, w1, w2, t0, t1, e, row0, row_end, n_tile, claims); break;
    }
}

template <bool SWIGLU, typename C>
__device__ __forceinline__ void stream8x(const GemmArgs& g, const TileLds& lds, int e, int row0, int row_end, int n_tile, bool rotate,
                                         C& claims) {
    switch ((row_end - row0 + 15) >> 4) {
#define MOE_S8X_CASE(n) case n: stream8x_tile<n, SWIGLU>(g, lds, e, row0, row_end, n_tile, rotate, claims); break;
    MOE_S8X_CASE(1) MOE_S8X_CASE(2) MOE_S8X_CASE(3) MOE_S8X_CASE(4) MOE_S8X_CASE(5) MOE_S8X_CASE(6)
    MOE_S8X_CASE(7) MOE_S8X_CASE(8) MOE_S8X_CASE(9) MOE_S8X_CASE(10) MOE_S8X_CASE(11)
#undef MOE_S8X_CASE
    default: stream8x_tile<12, SWIGLU>(g, lds, e, row0, row_end, n_tile, rotate, claims); break;
    }
}

// the expert that M tile q belongs to: pref[e] <= q < pref[e + 1]
struct ExpertAt { int e, first, tiles; };
__device__ __forceinline__ ExpertAt expert_at(const int* pref, int E, int q) {
    const int lane = threadIdx.x & 63;
    for (int e0 = 0;; e0 += 64) {
        const int i = min(e0 + lane, E - 1), a = pref[i], b = pref[i + 1];
        const uint64_t m = __ballot(a <= q && q < b);
        if (m != 0 || e0 + 64 >= E) {
            const int l = m != 0 ? (int)__builtin_ctzll(m) : 0;
            const int first = __builtin_amdgcn_readlane(a, l), end = __builtin_amdgcn_readlane(b, l);
            return ExpertAt{min(e0 + l, E - 1), first, end - first};
        }
    }
}

// The scan of a call whose experts may be cut lower: `cut` rows above which an expert is cut into tiles of equal height (neighbours on one
// XCD, which share its weights through the L2), 0: as tiles_of says.  A call of few tiles, a down projection of a few experts, leaves CUs
// without any while its tallest tiles, bound by the matrix cores above about 100 rows, take longest: cut as long as every tile has a
// CU.  Every workgroup finds the same.  Mixtral-8x22B, layers of 256 / 350 tokens (tallest experts 181 and 250 rows, 192 tiles for 256 CUs)
// 847 / 915 -> 831 / 899 us, of fewer tokens the same.  The three ways to count are scanned side by side: as a pass of its own in front of
// the scan, where the counts of Mixtral-8x7B at 256 to 400 tokens (66 to 110 rows) are not cut, it cost 2 to 5 of 570 us.
// At most NT experts; s_wtot: 3 NT / 64.
template <int NT>
__device__ __forceinline__ int cut_prefix_scan(const GemmArgs& g, int tid, int* s_wtot, ExpertOfThread& mine, int& cut) {
    const int lane = tid & 63, wave = tid >> 6;
    mine = ExpertOfThread{0, 0, 0, 0};
    if (tid < g.E) {
        mine.o0 = g.offsets[tid];
        mine.o1 = g.offsets[tid + 1];
    }
    const int c = mine.o1 - mine.o0, n[3] = {(c + 95) / 96, (c + 127) / 128, tiles_of<true>(c)};
    int inc[3] = {n[0], n[1], n[2]};
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int o = __shfl_up(inc[j], d);
            if (lane >= d) inc[j] += o;
        }
    }
#pragma unroll
    for (int j = 0; j < 3; ++j)
        if (lane == 63) s_wtot[3 * wave + j] = inc[j];
    __syncthreads();
    int before[3] = {0, 0, 0}, all[3] = {0, 0, 0};
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            if (w < wave) before[j] += s_wtot[3 * w + j];
            all[j] += s_wtot[3 * w + j];
        }
    }
    const bool low = (long)all[0] * g.n_tiles_n <= g.cut_cus, high = (long)all[1] * g.n_tiles_n <= g.cut_cus;
    cut = low ? 96 : high ? 128 : 0;
    mine.mt = low ? n[0] : high ? n[1] : n[2];
    mine.start = (low ? before[0] + inc[0] : high ? before[1] + inc[1] : before[2] + inc[2]) - mine.mt;
    return low ? all[0] : high ? all[1] : all[2];
}

// One workgroup per (M tile, N tile), in calls without persistent tiles (few rows per expert, odd K).  (tile_body is its counterpart in calls
// of both kinds: which rows a tile has, and which streamer computes them, is the same there, since a row's bits follow from it.)
// CUT: rows are cut lower where that fills the CUs (cut_prefix_scan), in an instantiation of its own: the other calls, DeepSeek-V2-Lite of 256 to
// 500 tokens, were 1 to 2 % slower with the few instructions in front of their tiles.
template <int WN, bool SWIGLU, bool W8, bool CUT>
__global__ __launch_bounds__(128 * WN) void grouped_gemm_kernel(GemmPair pair_of) {
    constexpr int NT = 128 * WN;
    static_assert(!(W8 && CUT), "fp8 rows are not cut: their sums follow the tile");
    // Three weight arrays of 32 KiB and token arrays of 16 KiB (fp8 weights: three, 128 rows; the second one 24 KiB)
    // or 24 KiB (bf16: two, 192 rows) -- the buffers of the weight streamers, written by DMA, as separate objects so
    // that a read of one waits for no DMA into another; gemm_tile's two stages (up to 128 token rows + 256 weight
    // rows) are two pairs of them.  fp8 tiles of 129 to 192 rows have two token buffers, the second array and the
    // first and third together.
    constexpr int TB = W8 ? 128 * ROW_B : 192 * ROW_B;
    __shared__ __attribute__((aligned(1024))) uint8_t lw0[S8_WBYTES];
    __shared__ __attribute__((aligned(1024))) uint8_t lw1[S8_WBYTES];
    __shared__ __attribute__((aligned(1024))) uint8_t lw2[S8_WBYTES];
    __shared__ __attribute__((aligned(1024))) uint8_t lt0[TB];
    __shared__ __attribute__((aligned(1024))) uint8_t lt1[192 * ROW_B];
    __shared__ __attribute__((aligned(1024))) uint8_t lt2[W8 ? TB : 16];
    static_assert(S8_TROWS * 256 <= 128 * ROW_B && S8_WBYTES == BN_ROWS * ROW_B, "regions of a streamer buffer");
    auto stage = [&](int i) { return Stage{i ? lt1 : lt0, i ? lw1 : lw0, i ? lw1 : lw0}; };
    const SBuf sb0{lw0, lt0}, sb1{lw1, lt1}, sb2{lw2, lt2};
    const TileLds lds{lw0, lw1, lw2, lt0, lt1, lt2};
    __shared__ int s_pref[MAX_E + 1];
    __shared__ int s_wtot[(CUT ? 3 : 1) * (NT / 64)];
    __shared__ int s_sel[5];
    const int tid = threadIdx.x;

    int v = dealt_tile(blockIdx.x & 7, blockIdx.x >> 3);
    OneTile one;
    const bool in_front = v < pair_of.shared_tiles;
    if (!in_front) v -= pair_of.shared_tiles;

    // ---- M-tile prefix over experts ----
    const GemmArgs& g = pair_of.p[in_front ? 1 : 0];
    ExpertOfThread mine;
    int cut = 0, run;
    if constexpr (CUT) run = cut_prefix_scan<NT>(g, tid, s_wtot, mine, cut);
    else run = mtile_prefix_scan<NT>(g, tid, s_pref, s_wtot, mine, [](int c) { return tiles_of<!W8>(c); }, [](int, int, int) {});
    if (v >= run * g.n_tiles_n) return;
    const bool s8_ok = !g.row_map || g.a_bytes < (1ull << 32);   // (the weight streamer addresses gathered rows with 32-bit offsets)
    const int q = v / g.n_tiles_n;  // global M-tile number
    // find e with prefix[e] <= q < prefix[e+1].  Up to NT experts every thread still holds its own
    // expert's prefix, tile count and row range: the one that owns q publishes them (one barrier,
    // no search, no second trip to memory for the offsets).  More experts: binary search in LDS.
    if (CUT || g.E <= NT) {
        if (tid < g.E && mine.start <= q && q < mine.start + mine.mt) {
            s_sel[0] = tid; s_sel[1] = mine.start; s_sel[2] = mine.mt; s_sel[3] = mine.o0; s_sel[4] = mine.o1;
        }
        __syncthreads();
    } else {
        if (tid == 0) s_pref[g.E] = run;
        __syncthreads();
        int lo = 0, hi = g.E;
        while (hi - lo > 1) {
            int mid = (lo + hi) >> 1;
            if (s_pref[mid] <= q) lo = mid; else hi = mid;
        }
        if (tid == 0) {
            s_sel[0] = lo; s_sel[1] = s_pref[lo]; s_sel[2] = s_pref[lo + 1] - s_pref[lo];
            s_sel[3] = g.offsets[lo]; s_sel[4] = g.offsets[lo + 1];
        }
        __syncthreads();
    }
    const int e = uni(s_sel[0]);
    const int pe = uni(s_sel[1]);
    const int mt_e = uni(s_sel[2]);
    int m_tile, n_tile;
    tile_in_expert(v - pe * g.n_tiles_n, mt_e, g.n_tiles_n, m_tile, n_tile);
    const int row_end = uni(s_sel[4]);
    const int first_row = uni(s_sel[3]);
    if (W8 && s8_ok) {
        // fp8 weights: the weight streamers.  Up to 64 rows where no persistent tile's summation order has to be matched: the
        // form that reads a lane's 16 weights at once.  Everything else -- up to 192 rows; what an expert's full 256-row
        // tiles leave over; 128-row slices of larger experts when the kernel serves the call by itself -- in the order of
        // persistent tiles.
        const int r0 = first_row + (mt_e > 1 ? m_tile * 128 : 0), r1 = mt_e > 1 ? min(row_end, r0 + 128) : row_end;
        const int rows = r1 - r0;
        if (g.alone && mt_e == 1 && rows <= 64) {
            if (rows <= 16) stream8_tile<1, SWIGLU>(g, sb0, sb1, sb2, e, r0, r1, n_tile, one);
            else if (rows <= 32) stream8_tile<2, SWIGLU>(g, sb0, sb1, sb2, e, r0, r1, n_tile, one);
            else if (rows <= 48) stream8_tile<3, SWIGLU>(g, sb0, sb1, sb2, e, r0, r1, n_tile, one);
            else stream8_tile<4, SWIGLU>(g, sb0, sb1, sb2, e, r0, r1, n_tile, one);
        } else {
            stream8x<SWIGLU>(g, lds, e, r0, r1, n_tile, g.alone, one);
        }
        return;
    }
    // The rows of this workgroup: the expert's (one tile: up to 192 rows), one half of an
    // expert of PAIR_LO .. PAIR_HI rows (bf16), or a 128-row slice.
    const int rows_e = row_end - first_row;
    const bool pair = !W8 && rows_e >= PAIR_LO && rows_e <= PAIR_HI;
    const int slice = cut ? ((rows_e + mt_e - 1) / mt_e + 15) & ~15 : pair ? half_rows(rows_e) : 128;
    const int t0 = mt_e > 1 ? first_row + m_tile * slice : first_row, t1 = mt_e > 1 ? min(row_end, t0 + slice) : row_end;
    if (CUT && t0 >= t1) return;    // (heights are whole groups of 16)
    if (!W8 && s8_ok) {
        // bf16 weights: the weight streamer in the persistent body's order
        if (mt_e == 1) stream16<SWIGLU, false>(g, lw0, lw1, lw2, lt0, lt1, e, t0, t1, n_tile, one);
        else stream16<SWIGLU, true>(g, lw0, lw1, lw2, lt0, lt1, e, t0, t1, n_tile, one);
        return;
    }
    // 4 GiB of gathered rows or more: the register-staged body, which addresses them with 64-bit offsets, 128 rows
    // at a time
    if (t1 - t0 <= 64) {
        gemm_tile<1, WN, SWIGLU, W8, true>(g, stage(0), stage(1), e, t0, t1, n_tile);
    } else if (mt_e == 1) {
        gemm_tile<2, WN, SWIGLU, W8, true>(g, stage(0), stage(1), e, t0, min(t1, t0 + 128), n_tile);
        if (t1 - t0 > 128) {
            __syncthreads();
            gemm_tile<2, WN, SWIGLU, W8, true>(g, stage(0), stage(1), e, t0 + 128, t1, n_tile);
        }
    } else {
        gemm_tile<2, WN, SWIGLU, W8, false>(g, stage(0), stage(1), e, t0, min(t1, t0 + 128), n_tile);
        if (t1 - t0 > 128) {
            __syncthreads();
            gemm_tile<2, WN, SWIGLU, W8, false>(g, stage(0), stage(1), e, t0 + 128, t1, n_tile);
        }
    }
}

// ---- half tiles: bf16 down projections of few tiles ----
//
// A down projection of few experts, or of small ones, has a fraction of a round or little more than one of 256-column tiles: the CUs left
// over idle, and so does the memory.  Here a tile is 128 columns x up to 64 rows, a workgroup 4 waves with half the LDS, two of which
// run on a CU: as many bytes in flight, twice as many pieces to fill the CUs with, and one's start and end beside the other's loop.  Experts
// above 64 rows are cut evenly into neighbours that share the weights through their XCD's L2.  The bits are those of whole tiles.  (Rule and
// figures: half_tiles_pay.)
constexpr int HALF_ROWS = 64;
inline __host__ __device__ int half_tiles_of(int count) { return (count + HALF_ROWS - 1) / HALF_ROWS; }
__global__ __launch_bounds__(256, 2) void grouped_gemm_half_kernel(GemmPair pair_of) {
    constexpr int NT = 256;
    __shared__ __attribute__((aligned(1024))) uint8_t lw0[S8_WBYTES / 2];
    __shared__ __attribute__((aligned(1024))) uint8_t lw1[S8_WBYTES / 2];
    __shared__ __attribute__((aligned(1024))) uint8_t lw2[S8_WBYTES / 2];
    __shared__ __attribute__((aligned(1024))) uint8_t lt0[HALF_ROWS * ROW_B];
    __shared__ __attribute__((aligned(1024))) uint8_t lt1[HALF_ROWS * ROW_B];
    __shared__ int s_pref[MAX_E + 1];
    __shared__ int s_wtot[NT / 64];
    const int tid = threadIdx.x;
    int v = dealt_tile(blockIdx.x & 7, blockIdx.x >> 3);
    const bool in_front = v < pair_of.shared_tiles;
    if (!in_front) v -= pair_of.shared_tiles;
    const GemmArgs& g = pair_of.p[in_front ? 1 : 0];
    ExpertOfThread mine;
    const int run = mtile_prefix_scan<NT>(g, tid, s_pref, s_wtot, mine, half_tiles_of, [](int, int, int) {});
    if (v >= run * g.n_tiles_n) return;
    if (tid == 0) s_pref[g.E] = run;
    __syncthreads();
    const ExpertAt x = expert_at(s_pref, g.E, v / g.n_tiles_n);
    const int first_row = uni(g.offsets[x.e]), rows_e = uni(g.offsets[x.e + 1]) - first_row;
    int m_tile, n_tile;
    tile_in_expert(v - x.first * g.n_tiles_n, x.tiles, g.n_tiles_n, m_tile, n_tile);
    const int slice = ((rows_e + x.tiles - 1) / x.tiles + 15) & ~15;
    const int r0 = first_row + m_tile * slice, r1 = min(first_row + rows_e, r0 + slice);
    if (r0 >= r1) return;                        // (heights are whole groups of 16)
    OneTile one;
    switch ((x.tiles > 1 ? 4 : 0) + ((r1 - r0 + 15) >> 4)) {
#define MOE_HALF_CASE(n, shared) case n + 4 * shared: stream16_tile<n, false, shared, OneTile, 4>(g, lw0, lw1, lw2, lt0, lt1, x.e, r0, r1, n_tile, one); break;
    MOE_HALF_CASE(1, false) MOE_HALF_CASE(2, false) MOE_HALF_CASE(3, false) MOE_HALF_CASE(4, false)
    MOE_HALF_CASE(1, true) MOE_HALF_CASE(2, true) MOE_HALF_CASE(3, true) MOE_HALF_CASE(4, true)
#undef MOE_HALF_CASE
    }
}

// ---- the combine of a few tokens at the end of their down projection ----
//
// tail.arrivals: a counter per column tile, minus the waves that will write its columns (an expert with rows each, and the
// shared expert); the dispatch of the call sets them.  The wave that brings a counter to zero finds every expert's columns
// written and adds them up: no wave waits for another.  What waves on other XCDs read leaves and arrives past the L2 of an XCD
// (relaxed atomics at agent scope), a wave's stores being complete before it counts itself.
__device__ __forceinline__ u32x4 load_shared_16(const uint16_t* p) {
    const uint64_t* q = reinterpret_cast<const uint64_t*>(p);
    const u32x2 a = __builtin_bit_cast(u32x2, __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    const u32x2 b = __builtin_bit_cast(u32x2, __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    return u32x4{a[0], a[1], b[0], b[1]};
}

// A wave's share of the call's slots (up to kTailTokens * kCombineMaxK of them), requested before its products: what is left
// behind the last arrival is a trip to memory for the rows
struct TailSlots {
    static constexpr int N = kTailTokens * kCombineMaxK / 64;
    int id[N], row[N];
    float w[N];
    __device__ __forceinline__ TailSlots(const CombineTail& tail) {
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const int i = min((int)threadIdx.x + 64 * u, tail.n * tail.k - 1);
            id[u] = tail.topk_idx[i];
            row[u] = tail.pos[i];
            w[u] = tail.topk_w[i];
        }
    }
};

// NCOL columns from n0 on of every token (at most kTailTokens), by one wave; a lane has 8 columns of a token.  lds: idle, 3 KiB
template <int MODE, int NCOL>
__device__ __forceinline__ void combine_columns(const CombineTail& tail, const TailSlots& slots, const uint16_t* y, const uint16_t* shared,
                                                int h, int n0, uint8_t* lds) {
    static_assert(kTailTokens * NCOL / 8 <= 64, "a chunk of 8 columns per lane");
    const int lane = threadIdx.x, k = tail.k, nk = tail.n * k;
    int* const rows = reinterpret_cast<int*>(lds);                    // [token][place in the summation order]
    float* const weights = reinterpret_cast<float*>(lds + kTailTokens * kCombineMaxK * 4);
    int* const ids = reinterpret_cast<int*>(lds + 2 * kTailTokens * kCombineMaxK * 4);
    if (MODE == MOE_COMBINE_BF16_SEQ) {
#pragma unroll
        for (int u = 0; u < TailSlots::N; ++u) ids[lane + 64 * u] = slots.id[u];
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < TailSlots::N; ++u) {
        const int i = lane + 64 * u;
        if (i >= nk) break;
        const int t = i / k;
        int a = i - t * k;
        if (MODE == MOE_COMBINE_BF16_SEQ) {
            a = 0;
            for (int v = 0; v < k; ++v) a += ids[t * k + v] < slots.id[u] ? 1 : 0;
        }
        rows[t * kCombineMaxK + a] = slots.row[u];
        weights[t * kCombineMaxK + a] = combine_weight<MODE>(slots.w[u]);
    }
    __syncthreads();
    const int t = lane / (NCOL / 8), col = n0 + 8 * (lane % (NCOL / 8));
    if (t >= tail.n || col >= h) return;
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    u32x4 sh = {0, 0, 0, 0}, res = {0, 0, 0, 0};
    if (shared) sh = load_shared_16(shared + (size_t)t * h + col);
    if (tail.residual) res = *reinterpret_cast<const u32x4*>(tail.residual + (size_t)t * h + col);
    for (int a0 = 0; a0 < k; a0 += 8) {
        u32x4 v[8];
#pragma unroll
        for (int b = 0; b < 8; ++b) v[b] = load_shared_16(y + (size_t)max(rows[t * kCombineMaxK + min(a0 + b, k - 1)], 0) * h + col);
#pragma unroll
        for (int b = 0; b < 8; ++b)
            if (a0 + b < k && rows[t * kCombineMaxK + a0 + b] >= 0) combine_add<MODE>(acc, v[b], weights[t * kCombineMaxK + a0 + b]);
    }
    *reinterpret_cast<u32x4*>(tail.out + (size_t)t * h + col) = combine_finish(acc, shared != nullptr, sh, tail.residual != nullptr, res);
}

// ---- thin kernel: calls in which no expert has more than 16 rows (decoding a few sequences), where thin_pays ----
//
// Such a call touches a few experts, and cut into tiles of 256 weight rows it has fewer tiles than the chip has CUs
// (one token of DeepSeek-V2-Lite: 66) or two and a half rounds of them.  Here the unit is a WAVE with 32 weight rows --
// 16 gate rows and the matching up rows, or 32 down rows (16 where that leaves most of the chip idle, thin_down_narrow) -- and
// the whole K, each wave a workgroup of its own: no barrier, six of them per CU, and nothing to wait for but its own DMA.  A
// stage is 128 bytes of each weight row (64 k of bf16, 128 of fp8: whole lines) and the same k of 16 token rows (rows that do not
// exist cost no request), NB stages in a ring.  Every matrix instruction gets the k values that the streamers above give it, in
// the same lanes and the same order, so a row's bits are those of a larger call (fp8: of a larger call whose experts have up
// to 64 rows).  The body is thin_columns (thin_gemm.h).
// Measured (us, tile kernel -> this): DeepSeek-V2-Lite, one token (8 x 1408 of 2048) 25 + 25 and 19 + 33 -> 17 and 14;
// DeepSeek-V3, 5 tokens (39 experts, fp8) 190 and 115 -> 187 and 92 = 6.0 TB/s.  Weights loaded into registers instead
// reach 4 ... 5 TB/s: a fragment load then takes half a line from each of 16 rows.
template <bool SWIGLU, bool W8, int NF, bool TAIL>
__global__ __launch_bounds__(64) void grouped_gemm_thin_kernel(GemmPair pair_of, CombineTail tail) {
    static_assert(!TAIL || NF == 1, "the combine's rule");
    constexpr int NCOL = SWIGLU ? 16 : 16 * NF;   // output columns of a wave
    constexpr int NB = 24576 / thin_stage_bytes<W8, NF>;               // stages in LDS
    __shared__ __attribute__((aligned(1024))) uint8_t lds[NB * thin_stage_bytes<W8, NF>];
    const int lane = threadIdx.x;
    const bool of_shared = (int)blockIdx.x < pair_of.shared_tiles;
    const GemmArgs& g = pair_of.p[of_shared ? 1 : 0];
    const int unit = (int)blockIdx.x - (of_shared ? 0 : pair_of.shared_tiles);
    const int N = g.N;
    const int tiles = (N + NCOL - 1) / NCOL;

    // the (unit / tiles)-th expert that has rows: 256 experts at a time, 4 per lane
    int left = unit / tiles, e = -1, row0 = 0, row_end = 0;
    for (int base = 0; base < g.E; base += 256) {
        int o[5], c = 0;
#pragma unroll
        for (int j = 0; j < 5; ++j) o[j] = g.offsets[min(base + 4 * lane + j, g.E)];
#pragma unroll
        for (int j = 0; j < 4; ++j) c += o[j + 1] > o[j] ? 1 : 0;
        int inc = c;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int up = __shfl_up(inc, d);
            if (lane >= d) inc += up;
        }
        const int tot = __builtin_amdgcn_readlane(inc, 63);
        if (left < tot) {
            int k = left - (inc - c), ce = 0, c0 = 0, c1 = 0;
            const uint64_t owner = __ballot(k >= 0 && k < c);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (o[j + 1] > o[j]) {
                    if (k == 0) { ce = base + 4 * lane + j; c0 = o[j]; c1 = o[j + 1]; }
                    --k;
                }
            const int l = __builtin_ctzll(owner);
            e = __builtin_amdgcn_readlane(ce, l);
            row0 = __builtin_amdgcn_readlane(c0, l);
            row_end = __builtin_amdgcn_readlane(c1, l);
            break;
        }
        left -= tot;
    }
    if (e < 0) return;
    [[maybe_unused]] const auto slots = [&] { if constexpr (TAIL) return TailSlots(tail); else return 0; }();
    const int n0 = (unit % tiles) * NCOL;
    thin_columns<SWIGLU, W8, NF, TAIL, NB>(ThinUnit{g.b0[e], SWIGLU ? g.b1[e] : nullptr, W8 ? g.s0[e] : nullptr, W8 && SWIGLU ? g.s1[e] : nullptr, g.a,
                                                    g.row_map, g.a_bytes, g.a_rows, g.c, g.K, N, row0, row_end}, n0, lds);
    if constexpr (TAIL) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's columns are where every XCD finds them
        int left_out = 0;
        if (lane == 0) left_out = __hip_atomic_fetch_add(tail.arrivals + unit % tiles, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_readfirstlane(left_out) != -1) return;
        asm volatile("" ::: "memory");
        const uint16_t* const y = pair_of.p[0].c;
        const uint16_t* const sh = pair_of.shared_tiles > 0 ? pair_of.p[1].c : nullptr;
        if (tail.mode == MOE_COMBINE_F32) combine_columns<MOE_COMBINE_F32, NCOL>(tail, slots, y, sh, N, n0, lds);
        else if (tail.mode == MOE_COMBINE_BF16_PROD) combine_columns<MOE_COMBINE_BF16_PROD, NCOL>(tail, slots, y, sh, N, n0, lds);
        else combine_columns<MOE_COMBINE_BF16_SEQ, NCOL>(tail, slots, y, sh, N, n0, lds);
    }
}


// ---- the gate and up projection of one fp8 MLP at few rows ----
//
// One wide MLP (DeepSeek-V3: 18432 columns) has tiles of 128 columns for about half of the CUs, and each takes what a CU can
// stream, 38 GB/s, or, from some 64 rows on, what its waves can multiply.  Here a wave has 8 columns, their gate rows and
// their up rows in one fragment of 16, and a workgroup as many waves (8 to 10) as make one tile for every CU: 9 for 18432 columns and
// 256 CUs.  Weights (whole lines, a wave's own) and token rows reach LDS by DMA, 128 k a stage, NB stages in a ring; a lane reads 16 weights
// at once, as in stream8_tile, so every weight is converted once.  Every tile starts its walk over k at a block of its own.
// What bounds it: up to 32 rows the weights' way from memory, above it LDS: every wave reads all token rows for its one fragment.
// DeepSeek-V3's dense MLP, whole call, us, thin kernel (up to 16 rows) or tile kernel -> this: 1 / 4 / 16 / 32 / 64 / 96 tokens 82 / 81 / 91 /
// 95 / 114 / 138 -> 77 / 75 / 77 / 85 / 107 / 132; 112 148 and 148, 128 156 and 161, so that it ends at 96 rows.
constexpr int DM_WAVES = 10, DM_ROWS = 96;       // at most
constexpr int dm_stages(int tg) { return tg == 1 ? 6 : tg == 2 ? 5 : tg <= 4 ? 4 : 3; }      // (what fits)
constexpr int dm_stage_bytes(int tg) { return DM_WAVES * 2048 + tg * 4096; }
template <int TG>                                // 16-row token groups (1 .. 6)
__device__ __forceinline__ void gate_up_few_rows(const GemmArgs& g, int n_rows, uint8_t* lds) {
    constexpr int NB = dm_stages(TG), SB = dm_stage_bytes(TG);
    constexpr int NDT = (TG + 1) / 2, NI = 2 + NDT;        // token DMA instructions per wave (4 rows each), all of a stage
    static_assert(TG >= 1 && 16 * TG <= DM_ROWS && (NB - 1) * NI < 64, "stages");
    const int lane = threadIdx.x & 63, wave = uni(threadIdx.x >> 6), waves = (int)blockDim.x >> 6;
    const int K = g.K, N = g.N, nk = K >> 7;
    const int rot = (int)blockIdx.x % nk;
    const int n0 = ((int)blockIdx.x * waves + wave) * 8;   // this wave's columns (N or more: none)
    const int col0 = min(n0, N - 8);
    const int row0 = uni(g.offsets[0]), row_end = min(uni(g.offsets[1]), row0 + n_rows);
    if (row0 >= row_end) return;
    auto block_of = [&](int p) { const int b = min(p, nk - 1) + rot; return b >= nk ? b - nk : b; };

    const uint8_t *bm0 = uni_ptr(g.b0[0]), *bm1 = uni_ptr(g.b1[0]);
    gptr_f32 sc0 = (gptr_f32)(uintptr_t)uni_ptr(g.s0[0]) + (col0 >> 7) * nk, sc1 = (gptr_f32)(uintptr_t)uni_ptr(g.s1[0]) + (col0 >> 7) * nk;
    // DMA: weights, instruction 0 the gate rows, 1 the up rows (fragment rows 0 .. 7 and 8 .. 15): row lane / 8, part lane % 8
    const int lr = lane >> 3, pp = lane & 7;
    uint32_t w_voff[2], t_voff[NDT], t_dst[NDT];
#pragma unroll
    for (int i = 0; i < 2; ++i) w_voff[i] = (uint32_t)(col0 + lr) * (uint32_t)K + (uint32_t)((pp ^ wsw(8 * i + lr)) << 4);
    const uint8_t* a_base = reinterpret_cast<const uint8_t*>(g.a) + (g.row_map ? (size_t)0 : (size_t)row0 * K * 2);
    const int a_records = g.row_map ? (int)(uint32_t)g.a_bytes : (row_end - row0) * K * 2;
#pragma unroll
    for (int i = 0; i < NDT; ++i) {               // token rows 4 (waves i + wave) + lane / 16, chunk lane % 16
        const int at = waves * i + wave, tr = 4 * at + (lane >> 4);
        const int r = min(row0 + tr, row_end - 1);
        const int src = g.row_map ? ((gptr_i32)(uintptr_t)g.row_map)[r] : r - row0;
        t_voff[i] = (uint32_t)src * (uint32_t)(K * 2) + (uint32_t)(((lane & 15) ^ tsw(tr)) << 4);
        if (row0 + tr >= row_end || (g.row_map && (unsigned)src >= (unsigned)g.a_rows)) t_voff[i] = 0xfffffff0u;
        t_dst[i] = (uint32_t)uni(at < 4 * TG ? DM_WAVES * 2048 + at * 1024 : -1);      // -1: past the staged rows
    }
    auto dma = [&](int p, int buf) __attribute__((always_inline)) {
        const int live = uni(p < nk ? -1 : 0);    // past the end: empty descriptors, the instructions still count
        uint8_t* d = lds + buf * SB;
        const uint32_t so = (uint32_t)block_of(p) * 128u;
        const __amdgpu_buffer_rsrc_t r0d = __builtin_amdgcn_make_buffer_rsrc((void*)bm0, 0, live, 0x00020000);
        const __amdgpu_buffer_rsrc_t r1d = __builtin_amdgcn_make_buffer_rsrc((void*)bm1, 0, live, 0x00020000);
        const __amdgpu_buffer_rsrc_t rad = __builtin_amdgcn_make_buffer_rsrc((void*)a_base, 0, live & a_records, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r0d, (lds_u8)(d + wave * 2048), 16, w_voff[0], so, 0, 2);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r1d, (lds_u8)(d + wave * 2048 + 1024), 16, w_voff[1], so, 0, 2);
#pragma unroll
        for (int i = 0; i < NDT; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rad, (lds_u8)((int)t_dst[i] < 0 ? lds + NB * SB : d + t_dst[i]), 16, t_voff[i], 2 * so, 0, 0);
    };

    const int frow = lane & 15, q = lane >> 4;
    const int fq = ((q & 1) << 1) | (q >> 1);
    const uint32_t w_rd = (uint32_t)(wave * 2048 + frow * 128), wkey = (uint32_t)wsw(frow);
    const uint32_t t_rd = (uint32_t)(DM_WAVES * 2048 + frow * 256), tkey = (uint32_t)tsw(frow);
    f32x4 acc[TG];
#pragma unroll
    for (int t = 0; t < TG; ++t) acc[t] = f32x4{0};
    // lane l holds the block scales of stage 64 i + l, requested before the DMA that the waits count
    float v0 = sc0[block_of(lane)], v1 = sc1[block_of(lane)];
#pragma unroll
    for (int i = 0; i < NB - 1; ++i) dma(i, i);
    asm volatile("s_waitcnt vmcnt(%2)" : "+v"(v0), "+v"(v1) : "n"((NB - 1) * NI));
    int buf = 0;
    for (int p = 0; p < nk; ++p) {
        // this wave's DMA of block p has landed and its reads of block p - 1 have returned, then everybody's: behind the barrier
        // that block's buffer takes block p + NB - 1
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((NB - 2) * NI) : "memory");
        if ((p & 63) == 0 && p > 0) {
            v0 = sc0[block_of(p + lane)];
            v1 = sc1[block_of(p + lane)];
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(v0), "+v"(v1));
        }
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const uint8_t* b = lds + buf * SB;
        const float c0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v0), p & 63));
        const float c1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v1), p & 63));
        const float scale = frow < 8 ? c0 : c1;
        u32x4 raw[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) raw[h] = *reinterpret_cast<const u32x4*>(b + w_rd + (((4 * h + fq) ^ wkey) << 4));
        dma(p + NB - 1, buf == 0 ? NB - 1 : buf - 1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2) {
                const uint32_t coff = (uint32_t)(((8 * h + 2 * fq + s2) ^ tkey) << 4);
                const bf16x8 wa = __builtin_bit_cast(bf16x8, dequant8(raw[h][2 * s2], raw[h][2 * s2 + 1], scale));
#pragma unroll
                for (int t = 0; t < TG; ++t) {
                    const bf16x8 tf = *reinterpret_cast<const bf16x8*>(b + t_rd + t * 16 * 256 + coff);
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa, tf, acc[t], 0, 0, 0);
                }
            }
        }
        buf = buf + 1 == NB ? 0 : buf + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no DMA may land in LDS after the workgroup has gone

    // A lane of the lower half-wave holds 4 gate columns of a row, the same lane of the upper half their up columns: the lower half
    // takes columns 0 and 1, the upper one 2 and 3
#pragma unroll
    for (int t = 0; t < TG; ++t) {
        f32x4 gate = {0, 0, 0, 0}, up = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float a = acc[t][i], b = acc[t][2 + i];
            const auto x = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
            uint32_t lo = x[0], hi = x[1];
            asm volatile("" : "+v"(lo), "+v"(hi));            // (here, with every lane, not where the store needs it)
            gate[i] = __builtin_bit_cast(float, lo);
            up[i] = __builtin_bit_cast(float, hi);
        }
        const u32x2 o = epilogue_pack<true>(gate, up);
        const int r = row0 + 16 * t + frow;
        if (r < row_end && n0 < N) *reinterpret_cast<uint32_t*>(g.c + (size_t)r * N + n0 + 4 * (q & 1) + 2 * (q >> 1)) = o[0];
    }
}
template <int TG>
__global__ __launch_bounds__(64 * DM_WAVES) void gate_up_few_rows_kernel(GemmArgs g, int n_rows) {
    // (1 KiB that nobody reads behind the stages)
    __shared__ __attribute__((aligned(1024))) uint8_t lds[dm_stages(TG) * dm_stage_bytes(TG) + 1024];
    static_assert(sizeof(lds) <= 160 * 1024, "LDS");
    gate_up_few_rows<TG>(g, n_rows, lds);
}

// ---- split kernel: the down projection of a dense fp8 MLP at few rows ----
//
// One MLP of few rows has hidden / 256 column tiles (DeepSeek-V3: 28) with a long k (18432), and a workgroup takes 0.8 to
// 1.7 us per 128 k however few others run: 28 CUs worked while the rest waited.  Here a tile's k is cut into slices, one
// workgroup each, so that tiles x slices fill the CUs once; the fp32 sums of the slices go to the workspace and
// add_slices_kernel adds them, in order, and rounds once.  Rows past 128 are cut into tiles of equal height; all tiles of a
// call run the same body, chosen by that height, so a row's bits do not depend on its place.  The M tiles of one piece of
// the weights are neighbours on one XCD.  (From 257 rows on they may run as 256-row tiles of the persistent body instead, split_plan.)
// Measured (DeepSeek-V3's dense MLP, both launches, us, without scratch -> with it): 1 token 119 -> 75, 17: 185 -> 87,
// 64: 231 -> 115, 128: 356 -> 161, 192: 516 -> 220, 256: 426 -> 273; of those the gate and up products take 49, 58, 76, 104, 150
// and 186.
__global__ __launch_bounds__(512) void grouped_gemm_split_kernel(GemmArgs g, int n_rows, SplitPlan plan, float* part) {
    __shared__ __attribute__((aligned(1024))) uint8_t lw0[S8_WBYTES];
    __shared__ __attribute__((aligned(1024))) uint8_t lw1[S8_WBYTES];
    __shared__ __attribute__((aligned(1024))) uint8_t lw2[S8_WBYTES];
    __shared__ __attribute__((aligned(1024))) uint8_t lt0[128 * ROW_B];
    __shared__ __attribute__((aligned(1024))) uint8_t lt1[128 * ROW_B];
    __shared__ __attribute__((aligned(1024))) uint8_t lt2[128 * ROW_B];
    const SBuf b0{lw0, lt0}, b1{lw1, lt1}, b2{lw2, lt2};
    const TileLds lds{lw0, lw1, lw2, lt0, lt1, lt2};
    const int local = blockIdx.x >> 3;
    const int piece = local / plan.m_tiles * 8 + (blockIdx.x & 7), m_tile = local % plan.m_tiles;
    if (piece >= plan.slices * g.n_tiles_n) return;
    const int slice = piece / g.n_tiles_n, n_tile = piece % g.n_tiles_n;
    const int base = uni(g.offsets[0]), stop = min(uni(g.offsets[1]), base + n_rows);
    const int r0 = base + m_tile * plan.rows, r1 = min(r0 + plan.rows, stop);
    if (r0 >= r1) return;
    const int first = slice * plan.blocks;
    const KSlice ks{first, min(plan.blocks, (g.K >> 7) - first), base, part + (size_t)slice * n_rows * g.N};
    const int groups = (r1 - r0 + 15) >> 4;
    OneTile none;
    if (plan.rows <= 64) {
        if (groups == 1) stream8_tile<1, false, true>(g, b0, b1, b2, 0, r0, r1, n_tile, none, ks);
        else if (groups == 2) stream8_tile<2, false, true>(g, b0, b1, b2, 0, r0, r1, n_tile, none, ks);
        else if (groups == 3) stream8_tile<3, false, true>(g, b0, b1, b2, 0, r0, r1, n_tile, none, ks);
        else stream8_tile<4, false, true>(g, b0, b1, b2, 0, r0, r1, n_tile, none, ks);
    } else {
        if (groups <= 5) stream8x_tile<5, false, true>(g, lds, 0, r0, r1, n_tile, true, none, ks);
        else if (groups == 6) stream8x_tile<6, false, true>(g, lds, 0, r0, r1, n_tile, true, none, ks);
        else if (groups == 7) stream8x_tile<7, false, true>(g, lds, 0, r0, r1, n_tile, true, none, ks);
        else stream8x_tile<8, false, true>(g, lds, 0, r0, r1, n_tile, true, none, ks);
    }
}

// y = bf16(part[0] + part[1] + ...), 4 columns per thread
__global__ __launch_bounds__(256) void add_slices_kernel(const float* __restrict__ part, const int32_t* __restrict__ offsets,
                                                         uint16_t* __restrict__ y, int n_rows, int N, int slices) {
    const int base = offsets[0], rows = min(offsets[1] - base, n_rows);
    const size_t at = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4, stride = (size_t)n_rows * N;
    if (rows <= 0 || at >= (size_t)rows * N) return;
    f32x4 sum = *reinterpret_cast<const f32x4*>(part + at);
#pragma unroll 4
    for (int s = 1; s < slices; ++s) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(part + s * stride + at);
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] += v[i];
    }
    *reinterpret_cast<u32x2*>(y + (size_t)base * N + at) = epilogue_pack<false>(sum, sum);
}

// lane id produced where it is used: the compiler cannot hoist it (and everything derived from it)
// out of the tile loop and keep it in registers through the k loop
__device__ __forceinline__ int fresh_lane() {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}

// Persistent body for BM = 256: one workgroup per CU walks its share of the tiles, and the software
// pipeline runs on across the tile boundary (a tile's last k-iterations already fetch the next tile's
// first stages, and the epilogue runs beside them).  What a fresh workgroup pays per tile -- launch,
// tile-prefix scan, pointer chase, first fetch, store drain: 6-8 us against 57 us of k loop for K = 2048 --
// is paid once per workgroup or overlaps the previous tile's work.
//
// Token rows (and bf16 weights) reach LDS by DMA: buffer_load_dwordx4 ... lds writes 64 lanes x 16 bytes
// to 1 KiB of consecutive LDS, each lane fetching the 16 bytes that belong at its position of the
// swizzled layout, so there are no staging registers, no LDS store instructions and no per-chunk load
// waits in the MFMA stream.  fp8 weights still go through registers (they are converted on the way), two
// k-stages ahead.  Three things make this worth it (the same loads issued as global_load ... lds in one array per
// stage measured 2 % slower than register staging; this form 3-5 % faster):
//  * buffer (MUBUF) loads.  The compiler models the FLAT-encoded global_load ... lds as a possible LDS
//    access through the flat aperture and from then on waits for ALL outstanding LDS operations
//    (lgkmcnt(0)) wherever an operand fragment is needed, which serialises the fragment reads.
//  * whatever a DMA fills while something else is read is an LDS array of its own.  An LDS access that may alias the
//    target of an outstanding DMA gets a wait for it in front.
//  * stage parities are literals (the k loop is unrolled by two), so reads of one stage provably do not
//    alias the DMA into the other.
//
// What bounds it: matrix cores 81 % (bf16) and 68 % (fp8) of the cycles at 1.71 and 1.83 GHz, the chip's power limit.  A
// stage lives in LDS for two iterations, but its pieces are read in the first half of one: replaced piece by piece
// (`iteration` below) every DMA has one to one and a half iterations to land, where refilling a whole stage behind one barrier
// left the last pieces half an iteration, less than a trip to L2 under load.  TFLOP/s, one barrier per iteration -> this,
// both in one process (vendor library: 1520, 1428): bf16, one group of 65536 rows, 7168 -> 2 x 2048 1392 -> 1498, 2048 -> 7168
// 1378 -> 1396; 8 experts, 32768 rows, 4096 <-> 14336 1273 -> 1383 and 1277 -> 1390; 160 experts, 196608 rows, 5120 <-> 1536
// 1190 -> 1271 and 1076 -> 1164.  fp8, 64 experts, 131072 rows, 7168 <-> 2048: 1259 -> 1282 and 1201 -> 1217; there the
// conversion, 64 vector instructions per 64 matrix instructions, is what is left (a tenth more with most of it taken out).
// PAIRED: with a second problem.  (An instantiation of its own: the choice per tile costs DeepSeek-V3's 65536 tokens 0.4 %.)
// SPLIT: the down projection of one MLP, its tiles once per slice of k, all of them here; the fp32 sums go to `split`.
// LDS of its workgroup: the two stages' token rows in halves, their weights, and tables.  Every piece that a DMA writes while another
// is read is an array of its own: as separate objects they provably do not alias (otherwise a read waits for every
// outstanding DMA).  The fp8 path writes the weight stages with ordinary LDS stores.
constexpr int PE = 512;                          // experts that the tables hold
struct PersistentTables {                        // (read by read_pair and read_pointers once the DMA has begun)
    unsigned long long ptr1[4];                  // the second problem's matrices and scales
    int off1[2];                                 // and its rows
    int wtot[8];
    int pref[PE + 1], off[PE + 1];               // M tiles in front of an expert, and its first row
};
struct PersistentLds {
    uint8_t *a0a, *a0b, *a1a, *a1b, *b0, *b1;
    unsigned long long* ptr;                     // [4][PE] matrices and scales of the experts
    PersistentTables* tables;
};
// Reads of tables that lie behind token rows in one array: as ordinary reads they would wait for every DMA into those rows.
__device__ __forceinline__ void read_pair(const int* p, int& a, int& b) {       // p[0], p[1]
    unsigned long long v;
    asm volatile("ds_read2_b32 %0, %1 offset1:1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"((uint32_t)(uintptr_t)(lds_u8)const_cast<int*>(p)) : "memory");
    a = uni((int)(uint32_t)v);
    b = uni((int)(v >> 32));
}
// N words, `stride` bytes apart
template <int N>
__device__ __forceinline__ void read_pointers(const unsigned long long* table, uint32_t stride, unsigned long long (&v)[4]) {
    const uint32_t at = (uint32_t)(uintptr_t)(lds_u8)const_cast<unsigned long long*>(table);
    if constexpr (N == 4)
        asm volatile("ds_read_b64 %0, %4\n\tds_read_b64 %1, %5\n\tds_read_b64 %2, %6\n\tds_read_b64 %3, %7\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(at), "v"(at + stride), "v"(at + 2 * stride), "v"(at + 3 * stride) : "memory");
    else if constexpr (N == 2)
        asm volatile("ds_read_b64 %0, %2\n\tds_read_b64 %1, %3\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v[0]), "=&v"(v[1]) : "v"(at), "v"(at + stride) : "memory");
    else
        asm volatile("ds_read_b64 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v[0]) : "v"(at) : "memory");
}
template <bool SWIGLU, bool W8, bool PAIRED, bool SPLIT>
__device__ __forceinline__ void persistent_body(const GemmPair& pair_of, const SplitArgs& split, const PersistentLds& L, int grid) {
    static_assert(!SPLIT || (!SWIGLU && W8 && !PAIRED), "slices of k: the down projection of one fp8 MLP");
    const GemmArgs& g = pair_of.p[0];            // the routed experts; the tiles of the second problem come first
    constexpr int MT = 4, WN = 4;
    constexpr int NT = 128 * WN;
    constexpr int BM = 64 * MT;
    constexpr int RB = NT / 4;                  // fp8: B rows per pass (rows are 4 chunks of 16 weights)
    constexpr int NB = BN_ROWS / RB;            // fp8: 16-byte global B chunks per thread per stage (2)
    constexpr int NBLK = SWIGLU ? 128 : 256;
    constexpr int ND = 4;                       // DMA instructions per wave and tile half (32 rows of 128 bytes = 4 x 1 KiB)
    uint8_t *const sA0a = L.a0a, *const sA0b = L.a0b, *const sA1a = L.a1a, *const sA1b = L.a1b, *const sB0 = L.b0, *const sB1 = L.b1;
    int *const s_pref = L.tables->pref, *const s_wtot = L.tables->wtot, *const s_off = L.tables->off, *const s_off1 = L.tables->off1;
    unsigned long long* const s_ptr1 = L.tables->ptr1;
    constexpr int NM = (SWIGLU ? 2 : 1) * (W8 ? 2 : 1);       // pointers of a tile: gate (down), up, then their scales

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wave_s = uni(wave);
    const int wm = wave_s & 1, wn = (wave_s >> 1) % WN;

    // M-tile prefix over experts; the experts' row offsets and matrix pointers go to LDS tables on the way
    ExpertOfThread mine;
    const int run = mtile_prefix_scan<NT>(g, tid, s_pref, s_wtot, mine, [&](int c) { return persistent_tiles(g, SPLIT ? min(c, split.n_rows) : c); }, [&](int e, int o0, int o1) {
        s_off[e] = o0;
        if (e == g.E - 1) s_off[g.E] = o1;
        L.ptr[e] = (unsigned long long)(uintptr_t)g.b0[e];
        if (SWIGLU) L.ptr[PE + e] = (unsigned long long)(uintptr_t)g.b1[e];
        if (W8) L.ptr[NM / 2 * PE + e] = (unsigned long long)(uintptr_t)g.s0[e];
        if (W8 && SWIGLU) L.ptr[3 * PE + e] = (unsigned long long)(uintptr_t)g.s1[e];
    });
    if (tid == 0) s_pref[g.E] = run;
    if (PAIRED && tid == 0) {
        const GemmArgs& s = pair_of.p[1];
        s_off1[0] = s.offsets[0];
        s_off1[1] = s.offsets[1];
        s_ptr1[0] = (unsigned long long)(uintptr_t)s.b0[0];
        if (SWIGLU) s_ptr1[1] = (unsigned long long)(uintptr_t)s.b1[0];
        if (W8) s_ptr1[NM / 2] = (unsigned long long)(uintptr_t)s.s0[0];
        if (W8 && SWIGLU) s_ptr1[3] = (unsigned long long)(uintptr_t)s.s1[0];
    }
    __syncthreads();
    // whole rounds, and the last one unless it is better off in pieces: one-workgroup tiles, whose own are counted for that
    const SharedTiles second_tiles = PAIRED ? shared_tiles_of<W8>(pair_of.p[1], uni(s_off1[0]), uni(s_off1[1])) : SharedTiles{};
    const int ptiles1 = second_tiles.persistent;
    // (of up to 512 experts: at most 1024 M tiles, the experts with a tall one above them)
    const int sums = g.tail_cus > 0 ? sum_over_experts<NT>(g, tid, s_wtot, [&](int c) { return own_tiles<W8>(g, c) + (has_tall_tile<W8>(g, c) ? 1 << 16 : 0); }) : 0;
    const int own = (sums & 0xffff) * g.n_tiles_n + second_tiles.own;
    const bool tall = (sums >> 16) > 0 || second_tiles.tall;
    const int slice_tiles = run * g.n_tiles_n;   // SPLIT: tiles of one slice
    const int all = SPLIT ? slice_tiles * split.plan.slices : slice_tiles + ptiles1, total = all - tail_of(g, all, own, tall).tiles;
    const PersistentPlan plan = SPLIT ? PersistentPlan{0, grid} : persistent_plan(g, total, own, grid);
    const int xcd = blockIdx.x & 7, place = blockIdx.x >> 3;
    // this workgroup's it-th tile, `total` or more past its last one
    auto tile_of = [&](int it) {
        if (it < plan.full) return (it * 8 + xcd) * (grid >> 3) + place;
        return place < (plan.width >> 3) ? plan.full * grid + ((it - plan.full) * 8 + xcd) * (plan.width >> 3) + place : total;
    };
    int it = 0;
    if (tile_of(0) >= total) return;

    // Token rows come through a buffer descriptor and 32-bit byte offsets.  Gathered rows (row_map): one
    // descriptor over all of x, whose size the launcher has checked against 4 GiB, so a row_map entry
    // outside x reads zeros instead of faulting.  Sorted rows: the descriptor starts at the tile's first row.
    const uint8_t *a_base = nullptr, *a_base_n = nullptr;
    int a_records = -1, a_records_n = -1;
    uint32_t a_voff[ND];                        // this wave's DMA offsets of the tile being fetched
    int a_row_n[ND];                            // and its rows of x of the next one
    // bf16 weights also by DMA: descriptors of the expert's matrices and per-lane offsets (gate and up: rows n0 .. n0 + 127
    // of either matrix, so one pair of offsets)
    constexpr int NBO = SWIGLU ? 2 : 4;
    uint32_t b_voff[ND], b_voff_n[ND];          // (NBO of them are used)
    const uint8_t *bm0 = nullptr, *bm1 = nullptr, *bm0_n = nullptr, *bm1_n = nullptr;
    // fp8 weights through registers
    uint32_t b8_voff[NB];
    const uint8_t *b8m0 = nullptr, *b8m1 = nullptr;
    int srow0 = 0, srow1 = 0;
    gptr_f32 sc0 = nullptr, sc1 = nullptr;
    int row0 = 0, row_end = 0, n0 = 0;
    int cur_e = 0;
    uint16_t* c_out = nullptr;                  // of the tile set up last: outputs and their row length
    int N_out = 0;
    // bf16 weights: k starts at another stage for every N tile (k_rotation); stage_of is the stage that pipeline step
    // kt fetches.  The rotation is adopted with the tile's DMA coordinates.
    // (So are the stages of a tile and the length of its token rows: the two problems may differ in them.)
    int rot = 0, rot_n = 0, nk_dma = 0, K_n = 0, nk_n = 0;
    auto stage_of = [&](int kt, int r) { const int kp = kt + r; return kp >= nk_dma ? kp - nk_dma : kp; };
    auto setup = [&](int v) {
        const int l = fresh_lane();
        const int t = wave_s * 64 + l;
        const bool second = PAIRED && v < ptiles1;
        // (selects, not a reference to either: that would be loads from the arguments, waited for on every tile)
        const GemmArgs& g1 = pair_of.p[1];
        const int K = second ? g1.K : g.K, N = second ? g1.N : g.N, nk = K / BK, tiles_n = second ? g1.n_tiles_n : g.n_tiles_n;
        const int32_t* const row_map = SWIGLU ? (second ? g1.row_map : g.row_map) : nullptr;
        int m_tile, n_tile, e, first, kb0 = 0;  // kb0: first block of 128 k
        nk_n = nk;
        int slice = 0;
        if (SPLIT) {
            slice = v / slice_tiles;
            v -= slice * slice_tiles;
            kb0 = slice * split.plan.blocks;
            nk_n = 2 * min(split.plan.blocks, (K >> 7) - kb0);
        }
        if (second) {
            e = 0;
            read_pair(s_off1, first, row_end);
            tile_in_expert(v, ptiles1 / tiles_n, tiles_n, m_tile, n_tile);
        } else {
            v -= ptiles1;
            const int q = v / tiles_n;
            int pe, pe_end;
            read_pair(s_pref + cur_e, pe, pe_end);
            while (pe_end <= q) read_pair(s_pref + ++cur_e, pe, pe_end);
            e = cur_e;
            const int mt_e = pe_end - pe;
            read_pair(s_off + e, first, row_end);
            if (SPLIT) row_end = min(row_end, first + split.n_rows);
            tile_in_expert(v - pe * tiles_n, mt_e, tiles_n, m_tile, n_tile);
        }
        row0 = first + m_tile * BM;
        n0 = n_tile * NBLK;
        // (SPLIT: the slice's sums of row `first`, moved so that row numbers stay those of the sorted rows)
        if (SPLIT) c_out = reinterpret_cast<uint16_t*>(split.part + ((ptrdiff_t)slice * split.n_rows - first) * N);
        else c_out = second ? g1.c : g.c;
        N_out = N;
        K_n = K;
        rot_n = W8 ? 0 : k_rotation<false>(n_tile, nk);
        // DMA instruction i of this wave fills rows 16*wave + 8*(i&1) .. +7 of the 128 rows of half i/2: lane l supplies
        // row +l/8 and the 16 bytes that belong at physical chunk l%8, i.e. logical chunk (l%8) ^ swz(row).  Row r of
        // half h of the token stage is row 128*(r/64) + 64*h + r%64 of the tile, row r of half h of the weight stage its
        // row 128*h + r.
        const int lr = l >> 3, pc = l & 7;
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            const int rt = ((wave_s >> 2) << 7) + ((i >> 1) << 6) + 16 * (wave_s & 3) + 8 * (i & 1) + lr;   // row of the tile
            const int r = min(row0 + rt, row_end - 1);
            a_row_n[i] = row_map ? ((gptr_i32)(uintptr_t)row_map)[r] : r - row0;   // (down: sorted rows)
        }
        a_base_n = reinterpret_cast<const uint8_t*>(second ? g1.a : g.a) + (row_map ? (size_t)0 : (size_t)row0 * K * 2) + (SPLIT ? kb0 * 256 : 0);
        a_records_n = row_map ? (int)(uint32_t)(second ? g1.a_bytes : g.a_bytes) : -1;
        unsigned long long ptr[4] = {};
        read_pointers<NM>(second ? s_ptr1 : L.ptr + e, second ? 8u : PE * 8u, ptr);
        const uint8_t* bmat0 = uni_ptr(reinterpret_cast<const void*>((uintptr_t)ptr[0]));
        const uint8_t* bmat1 = SWIGLU ? uni_ptr(reinterpret_cast<const void*>((uintptr_t)ptr[1])) : bmat0;
        if (W8) {
            sc0 = (gptr_f32)(uintptr_t)uni_ptr(reinterpret_cast<const void*>((uintptr_t)ptr[NM / 2]));
            sc1 = SWIGLU ? (gptr_f32)(uintptr_t)uni_ptr(reinterpret_cast<const void*>((uintptr_t)ptr[3])) : sc0;
            const int brow = t >> 2, bcol_b = (t & 3) << 4, KB = K >> 7;
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                int r = brow + RB * i;
                int n = SWIGLU ? (n0 + (r & 127)) : (n0 + r);
                b8_voff[i] = (uint32_t)min(n, N - 1) * (uint32_t)K + (uint32_t)bcol_b;
            }
            b8m0 = bmat0 + (SPLIT ? kb0 * 128 : 0); b8m1 = bmat1 + (SPLIT ? kb0 * 128 : 0);
            if (SWIGLU) { srow0 = (n0 >> 7) * KB; srow1 = srow0; }
            else        { srow0 = (n0 >> 7) * KB + kb0; srow1 = min((n0 >> 7) + 1, (N >> 7) - 1) * KB + kb0; }
        } else {
            bm0_n = bmat0; bm1_n = bmat1;
#pragma unroll
            for (int i = 0; i < NBO; ++i) {
                const int n = n0 + 128 * (i >> 1) + 16 * wave_s + 8 * (i & 1) + lr;
                const int lc = pc ^ (lr ^ (i & 1));
                b_voff_n[i] = (uint32_t)min(n, N - 1) * (uint32_t)(K * 2) + (uint32_t)(lc * 16);
            }
        }
    };
    auto adopt = [&]() {   // the next tile's DMA coordinates become the current ones
        // (the row loads are waited for here, half an iteration after they were issued, not where they are issued: such a wait
        // covers every older DMA)
        const int l = fresh_lane(), lr = l >> 3;
#pragma unroll
        for (int i = 0; i < ND; ++i)             // swz(row): row & 7 == lr, (row >> 3) & 1 == i & 1
            a_voff[i] = (uint32_t)a_row_n[i] * (uint32_t)(K_n * 2) + (uint32_t)(((l & 7) ^ lr ^ (i & 1)) << 4);
        if (!W8) {
#pragma unroll
            for (int i = 0; i < NBO; ++i) b_voff[i] = b_voff_n[i];
            bm0 = bm0_n; bm1 = bm1_n;
        }
        a_base = a_base_n;
        a_records = a_records_n;
        nk_dma = SPLIT ? nk_n : K_n / BK;
        rot = rot_n;
    };
    auto dma_a = [&](int st, int kt, int i) __attribute__((always_inline)) {
        uint8_t* d = st ? (i >= 2 ? sA1b : sA1a) : (i >= 2 ? sA0b : sA0a);
        const __amdgpu_buffer_rsrc_t rsrcA = __builtin_amdgcn_make_buffer_rsrc((void*)a_base, 0, a_records, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcA, (lds_u8)(d + (16 * wave_s + 8 * (i & 1)) * ROW_B), 16, a_voff[i],
                                                 (uint32_t)((W8 ? kt : stage_of(kt, rot)) * BK * 2), 0, 0);
    };
    auto dma_b = [&](int st, int kt, int i) __attribute__((always_inline)) {
        uint8_t* d = st ? sB1 : sB0;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)((SWIGLU && i >= 2) ? bm1 : bm0), 0, -1, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_u8)(d + (128 * (i >> 1) + 16 * wave_s + 8 * (i & 1)) * ROW_B), 16,
                                                 b_voff[SWIGLU ? (i & 1) : i], (uint32_t)(stage_of(kt, rot) * BK * 2), 0, 0);
    };
    // fp8 weight path (registers): thread t owns row t/4 (+128 i), chunks 2q, 2q+1 of the bf16 row
    const int brow = tid >> 2;
    uint32_t b_lds[2];
    const bool b_swap = W8 && ((brow >> 1) & 1);
    {
        int qd = tid & 3, sw = swz(brow), first = b_swap ? 1 : 0;
        b_lds[0] = (uint32_t)(brow * ROW_B + (((2 * qd + first) ^ sw) << 4));
        b_lds[1] = (uint32_t)(brow * ROW_B + (((2 * qd + 1 - first) ^ sw) << 4));
    }
    u32x4 rb[NB];
    float rs[2];
    auto load_b8 = [&](int i, uint32_t kofs) {
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)((SWIGLU && i >= NB / 2) ? b8m1 : b8m0), 0, -1, 0x00020000);
        return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, b8_voff[i], kofs, 0));
    };
    // Block scales come through buffer loads too, although their address is the same for every lane: as loads
    // through a pointer they could become scalar loads, which share a counter with the operand reads and return out of order.
    auto load_scale = [&](gptr_f32 sc, int idx) {
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)sc, 0, -1, 0x00020000);
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, 0, idx * 4, 0));
    };
    auto load_chunk = [&](int b, int kt) {      // chunk b of stage kt and its block scale: two loads
        rb[b] = load_b8(b, (uint32_t)(kt * BK));
        if (b / (NB / 2) == 0) rs[0] = load_scale(sc0, srow0 + (kt >> 1));
        else rs[1] = load_scale(sc1, srow1 + (kt >> 1));
    };
    auto b_item = [&](int it, uint8_t* Bs, int kn) {   // it in 0 .. 2*NB-1: half it%2 of chunk it/2
        const int b = it >> 1, half = it & 1;
        const u32x4 o = dequant8(rb[b][2 * half], rb[b][2 * half + 1], rs[b / (NB / 2)]);
        *reinterpret_cast<u32x4*>(Bs + ((half ^ (b_swap ? 1 : 0)) ? b_lds[1] : b_lds[0]) + b * RB * ROW_B) = o;
        if (half == 1) load_chunk(b, kn);
    };

    const int frow = lane & 15, fquad = lane >> 4, fkey = swz(frow);
    const int fchunk = ((fquad & 1) << 1) | (fquad >> 1);
    constexpr int TM = 2 * MT, TN = 4;
    // operand rows: fragment row = base + lane % 16; tokens: 64 rows of either half per wave row; weights: TN fragments
    // of 16 rows, for SWIGLU the first half from the gate rows and the second from the matching up rows
    const uint32_t t_rd = (uint32_t)((wm * 64 + frow) * ROW_B);
    const uint32_t w_rd = (uint32_t)((wn * (SWIGLU ? 32 : 64) + frow) * ROW_B);
    auto w_row = [](int j) { return SWIGLU ? (j < TN / 2 ? 0 : 128) + 16 * (j % (TN / 2)) : 16 * j; };
    const uint32_t coff[2] = {(uint32_t)((fchunk ^ fkey) << 4), (uint32_t)(((4 + fchunk) ^ fkey) << 4)};
    f32x4 acc[TM][TN];
    // A stage is multiplied in 8 sub-phases: token part q = u/2 (two 16-row tiles of the wave's 128 rows) x 32-wide
    // k-step s = u%2.  Slot v of an iteration issues the matrix instructions of sub-phase v - 2 and requests the
    // operands of sub-phase v.
    bf16x8 wfr[2][TN], tq[2][2];
    auto read_w = [&](const uint8_t* Bs, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < TN; ++j) wfr[s][j] = *reinterpret_cast<const bf16x8*>(Bs + w_rd + w_row(j) * ROW_B + coff[s]);
    };
    auto read_tq = [&](int st, int u) __attribute__((always_inline)) {
        const int q = u >> 1, s = u & 1;
        const uint8_t* As = st ? (q >= 2 ? sA1b : sA1a) : (q >= 2 ? sA0b : sA0a);
#pragma unroll
        for (int i = 0; i < 2; ++i) tq[u & 1][i] = *reinterpret_cast<const bf16x8*>(As + t_rd + (32 * (q & 1) + 16 * i) * ROW_B + coff[s]);
    };
    auto mfma_sub = [&](int u, bool zero) __attribute__((always_inline)) {
        const int q = u >> 1, s = u & 1;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int jx = 0; jx < TN; ++jx) {
                const int j = ((i + u) & 1) ? TN - 1 - jx : jx;
                const f32x4 c = zero && s == 0 ? f32x4{0} : acc[q * 2 + i][j];
                acc[q * 2 + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wfr[s][j], tq[u & 1][i], c, 0, 0, 0);
            }
    };
    // Iteration kt multiplies stage kt out of buffer par.  Two barriers: behind the first every wave has left stage
    // kt - 1, whose weights and second half of the token rows are replaced (by stage kt + 1); the first four slots
    // read all of a stage's weights and the first half of its token rows, and behind the second barrier those are
    // replaced in turn, by stage kt + 2.
    //   bf16: slots 0-3 bring weights 2, 3 and tokens 2, 3 of stage k1 (= kt + 1), slots 4-7 tokens 0, 1 and weights 0, 1 of
    //   stage k2 (= kt + 2).  fp8: slots 0, 1 tokens 2, 3 of stage k1; slots 2-5 convert the weight registers (stage kt + 1)
    //   into the other weight buffer and refill them with stage k2; slots 6, 7 tokens 0, 1 of stage k2.
    // Waits.  Loads retire in issue order, DMA into LDS and loads into registers alike (measured), but the compiler may move a
    // load into registers across a DMA, and nothing is known of stores: the waits count DMA operations only, whose number
    // and order the source fixes, so whatever else is in flight makes them stricter.  VM_X: DMA
    // issued after the last one that the first four slots read; VM_Y: after the last one that the others read; VM_TURN: after a
    // tile's first stage, waited for in front of the stores of the tile before, so that the first iteration need not wait.
    // first / second: the tile's first two iterations (sub-phases 6 and 7 of the first run in the second); turn: from the second
    // half on the DMA belongs to the next tile.
    constexpr int VM_X = W8 ? 4 : 6, VM_Y = W8 ? 4 : 8, VM_TURN = W8 ? 2 : 4;
    auto iteration = [&](int k1, int k2, int par, auto first, auto second, auto turn) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first)::value, SECOND = decltype(second)::value;
        const uint8_t* rdB = par ? sB1 : sB0;
        uint8_t* wrB = par ? sB0 : sB1;
        if (FIRST) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(VM_X) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            if (v == 4) {
                if (turn) adopt();
                if (FIRST) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(VM_Y) : "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            }
            if (W8) {
                if (v < 2) dma_a(par ^ 1, k1, v + 2);
                else if (v < 4) b_item(v - 2, wrB, k2);
                else if (v < 6) b_item(v - 2, wrB, k2);
                else dma_a(par, k2, v - 6);
            } else {
                if (v < 2) dma_b(par ^ 1, k1, v + 2);
                else if (v < 4) dma_a(par ^ 1, k1, v);
                else if (v < 6) dma_a(par, k2, v - 4);
                else dma_b(par, k2, v - 6);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (v >= 2) mfma_sub(v - 2, FIRST);
            else if (!FIRST) mfma_sub(6 + v, SECOND);
            read_tq(par, v);
            if (v < 2) read_w(rdB, v);
            // (fp8: two vector instructions of the conversion behind every matrix instruction, which hides them; in a clump
            // in front the waves of a SIMD, in step, leave the matrix core idle.  Gate and up 1226 -> 1251 TFLOP/s; the down
            // projection, whose registers hold less, runs the same either way and is left to the compiler)
            if (W8 && SWIGLU && v >= 2 && v < 6) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    static_assert(ND == 4 && (!W8 || NB == 2), "slot plan");
    // ---- tiles ----
    setup(tile_of(0));
    adopt();
    // prologue: what the iterations before the first would have issued, all of it landed (the scheduler orders it as it likes)
#pragma unroll
    for (int i = 0; i < ND; ++i) { dma_a(0, 0, i); if (!W8) dma_b(0, 0, i); }
    dma_a(1, 1, 0); dma_a(1, 1, 1);
    if (W8) {
        load_chunk(0, 0);
        load_chunk(1, 0);
#pragma unroll
        for (int it = 0; it < 4; ++it) b_item(it, sB0, 1);
    } else {
        dma_b(1, 1, 0); dma_b(1, 1, 1);
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);     // vmcnt(0), as an instruction that the compiler's own count knows
    constexpr int CW = SWIGLU ? 8 * TN : 16 * TN;    // output columns of this wave
    for (;;) {
        const int out_row0 = row0, out_row_end = row_end, out_n0 = n0, N = N_out, nk = nk_dma;
        uint16_t* const c = c_out;
        bool more = false;
        auto next_tile = [&]() {
            const int v = tile_of(++it);
            more = v < total;
            setup(more ? v : tile_of(it - 1));
        };
        constexpr std::true_type yes{};
        constexpr std::false_type no{};
        const bool only = nk == 2;               // (the first pair is the last one: not a copy of its own)
        if (only) next_tile();
        iteration(1, only ? 0 : 2, 0, yes, no, only);
        iteration(only ? 0 : 2, only ? 1 : 3, 1, no, yes, no);
        if (!only) {
            for (int kt = 2; kt < nk - 2; kt += 2) {
                iteration(kt + 1, kt + 2, 0, no, no, no);
                iteration(kt + 2, kt + 3, 1, no, no, no);
            }
            next_tile();
            iteration(nk - 1, 0, 0, no, no, yes);
            iteration(0, 1, 1, no, no, no);
        }
        // Epilogue.  A lane holds 4 consecutive columns (8 bytes) of one row per accumulator.  Gate and up: a wave has 32
        // columns, 64 bytes of a row; neighbouring lane groups exchange halves and store them from the registers.  Down: 64
        // columns, a whole 128-byte line of a row, put together in LDS, 16 rows at a time, in the wave's 2 KiB of the one piece
        // of a stage that no DMA writes before the next tile's first barrier.
        if (!SWIGLU && !SPLIT) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // every wave has read that piece
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
        mfma_sub(6, false);
        mfma_sub(7, false);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0)" :: "n"(VM_TURN) : "memory");
        {
            const int l = fresh_lane();
            const int fr = l & 15, q = l >> 4;
            const int rows_here = min(BM, out_row_end - out_row0) - wm * 128, ncol0 = out_n0 + wn * CW;
            const uint8_t* out = uni_ptr(SPLIT ? c + 2 * ((ptrdiff_t)(out_row0 + wm * 128) * N + ncol0) : c + (size_t)(out_row0 + wm * 128) * N + ncol0);
            uint8_t* ep = sA1b + wave_s * 2048;
#pragma unroll
            for (int mi = 0; mi < TM; ++mi) {
                if (SPLIT) {                     // sums: 16 bytes of a row per lane and fragment
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        const int r = 16 * mi + fr, col = 16 * j + 4 * q;
                        store16<0>(__builtin_bit_cast(u32x4, acc[mi][j]), out, r < rows_here && ncol0 + col < N ? (uint32_t)(r * N + col) * 4u : 0x80000000u);
                    }
                } else if (SWIGLU) {
                    const u32x4 o = pair_columns(epilogue_pack<true>(acc[mi][0], acc[mi][2]), epilogue_pack<true>(acc[mi][1], acc[mi][3]));
                    const int r = 16 * mi + fr, col = 16 * (q & 1) + 8 * (q >> 1);
                    store16<0>(o, out, r < rows_here && ncol0 + col < N ? (uint32_t)(r * N + col) * 2u : 0x80000000u);
                } else {
#pragma unroll
                    for (int jj = 0; jj < 2; ++jj) {
                        const u32x4 o = pair_columns(epilogue_pack<false>(acc[mi][2 * jj], acc[mi][2 * jj]),
                                                     epilogue_pack<false>(acc[mi][2 * jj + 1], acc[mi][2 * jj + 1]));
                        *reinterpret_cast<u32x4*>(ep + fr * 128 + (((4 * jj + 2 * (q & 1) + (q >> 1)) ^ (fr & 7)) << 4)) = o;
                    }
#pragma unroll
                    for (int ps = 0; ps < 2; ++ps) {
                        const int rr = 8 * ps + (l >> 3), r = 16 * mi + rr, col = 8 * (l & 7);
                        const u32x4 o = *reinterpret_cast<const u32x4*>(ep + rr * 128 + (((l & 7) ^ (rr & 7)) << 4));
                        store16<2>(o, out, r < rows_here && ncol0 + col < N ? (uint32_t)(r * N + col) * 2u : 0x80000000u);
                    }
                }
            }
        }
        if (!more) break;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no DMA may land in LDS after the workgroup has gone
}

// ---- both kinds of tiles in one launch: calls of many rows per expert (both_kinds) ----
//
// One persistent workgroup per CU comes first; the tiles of one workgroup run on CUs that the plan leaves to them or as CUs fall free,
// claimed by the workgroups that are there or in workgroups of their own (Claims), so that the two kinds overlap and the launch
// drains once.  As two launches, one behind the other, the second's workgroups waited for the first's last tile (a second stream costs more than it gains).  Layers, us, two launches -> this: DeepSeek-V2-Lite, 1500 / 2200 /
// 3000 / 4096 tokens 423 / 514 / 589 / 701 -> 411 / 493 / 577 / 689, DeepSeek-V3 4500 / 9000 4385 / 7907 -> 4276 / 7840, DeepSeek-V2-236B
// 4000 / 9000 2286 / 3743 -> 2276 / 3735, Mixtral-8x7B 700 / 2500 714 / 1694 -> 692 / 1687; 16384 tokens and more the same.
// The two bodies take the call's arguments from two copies of them: loads that both need would move in front of the branch, and so
// many scalar registers alive there cost the down projection 320 to 376 bytes of spills (236 -> 308 us, DeepSeek-V2-Lite, 4096 tokens).
//
// A workgroup of one tile: the routed experts' own tiles, the shared expert's, then the pieces of the tiles that the persistent
// workgroups leave at the end of THEIR tile space, neighbours on one XCD (the prefix is rebuilt over that space).
struct TileTables {
    int own[PE + 1], persistent[PE + 1], off[PE + 1], wtot[8], tall[8], claim;      // M tiles of either kind in front of an expert, its first row
};
template <bool SWIGLU, bool W8, bool CLAIMS>
__device__ __forceinline__ void tile_body(const GemmPair& pair_of, const TileLds& lds, TileTables& t, int block) {
    constexpr int NT = 512;
    const int tid = threadIdx.x, xcd = block & 7;
    const bool claiming = CLAIMS && pair_of.claims != nullptr;
    const GemmArgs& ga = pair_of.p[0];
    int shared_first = 0, shared_end = 0;    // (requested here, so that the answer comes with that to the scan's loads)
    if (pair_of.shared_rows > 0) {
        shared_first = pair_of.p[1].offsets[0];
        shared_end = pair_of.p[1].offsets[1];
    }
    ExpertOfThread mine;
    const int run = mtile_prefix_scan<NT>(ga, tid, t.own, t.wtot, mine, [&](int c) { return own_tiles<W8>(ga, c); }, [&](int e, int o0, int o1) {
        t.off[e] = o0;
        if (e == ga.E - 1) t.off[ga.E] = o1;
    });
    if (tid == 0) t.own[ga.E] = run;
    const uint64_t tall_lanes = __ballot(has_tall_tile<W8>(ga, mine.o1 - mine.o0));
    if ((tid & 63) == 0) t.tall[tid >> 6] = tall_lanes != 0;
    SharedTiles s{};
    if (pair_of.shared_rows > 0) s = shared_tiles_of<W8>(pair_of.p[1], uni(shared_first), uni(shared_end));
    const int own = uni(run) * ga.n_tiles_n;
    int v = dealt_tile(xcd, block >> 3), total_p = 0;
    Tail tail{0, 2};
    __syncthreads();                     // t.wtot has been read, t.own is whole
    if (claiming || v >= own + s.own) {
        const int run_p = mtile_prefix_scan<NT>(ga, tid, t.persistent, t.wtot, mine, [&](int c) { return persistent_tiles(ga, c); }, [](int, int, int) {});
        if (tid == 0) t.persistent[ga.E] = run_p;
        total_p = uni(run_p) * ga.n_tiles_n + s.persistent;
        int tall = s.tall;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) tall |= t.tall[w];
        tail = tail_of(ga, total_p, own + s.own, uni(tall) != 0);
        __syncthreads();
    }
    const int limit = own + s.own + tail.pieces * tail.tiles;
    Claims claims{CLAIMS ? pair_of.claims : nullptr, xcd, limit, 0};
    if (claiming) {
        claims.ask();
        v = claims.take(&t.claim);
    } else if (v >= limit) {
        return;
    }
    for (; v >= 0; v = claims.take(&t.claim)) {
        const int* pref = t.own;
        int piece = -1, shared = 0, at = v;   // shared: tiles of the shared expert in front of the routed experts' in the space `at` counts in
        bool of_shared = false;
        if (v >= own + s.own) {              // a piece of one of the last persistent tiles
            const int h = v - own - s.own, of = h / tail.pieces;
            at = total_p - tail.tiles + of;
            piece = h - of * tail.pieces;
            pref = t.persistent;
            shared = s.persistent;
            of_shared = at < shared;
            if (!of_shared) at -= shared;
        } else if (v >= own) {
            at = v - own;
            shared = s.own;
            of_shared = true;
        }
        int which = uni(of_shared ? 1 : 0);
        asm volatile("" : "+s"(which));      // (else the arguments of both problems are loaded and prepared in front of the loop)
        const GemmArgs& g = pair_of.p[which];
        const ExpertAt x = of_shared ? ExpertAt{0, 0, shared / g.n_tiles_n} : expert_at(pref, g.E, at / g.n_tiles_n);
        const int e = x.e, o0 = of_shared ? s.first : uni(t.off[e]), row_end = of_shared ? s.end : uni(t.off[e + 1]), mt_e = x.tiles;
        int m_tile, n_tile;
        tile_in_expert(at - x.first * g.n_tiles_n, mt_e, g.n_tiles_n, m_tile, n_tile);
        int r0, r1;
        bool neighbours = true;
        if (piece >= 0) {                    // of a 256-row tile of the persistent body's space
            r0 = o0 + m_tile * 256 + piece * piece_rows(tail.pieces);
            r1 = min(min(row_end, o0 + (m_tile + 1) * 256), r0 + piece_rows(tail.pieces));
            if (r0 >= r1) {
                claims.ask();
                continue;
            }
        } else {
            const int first_row = o0 + (g.rem_split ? ((row_end - o0) & ~255) : 0), rows_e = row_end - first_row;
            const int slice = !W8 && rows_e >= PAIR_LO ? half_rows(rows_e) : 128;
            r0 = mt_e > 1 ? first_row + m_tile * slice : first_row;
            r1 = mt_e > 1 ? min(row_end, r0 + slice) : row_end;
            neighbours = mt_e > 1;
        }
        if (W8) stream8x<SWIGLU>(g, lds, e, r0, r1, n_tile, false, claims);
        else if (neighbours) stream16<SWIGLU, true>(g, lds.w0, lds.w1, lds.w2, lds.t0, lds.t1, e, r0, r1, n_tile, claims);
        else stream16<SWIGLU, false>(g, lds.w0, lds.w1, lds.w2, lds.t0, lds.t1, e, r0, r1, n_tile, claims);
    }
}
// CLAIMS: the call may bring counters.  Calls that do not (one MLP, the stand-alone entry points) have an instantiation without the loop:
// what the compiler prepares in front of it for every form of tile cost their launches 1.5 to 3 us (one fp8 MLP, 1100 rows, hidden 4096,
// intermediate 2048, gate and up / down 62.0 / 38.8 -> 59.0 / 37.2 us; 800 rows, 5120 x 3072, 74.1 / 48.2 -> 71.0 / 46.7).  A joint
// call without counters, a layer's stages one by one, runs in that with them.
template <bool SWIGLU, bool W8, bool PAIRED, bool CLAIMS>
__global__ __launch_bounds__(512) void grouped_gemm_both_kernel(GemmPair persistent_of, GemmPair tiles_of, int persistent_grid) {
    // The streamers' three weight buffers and token buffers.  The persistent body has its weights in the first two and its token
    // rows in the lower 16 KiB of the others, with its tables behind two of those.  (bf16: the whole LDS of a CU.)
    constexpr int TOKENS = 128 * ROW_B;
    __shared__ __attribute__((aligned(1024))) uint8_t lw0[S8_WBYTES];
    __shared__ __attribute__((aligned(1024))) uint8_t lw1[S8_WBYTES];
    __shared__ __attribute__((aligned(1024))) uint8_t lw2[S8_WBYTES];
    __shared__ __attribute__((aligned(1024))) uint8_t lt0[W8 ? TOKENS : 192 * ROW_B];
    __shared__ __attribute__((aligned(1024))) uint8_t lt1[192 * ROW_B];
    __shared__ __attribute__((aligned(1024))) uint8_t lt2[TOKENS];
    __shared__ __attribute__((aligned(16))) uint8_t tile_tables[W8 ? sizeof(TileTables) : 16];
    static_assert(TOKENS + 4 * PE * 8 <= S8_WBYTES && TOKENS + sizeof(PersistentTables) <= 192 * ROW_B && sizeof(TileTables) <= TOKENS, "tables");
    if ((int)blockIdx.x < persistent_grid) {
        persistent_body<SWIGLU, W8, PAIRED, false>(persistent_of, SplitArgs{}, PersistentLds{lt0, lt1, lt2, lw2, lw0, lw1,
                                                   reinterpret_cast<unsigned long long*>(lw2 + TOKENS),
                                                   reinterpret_cast<PersistentTables*>(lt1 + TOKENS)}, persistent_grid);
        if (!CLAIMS || tiles_of.claims == nullptr) return;
        __syncthreads();                 // every wave has left the persistent body's LDS
    }
    TileTables& t = *reinterpret_cast<TileTables*>(W8 ? tile_tables : lt2);      // (the bf16 streamer has two token buffers)
    tile_body<SWIGLU, W8, CLAIMS>(tiles_of, TileLds{lw0, lw1, lw2, lt0, lt1, lt2}, t, (int)blockIdx.x - (CLAIMS && tiles_of.claims ? 0 : persistent_grid));
}

// The persistent body alone: one MLP's down projection in slices of k
__global__ __launch_bounds__(512) void grouped_gemm_persistent_split_kernel(GemmPair pair_of, SplitArgs split) {
    __shared__ __attribute__((aligned(1024))) uint8_t a0a[128 * ROW_B];
    __shared__ __attribute__((aligned(1024))) uint8_t a0b[128 * ROW_B];
    __shared__ __attribute__((aligned(1024))) uint8_t a1a[128 * ROW_B];
    __shared__ __attribute__((aligned(1024))) uint8_t a1b[128 * ROW_B];
    __shared__ __attribute__((aligned(1024))) uint8_t b0[BN_ROWS * ROW_B];
    __shared__ __attribute__((aligned(1024))) uint8_t b1[BN_ROWS * ROW_B];
    __shared__ unsigned long long ptr[4 * PE];
    __shared__ PersistentTables tables;
    persistent_body<false, true, false, true>(pair_of, split, PersistentLds{a0a, a0b, a1a, a1b, b0, b1, ptr, &tables}, (int)gridDim.x);
}

// CUs of the current device (one persistent workgroup on each)
inline int cu_count() {
    static int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    if (cached[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 0;
        cached[dev] = n;
    }
    return cached[dev];
}

// tiles of one workgroup each, whole rounds of 8 groups of 4
inline long tile_grid(long tiles) { return (tiles + 31) / 32 * 32; }

// Whether a bf16 down projection of tiles of one workgroup alone runs in half tiles: whole ones for at most half of the CUs, and rows that
// few experts have more than HALF_ROWS of; or whole ones for a second, part-filled round, and so few rows that hardly any expert is cut.
// Layers, us, whole -> half.  Half a round, Mixtral-8x7B, 20 / 64 / 128 / 200 tokens (means of 5 to 50 rows) 505 / 520 / 537 / 557 -> 459 / 471 / 485 /
// 500, 256 570 -> 576; two rounds, DeepSeek-V2-Lite, 20 / 32 / 64 / 128 (2 to 12) 130 / 137 / 152 / 176 -> 124 / 129 / 147 / 166, 256 and 400 the same and
// 205 -> 212.  Three quarters of a round, Mixtral-8x22B, 20 / 64 / 256: 775 / 755 / 834 whole, 790 / 778 / 937 in halves.
bool half_tiles_pay(const GemmArgs& g, int n_rows) {
    const long tiles = (long)(g.E < n_rows ? g.E : n_rows) * g.n_tiles_n, cus = cu_count();
    if (2 * tiles <= cus) return n_rows <= 48L * g.E;
    return tiles > cus && tiles <= 2 * cus && n_rows <= 16L * g.E;
}
int launch_half(GemmPair pair, int n_rows, hipStream_t st) {
    if (pair.shared_tiles > 0) {                 // (as many 256-column tiles of up to 192 rows; the host's bound of its rows follows)
        pair.p[1].n_tiles_n = (pair.p[1].N + 127) / 128;
        pair.shared_tiles = half_tiles_of(pair.shared_rows) * pair.p[1].n_tiles_n;
    }
    GemmArgs& g = pair.p[0];
    g.n_tiles_n = (g.N + 127) / 128;
    const long grid = tile_grid(((long)n_rows / HALF_ROWS + g.E) * g.n_tiles_n + pair.shared_tiles);
    hipLaunchKernelGGL(grouped_gemm_half_kernel, dim3((unsigned)grid), dim3(256), 0, st, pair);
    MOE_HIP_CHECK(hipGetLastError());
    return MOE_OK;
}

template <int WN, bool SWIGLU, bool W8>
int launch_tiles(const GemmPair& pair, int n_rows, hipStream_t st) {
    auto kern = grouped_gemm_kernel<WN, SWIGLU, W8, false>;
    const GemmArgs& g = pair.p[0];
    if constexpr (!W8 && !SWIGLU)
        if (half_tiles_pay(g, n_rows)) return launch_half(pair, n_rows, st);
    long tiles = ((long)n_rows / 128 + g.E) * g.n_tiles_n;             // sum_e tiles_of(c_e) <= sum_e (c_e / 128 + 1)
    if constexpr (!W8)
        if (g.cut_cus > 0) {
            kern = grouped_gemm_kernel<WN, SWIGLU, W8, true>;
            if (tiles < g.cut_cus) tiles = g.cut_cus;                  // (no more than that where rows are cut lower)
        }
    const long grid = tile_grid(tiles + pair.shared_tiles);
    if (grid > 0x7fffffffL) {
        set_error("grouped gemm: %ld workgroups exceed the grid limit", grid);
        return MOE_ERR_INVALID;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(128 * WN), 0, st, pair);
    MOE_HIP_CHECK(hipGetLastError());
    return MOE_OK;
}

// waves of 32 columns that the thin kernel's down projection has at most
inline long thin_down_waves(int E, int n_rows, bool shared, int N) { return ((E < n_rows ? E : n_rows) + (shared ? 1L : 0L)) * ((N + 31) / 32); }
// Up to two waves per CU: 16 columns each instead of 32, so that twice as many stages are on their way, and the waves combine
// too, which saves a launch where the host takes as long as the GPU.  Down projection and combine, us, in two launches -> this
// (16 columns): DeepSeek-V2-Lite, 1 token (448 waves) 13.5 + 4.7 -> 16.3; Mixtral-8x7B, 1 token (256) 56.1 + 5.7 -> 45.1, the call 161 ->
// 144.  Beyond, nothing is gained: DeepSeek-V2-Lite, 3 tokens (1216) 17.0 + 5.0 -> 22.8 with 32 columns, Mixtral-8x22B, 2 tokens (768),
// the call 405 -> 408.
inline bool thin_down_narrow(long waves) { return waves <= 2L * cu_count(); }

template <bool SWIGLU, bool W8>
int launch_thin(const GemmArgs& g, int n_rows, const GemmArgs* shared, LayerCall* call, hipStream_t st) {
    GemmPair pair{};
    pair.p[0] = g;
    if (shared) pair.p[1] = *shared;
    const long experts = g.E < n_rows ? g.E : n_rows;
    auto launch = [&](auto kernel, int ncol, const CombineTail& t) -> int {
        pair.shared_tiles = shared ? (shared->N + ncol - 1) / ncol : 0;
        const long grid = experts * ((g.N + ncol - 1) / ncol) + pair.shared_tiles;
        if (grid > 0x7fffffffL) {
            set_error("grouped gemm: %ld workgroups exceed the grid limit", grid);
            return MOE_ERR_INVALID;
        }
        hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64), 0, st, pair, t);
        MOE_HIP_CHECK(hipGetLastError());
        return MOE_OK;
    };
    if constexpr (SWIGLU) {
        return launch(grouped_gemm_thin_kernel<true, W8, 2, false>, 16, CombineTail{});
    } else {
        const long waves = thin_down_waves(g.E, n_rows, shared != nullptr, g.N);
        if (!thin_down_narrow(waves)) return launch(grouped_gemm_thin_kernel<false, W8, 2, false>, 32, CombineTail{});
        if (!call || !call->tail) return launch(grouped_gemm_thin_kernel<false, W8, 1, false>, 16, CombineTail{});
        call->combined = true;
        return launch(grouped_gemm_thin_kernel<false, W8, 1, true>, 16, *call->tail);
    }
}

// 4 GiB of gathered rows or more: only the register-staged body addresses them
inline bool gather_fits(const GemmArgs& g) { return !g.row_map || g.a_bytes < (1ull << 32); }

// How the down projection of one MLP is cut in k, slices == 0 where that does not pay: only where k is long (32 blocks, 4096), so
// that what the slices save outweighs their sums' way through memory, and where its own tiles leave CUs idle.
//  * up to 256 rows on the split kernel: as many slices as fill the CUs once, of 8 blocks or more (a shorter k loop is mostly
//    its own start), at most 16.
//  * above, up to a round of 256-row tiles, whichever of three takes least by these counts (us), each at its best number of slices: uncut,
//    1.55 a block of k while the pieces leave a third of the CUs idle, 15 % more up to a round of them and 60 % beyond; the split
//    kernel, one round, 0.9 + 0.0055 a row of its tiles a block and 0.37 per MB of sums; the persistent body's 256-row tiles, 2.8
//    a block, 20 a further round and 0.16 per MB.  The split kernel's lower tiles win where slices are short or tiles few.
// Measured: h of 1024 to 8192, k of 4096 to 18432, 257 to 3000 rows, all three at every number of slices: the counts are within 12 %
// and the choice 0.5 % behind the best of them in the mean, 5 % at most.  Down projection, us, uncut / split kernel / 256-row tiles:
// h 7168, k 18432, 257 rows 212 / 112 / 121, 400: 238 / 133 / 125, 640: 216 / - / 170, 1000: 264 / - / 231, 1300: 360 / - / 340;
// 4096, 14336, 257: 164 / 50 / 63, 768: 167 / 102 / 91; 2048, 5632, 257: 72 / 24 / 40, 1000: 71 / 37 / 44; 1024, 4096, 1000: 55 / 26 / 40.
SplitPlan split_plan(int n_rows, int K, int n_tiles_n) {
    const int nblk = K / 128, cus = cu_count();
    if (nblk < 32 || n_rows < 1 || cus < 8) return SplitPlan{};
    int m = (n_rows + 127) / 128;
    const int rows = m <= 1 ? n_rows : ((n_rows + m - 1) / m + 15) / 16 * 16;
    if (n_rows <= 256) {
        if ((long)m * n_tiles_n * 2 > cus) return SplitPlan{};
        m = (n_rows + rows - 1) / rows;
        int s = cus / (m * n_tiles_n);
        s = s < nblk / 8 ? s : nblk / 8;
        s = s < 16 ? s : 16;
        const int blocks = (nblk + s - 1) / s;
        return SplitPlan{m, rows, (nblk + blocks - 1) / blocks, blocks};
    }
    m = (n_rows + rows - 1) / rows;
    const int m256 = (n_rows + 255) / 256, left = n_rows & 255;
    const long tiles = (long)m256 * n_tiles_n;
    if (tiles > cus) return SplitPlan{};
    const bool own = left > 0 && left <= 192;                        // (uncut, these rows are a one-workgroup tile)
    const long pieces = (2 * (m256 - (own ? 1 : 0)) + (own ? 1 : 0)) * (long)n_tiles_n;
    double best = 4.0 + 1.55 * nblk * (3 * pieces <= 2 * cus ? 1.0 : pieces <= cus ? 1.15 : 1.6);
    SplitPlan plan{};
    auto consider = [&](double us, const SplitPlan& p) {
        if (us < best) {
            best = us;
            plan = p;
        }
    };
    for (int s = 2; s <= 16 && nblk / s >= 8; ++s) {
        const int blocks = (nblk + s - 1) / s, slices = (nblk + blocks - 1) / blocks;
        const double mb = 1e-6 * slices * n_rows * (double)n_tiles_n * 1024;
        if (((long)slices * n_tiles_n + 7) / 8 * 8 * m <= cus)
            consider(8.0 + blocks * (0.9 + 0.0055 * rows) + 0.37 * mb, SplitPlan{m, rows, slices, blocks});
        const long rounds = (tiles * slices + cus - 1) / cus;
        consider(16.0 + 20.0 * (rounds - 1) + 2.8 * rounds * blocks + 0.16 * mb, SplitPlan{m256, 256, slices, blocks});
    }
    return plan;
}

// waves of a workgroup of gate_up_few_rows_kernel, 0 where the others serve the call: one MLP, up to 96 rows, of as many columns as
// make a workgroup of 8 to 10 waves for every CU.  (Fewer columns: what its workgroups would have to share of the token rows grows.)
int few_rows_waves(const GemmArgs& g, int n_rows) {
    const int cus = cu_count();
    if (g.E != 1 || n_rows > DM_ROWS || cus < 8) return 0;
    const int waves = (g.N / 8 + cus - 1) / cus;
    return waves >= 8 && waves <= DM_WAVES && g.K < 1 << 15 ? waves : 0;
}
int launch_few_rows(const GemmArgs& g, int n_rows, int waves, hipStream_t st) {
    const dim3 grid((unsigned)((g.N / 8 + waves - 1) / waves)), block((unsigned)(64 * waves));
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, st, g, n_rows); };
    switch ((n_rows + 15) / 16) {
#define MOE_DM_CASE(n) case n: launch(gate_up_few_rows_kernel<n>); break;
    MOE_DM_CASE(1) MOE_DM_CASE(2) MOE_DM_CASE(3) MOE_DM_CASE(4) MOE_DM_CASE(5)
#undef MOE_DM_CASE
    default: launch(gate_up_few_rows_kernel<6>); break;
    }
    MOE_HIP_CHECK(hipGetLastError());
    return MOE_OK;
}

int launch_split(const GemmArgs& g, int n_rows, const SplitPlan& plan, float* part, hipStream_t st) {
    const int pieces = plan.slices * g.n_tiles_n;
    if (plan.rows == 256) {
        GemmPair pair{};
        pair.p[0] = g;
        pair.p[0].rem_split = 1;                 // every row on this kernel's tiles, the last one padded
        const long tiles = (long)pieces * plan.m_tiles, ncu = (cu_count() / 8) * 8, grid = (tiles + 7) / 8 * 8;
        hipLaunchKernelGGL(grouped_gemm_persistent_split_kernel, dim3((unsigned)(grid < ncu ? grid : ncu)), dim3(512), 0, st, pair,
                           SplitArgs{plan, n_rows, part});
    } else {
        hipLaunchKernelGGL(grouped_gemm_split_kernel, dim3((pieces + 7) / 8 * 8 * plan.m_tiles), dim3(512), 0, st, g, n_rows, plan, part);
    }
    hipLaunchKernelGGL(add_slices_kernel, dim3((unsigned)(((size_t)n_rows * g.N / 4 + 255) / 256)), dim3(256), 0, st, part, g.offsets, g.c,
                       n_rows, g.N, plan.slices);
    MOE_HIP_CHECK(hipGetLastError());
    return MOE_OK;
}

// Whether a call in which no expert has more than 16 rows goes to the thin kernel, `shared` a second problem of the launch
// or NULL.  Where rows are few for the number of experts it does: which experts have rows, and so how many tiles there are, is not
// known here, and the tile kernel loses most where they fill its last round badly.  From three rows per expert on nearly all
// have some.  Both kernels then stream the same weights, and what differs is how full their rounds are: a tile of 256 weight rows is
// a workgroup of the tile kernel, one per CU, and 8 waves of the thin kernel, six per CU, so a round of the latter is 3/4 as many
// tiles.  A wave's token rows cost it 1 % each; K up to 2048 costs the tile kernel 7 % around its short k loop; and with K of 8192
// and more the tile kernel streams at the full rate from 139 of 256 tiles on, the thin one not always.  Measured (us, thin / tile):
//   Mixtral-8x22B, 3 rows each  gate/up 474 / 466, down 279 / 234;  16 rows 526 / 480, 266 / 234;  layer, 12 tokens 687 / 675, 16: 778 / 739
//   Mixtral-8x7B, 3 rows each   gate/up 278 / 289, down 138 / 182;  16 rows 298 / 294, 150 / 187
//   DeepSeek-V2-236B, 4 rows    gate/up 758 / 751, down 382 / 396;  16 rows 844 / 769, 454 / 434
//   DeepSeek-V3, 4 rows         gate/up 1128 / 1104, down 585 / 594;  16 rows 1367 / 1146, 751 / 680
// and below three rows per expert, layers: Mixtral-8x22B, 8 tokens 408 / 461; DeepSeek-V2-236B, 6 tokens 221 / 261; V2-Lite, 16: 99 / 114.
bool thin_pays(const GemmArgs& g, int n_rows, const GemmArgs* shared) {
    if (n_rows < 3L * g.E) return true;
    const double tiles = (double)g.E * g.n_tiles_n + (shared ? shared->n_tiles_n : 0);
    const double cus = cu_count(), round = 0.75 * cus;
    if (g.K >= 8192 && tiles <= round && tiles > 139.0 / 256 * cus) return false;
    const double thin = std::ceil(tiles / round) * round * (1.0 + 0.01 * ((double)n_rows / g.E - 1.0));
    return thin < std::ceil(tiles / cus) * cus * (g.K <= 2048 ? 1.07 : 1.0);
}

// The persistent body needs an even number of k-stages for its hand-over (fp8 sizes always have one), keeps per-expert
// tables for up to 512 experts and addresses gathered rows with 32-bit offsets.
inline bool persistent_fits(const GemmArgs& g) { return g.K % 128 == 0 && g.E <= 512 && gather_fits(g) && cu_count() >= 8; }

// the rules by which a call's tiles fall to the two kinds of workgroups (reasons in launch_mt)
template <bool W8>
GemmArgs both_kernels(GemmArgs g) {
    g.alone = 0;
    g.cold_max = 192;
    g.rem_split = W8 ? 1 : 0;
    g.pair_rows = W8 ? 0 : 1;
    g.tail_cus = (cu_count() / 8) * 8;     // the persistent workgroups when there is a round of tiles or more
    return g;
}

template <bool SWIGLU, bool W8>
int launch_both(const GemmPair& pair, int n_rows, hipStream_t st) {
    const GemmArgs& g = pair.p[0];
    const SharedTiles shared = pair.shared_rows > 0 ? shared_tiles_bound<W8>(pair.p[1], pair.shared_rows) : SharedTiles{};
    const long ncu = (cu_count() / 8) * 8, own = ((long)n_rows / 256 + g.E) * g.n_tiles_n + shared.persistent;
    const long persistent = own < ncu ? (own + 7) / 8 * 8 : ncu;
    // one tile per expert that has rows (bf16 weights: two), the shared expert's, and a last round's pieces (at most two for each CU)
    const long tiles = tile_grid((W8 ? 1 : 2) * (long)(g.E < n_rows ? g.E : n_rows) * g.n_tiles_n + shared.own + 2 * g.tail_cus);
    const long grid = pair.claims ? ncu : persistent + tiles;
    if (grid > 0x7fffffffL) {
        set_error("grouped gemm: %ld workgroups exceed the grid limit", grid);
        return MOE_ERR_INVALID;
    }
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(512), 0, st, pair, pair, (int)persistent); };
    if (pair.shared_rows > 0) launch(grouped_gemm_both_kernel<SWIGLU, W8, true, true>);
    else if (pair.claims) launch(grouped_gemm_both_kernel<SWIGLU, W8, false, true>);
    else launch(grouped_gemm_both_kernel<SWIGLU, W8, false, false>);
    MOE_HIP_CHECK(hipGetLastError());
    return MOE_OK;
}

// counters for one launch of a layer call
inline int32_t* next_claims(LayerCall* call) {
    if (!call || !call->claims) return nullptr;
    int32_t* const c = call->claims;
    call->claims += kClaimInts;
    return c;
}

// max_rows: no expert has more rows (callers that do not know pass n_rows)
template <bool SWIGLU, bool W8>
int launch_mt(const GemmArgs& g0, int n_rows, int max_rows, void* workspace, size_t workspace_bytes, LayerCall* call, hipStream_t st) {
    GemmArgs g = g0;
    if constexpr (W8 && !SWIGLU) {
        const SplitPlan plan = g.E == 1 && workspace ? split_plan(n_rows, g.K, g.n_tiles_n) : SplitPlan{};
        if (plan.slices > 1 && workspace_bytes >= (size_t)plan.slices * n_rows * g.N * 4)
            return launch_split(g, n_rows, plan, static_cast<float*>(workspace), st);
    }
    if constexpr (W8 && SWIGLU) {
        const int waves = gather_fits(g) ? few_rows_waves(g, n_rows) : 0;
        if (waves > 0) return launch_few_rows(g, n_rows, waves, st);
    }
    if (max_rows <= 16 && gather_fits(g) && thin_pays(g, n_rows, nullptr)) return launch_thin<SWIGLU, W8>(g, n_rows, nullptr, call, st);
    GemmPair pair{};
    pair.claims = next_claims(call);
    // (One MLP of up to 192 rows has tiles of one workgroup alone too, and the sums of a call of both kinds.  As such a call its
    // persistent workgroups found no tile and took the first 5 us: DeepSeek-V3's dense MLP, 128 / 160 / 192 tokens 167 / 183 / 203 -> 152 / 175 /
    // 189 us with one upload less.)
    const bool one_kind = !both_kinds<W8>(n_rows, g.E, g.K, g.N) || !persistent_fits(g);
    if (one_kind || (g.E == 1 && n_rows <= 192)) {
        g.alone = one_kind;
        if (!W8 && (long)g.E * g.n_tiles_n <= cu_count()) g.cut_cus = cu_count();
        pair.p[0] = g;
        return launch_tiles<4, SWIGLU, W8>(pair, n_rows, st);
    }
    // The counts themselves live on the device; only their mean is known here.  Every expert goes by its own count: what
    // fits one tile of a workgroup of its own runs there, at its own height and without 256-row padding, the rest on the
    // persistent workgroups' 256-row tiles.  (As two launches:) DeepSeek-V2-Lite, 4096 tokens (64 experts of
    // 0 ... 3989 rows, 47 of them below 193, whose 256-row tiles were 49 % padding): block step 0.923 -> 0.847 ms,
    // routed gate/up 0.395 -> 0.355 ms; DeepSeek-V2-236B, 32768 tokens: 11.48 -> 11.39 ms.
    // fp8 weights: the rule is applied to what an expert's full 256-row tiles leave over.  A ragged
    // last tile costs a persistent workgroup a full tile of MFMA time; a one-workgroup tile streams the expert's weights
    // once more for it, and fp8 weights are half the bytes.  DeepSeek-V3, 65536 tokens (256 experts of 581 ... 3941
    // rows, every second one with at most 128 rows over): block step 46.3 -> 45.8 ms, routed gate/up 25.2 -> 24.8,
    // down 12.9 -> 12.7 (with up to 64 or 96 rows over 46.2 - 46.3; with all, as two 128-row tiles, 47.1).  Up to 192
    // rows over, on the streamer form for 129 to 192 rows: the headline step stays (45.95 -> 45.85), DeepSeek-V3 at
    // 3584 / 4096 / 8192 tokens 4.53 -> 3.99, 4.64 -> 4.31, 7.50 -> 7.41 ms (at 4096 tokens 109 of the 256 experts hold
    // 129 to 192 rows, which were padded 256-row tiles).  With bf16
    // weights it is break-even (Mixtral-8x7B 9.28 -> 9.23 ms, DeepSeek-V2-236B 11.34 -> 11.42) and not done.
    // Last round of the persistent body (tail_of above), as halves: Mixtral-8x22B, 8192 tokens, down projection (6.4 rounds
    // of 0.4 ms) 2.82 -> 2.66 ms, step 8.31 -> 8.13; Mixtral-8x7B 9.39 -> 9.27 ms; DeepSeek-V2-Lite 0.855 -> 0.821 ms
    // (its shared expert's 128 down tiles become 256 half tiles: 0.071 -> 0.055 ms); DeepSeek-V2-236B 11.43 -> 11.46,
    // DeepSeek-V3 46.56 -> 46.54: short rounds gain nothing, a partial round of few CUs runs at a higher clock anyway.
    pair.p[0] = both_kernels<W8>(g);
    // One fp8 expert (a dense MLP): the rows are known here.  What its full tiles leave over goes to the persistent body's space too,
    // as a padded tile, where that shortens the rounds by the same count.  It does where the last round then runs in three or four
    // pieces a tile, which tiles of another kind beside it rule out: calls of few tiles, and of a few more than whole rounds.  Whole MLP
    // without scratch, us, apart -> padded: hidden 5120, intermediate 3072, 300 / 440 / 660 rows 118 / 148 / 133 -> 100 / 99 / 115, 7168 x 2048 129 /
    // 163 / 146 -> 112 / 110 / 117, 2048 x 4096 93 / 117 / 104 -> 83 / 84 / 87, DeepSeek-V3's (its down projection) 377 / 548 / 583 -> 352 / 452 / 575.  Done
    // always, it would be 441 instead of 352 at 300 rows, 726 (651) at 800, 1070 (985) at 1300, 1489 (1396) at 2100.
    if (W8 && g.E == 1 && own_tiles<W8>(pair.p[0], n_rows) > 0) {
        const int cus = pair.p[0].tail_cus, full = (n_rows >> 8) * g.n_tiles_n;
        const RoundCost apart = round_cost(full, g.n_tiles_n, (n_rows & 255) > kTallRows, cus), padded = round_cost(full + g.n_tiles_n, 0, false, cus);
        const int a = apart.move < apart.keep ? apart.move : apart.keep, b = padded.move < padded.keep ? padded.move : padded.keep;
        if (b < a) pair.p[0].cold_max = 0;
    }
    return launch_both<SWIGLU, W8>(pair, n_rows, st);
}

inline bool joint_thin(const GemmArgs& routed, int n_rows, int max_rows, const GemmArgs& shared, int n_shared) {
    return max_rows <= 16 && n_shared <= 16 && thin_pays(routed, n_rows, &shared);
}

// The shared expert's tiles in the routed experts' launches.  both: see joint_both; shared.alone: see joint_alone.
template <bool SWIGLU, bool W8>
int launch_joint(const GemmArgs& routed, int n_rows, int max_rows, const GemmArgs& shared, int n_shared, bool both, LayerCall* call, hipStream_t st) {
    if (joint_thin(routed, n_rows, max_rows, shared, n_shared))
        return launch_thin<SWIGLU, W8>(routed, n_rows, SWIGLU && call && call->shared_gate_up_done ? nullptr : &shared, call, st);
    GemmPair pair{{routed, shared}, 0, 0, next_claims(call)};
    if (!both) {
        pair.p[0].alone = 1;
        pair.shared_tiles = tiles_of<!W8>(n_shared) * shared.n_tiles_n;
        pair.shared_rows = n_shared;
        return launch_tiles<4, SWIGLU, W8>(pair, n_rows, st);
    }
    pair.p[0] = both_kernels<W8>(routed);
    pair.p[1] = both_kernels<W8>(shared);
    pair.shared_rows = n_shared;
    return launch_both<SWIGLU, W8>(pair, n_rows, st);
}

int check_group(const moe_mlp_group& m, int32_t hidden, bool w8, const char* who) {
    MOE_REQUIRE(m.n_rows >= 0, "%s: n_rows %d < 0", who, m.n_rows);
    if (m.n_rows == 0) return MOE_OK;
    MOE_REQUIRE(m.x && m.w_gate && m.w_up && m.w_down && m.offsets && m.act && m.y, "%s: NULL pointer argument", who);
    MOE_REQUIRE(m.x_rows >= 1, "%s: x_rows %d < 1", who, m.x_rows);
    MOE_REQUIRE(!w8 || (m.s_gate && m.s_up && m.s_down), "%s: NULL scale pointer array", who);
    MOE_REQUIRE(m.n_experts >= 1 && m.n_experts <= MAX_E, "%s: n_experts %d outside [1,%d]", who, m.n_experts, MAX_E);
    const int align = w8 ? 128 : 64;
    MOE_REQUIRE(hidden > 0 && hidden % align == 0, "%s: hidden %d must be a positive multiple of %d", who, hidden, align);
    MOE_REQUIRE(m.inter > 0 && m.inter % align == 0, "%s: intermediate %d must be a positive multiple of %d", who, m.inter,
                align);
    return MOE_OK;
}

GemmArgs gate_up_args(const moe_mlp_group& m, int32_t hidden) {
    GemmArgs g{};
    g.a = static_cast<const uint16_t*>(m.x);
    g.row_map = m.row_map;
    g.a_bytes = (size_t)m.x_rows * (size_t)hidden * 2;
    g.a_rows = m.x_rows;
    g.b0 = m.w_gate; g.b1 = m.w_up; g.s0 = m.s_gate; g.s1 = m.s_up;
    g.offsets = m.offsets;
    g.c = static_cast<uint16_t*>(m.act);
    g.E = m.n_experts; g.K = hidden; g.N = m.inter;
    g.n_tiles_n = (m.inter + 127) / 128;
    return g;
}

GemmArgs down_args(const moe_mlp_group& m, int32_t hidden) {
    GemmArgs g{};
    g.a = static_cast<const uint16_t*>(m.act);
    g.b0 = m.w_down; g.s0 = m.s_down;
    g.offsets = m.offsets;
    g.c = static_cast<uint16_t*>(m.y);
    g.E = m.n_experts; g.K = m.inter; g.N = hidden;
    g.n_tiles_n = (hidden + 255) / 256;
    return g;
}

// no expert of the group has more rows than this
int row_bound(const moe_mlp_group& m) { return m.max_rows > 0 && m.max_rows < m.n_rows ? m.max_rows : m.n_rows; }

// Whether a call of the group by itself, with the scratch that it brings, cuts its down projection into slices of k
bool sliced(const moe_mlp_group& m, int32_t hidden) {
    const size_t need = moe_mlp_workspace_bytes(&m, hidden);
    return need > 0 && m.workspace && m.workspace_bytes >= need;
}

// Whether 256-row tiles of the group (its gate and up projection) are fewer than 3/8 of the CUs
bool few_tiles(const moe_mlp_group& m, long cus) { return (long)(m.n_rows / 256 + 1) * ((m.inter + 127) / 128) * 8 < 3 * cus; }

bool both_kinds_of(bool w8, const moe_mlp_group& m, int32_t hidden) {
    return (w8 ? both_kinds<true> : both_kinds<false>)(m.n_rows, m.n_experts, hidden, m.inter);
}

// Whether a joint call has tiles of both kinds: the routed experts' call would, and the persistent body can address both problems.
// (Where it cannot, for sizes that are odd multiples of 64, the call has one kind of tiles, like one of a lower mean.)
bool joint_both(bool w8, const moe_mlp_group& routed, const moe_mlp_group& shared, int32_t hidden) {
    return both_kinds_of(w8, routed, hidden) && shared.n_rows >= 128 && hidden % 128 == 0 && routed.inter % 128 == 0 &&
           shared.inter % 128 == 0 && routed.n_experts <= 512 && cu_count() >= 8;
}

// Whether the shared expert's tiles join the routed experts' launches.  Where the joint call has both kinds of tiles they do if a
// call of its own would have both as well (128 rows, no slices of k), up to four rounds of tiles of its own (beyond, the same
// within 0.2 %): the two then fill their last rounds together.  Where it has one-workgroup tiles (or the
// thin kernel's waves) alone, below a mean of 128 rows, a few tiles always do; more of them up to two of that kernel's 128-row tiles, all that
// the shared expert gets there, per CU, unless its own call is in slices.
// Layers, us, apart -> joined.  Both kinds: DeepSeek-V2-Lite 1400 / 2000 / 2777 / 4096 tokens 439 / 514 / 585 / 725 -> 397 / 470 /
// 563 / 699; DeepSeek-V3 4096 / 6000 4046 / 5498 -> 4004 / 5367, 16384 the same.  One kind: DeepSeek-V2-Lite 1024 / 1300 366 /
// 409 -> 322 / 351, its hidden size 2112 instead of 2048, 1000 tokens, 335 -> 316; DeepSeek-V2-236B 1024 / 1500 1463 / 1641 -> 1416 / 1615, 2048 the same, 3000 2074 -> 2090 (not joined: 576 tiles);
// DeepSeek-V3 1500 / 2997 / 4000 2507 / 3437 / 4139 -> 2470 / 3382 / 4120.
bool joins(const moe_mlp_group& routed, const moe_mlp_group& shared, int32_t hidden) {
    if (routed.n_rows < 1 || shared.n_rows < 1 || routed.n_experts < 1 || shared.n_experts != 1 || hidden < 1) return false;
    if (routed.row_map && (size_t)routed.x_rows * (size_t)hidden * 2 >= (1ull << 32)) return false;
    if (shared.row_map && (size_t)shared.x_rows * (size_t)hidden * 2 >= (1ull << 32)) return false;
    const long cus = cu_count(), cols = (shared.inter + 127) / 128, rows = shared.n_rows;
    if (joint_both(routed.fp8, routed, shared, hidden)) return (rows + 255) / 256 * cols <= 4 * cus && !sliced(shared, hidden);
    return routed.n_rows / routed.n_experts < 128 &&
           (few_tiles(shared, cus) || ((rows + 127) / 128 * cols <= 2 * cus && !sliced(shared, hidden)));
}

// fp8 weights, a joint call that one kernel serves: whether the shared expert's sums start at the stages of that kernel's own
// calls.  They do where it is small, 256-row tiles for less than 3/8 of the CUs, and where a call of its own would do the same (a
// mean below 128); else at stage 0, as in a call of its own, whose bits it then has.  DeepSeek-V3, us, 1300 /
// 1500 / 2997 / 4000 tokens (all of the second kind): started as the first kind 2337 / 2437 / 3387 / 4082, at stage 0
// 2340 / 2449 / 3392 / 4081.
int joint_alone(const moe_mlp_group& shared) { return shared.n_rows < 128 || few_tiles(shared, cu_count()); }

template <bool W8>
int grouped_swiglu(const moe_mlp_group& m, int32_t hidden, int32_t phases, LayerCall* call, void* stream, const char* who) {
    MOE_REQUIRE(phases >= MOE_PHASE_GATE_UP && phases <= MOE_PHASE_BOTH, "%s: bad phases %d", who, phases);
    int rc = check_group(m, hidden, W8, who);
    if (rc != MOE_OK || m.n_rows == 0) return rc;
    hipStream_t st = as_stream(stream);
    if (phases & MOE_PHASE_GATE_UP) rc = launch_mt<true, W8>(gate_up_args(m, hidden), m.n_rows, row_bound(m), nullptr, 0, call, st);
    if (rc == MOE_OK && (phases & MOE_PHASE_DOWN)) 
        rc = launch_mt<false, W8>(down_args(m, hidden), m.n_rows, row_bound(m), m.workspace, m.workspace_bytes, call, st);
    return rc;
}

template <bool W8>
int grouped_swiglu_joint(const moe_mlp_group& r, const moe_mlp_group& s, int32_t hidden, int32_t phases, LayerCall* call, void* stream, const char* who) {
    MOE_REQUIRE(phases >= MOE_PHASE_GATE_UP && phases <= MOE_PHASE_BOTH, "%s: bad phases %d", who, phases);
    int rc = check_group(r, hidden, W8, who);
    if (rc == MOE_OK) rc = check_group(s, hidden, W8, who);
    if (rc != MOE_OK) return rc;
    if (!joins(r, s, hidden)) {
        if (call) call->tail = nullptr;              // (what the routed experts add up is not the whole layer)
        rc = grouped_swiglu<W8>(r, hidden, phases, call, stream, who);
        return rc != MOE_OK ? rc : grouped_swiglu<W8>(s, hidden, phases, call, stream, who);
    }
    hipStream_t st = as_stream(stream);
    GemmArgs gate_up = gate_up_args(s, hidden), down = down_args(s, hidden);
    const bool both = joint_both(W8, r, s, hidden);
    if (W8) gate_up.alone = down.alone = joint_alone(s);
    if (phases & MOE_PHASE_GATE_UP)
        rc = launch_joint<true, W8>(gate_up_args(r, hidden), r.n_rows, row_bound(r), gate_up, s.n_rows, both, call, st);
    if (rc == MOE_OK && (phases & MOE_PHASE_DOWN))
        rc = launch_joint<false, W8>(down_args(r, hidden), r.n_rows, row_bound(r), down, s.n_rows, both, call, st);
    return rc;
}

// out = bf16(f32(q) * scale[i/128, j/128]); one thread per 16 consecutive elements of a row
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ q, const float* __restrict__ scale,
                                                      int rows, int cols, uint16_t* __restrict__ out) {
    const int chunks = (cols + 15) / 16;
    const long id = (long)blockIdx.x * 256 + threadIdx.x;
    if (id >= (long)rows * chunks) return;
    const int r = (int)(id / chunks), c0 = (int)(id % chunks) * 16;
    const int nbc = (cols + 127) / 128;
    const float s = scale[(size_t)(r >> 7) * nbc + (c0 >> 7)];  // a 16-aligned run never crosses a 128 boundary
    const size_t base = (size_t)r * cols + c0;
    if (c0 + 16 <= cols && (base & 15) == 0) {
        u32x4 l, h;
        dequant16(*reinterpret_cast<const u32x4*>(q + base), s, l, h);
        *reinterpret_cast<u32x4*>(out + base) = l;
        *reinterpret_cast<u32x4*>(out + base + 8) = h;
    } else {
        for (int j = c0; j < cols && j < c0 + 16; ++j) {
            f32x2 f = __builtin_amdgcn_cvt_pk_f32_fp8((uint32_t)q[(size_t)r * cols + j], false);
            out[(size_t)r * cols + j] = (uint16_t)(pack_bf16(f[0] * s, 0.0f) & 0xffffu);
        }
    }
}

int swiglu_groups(const moe_mlp_group& routed, const moe_mlp_group* shared, int32_t hidden, int32_t fp8, int32_t phases, LayerCall* call,
                  void* stream) {
    const char* who = "moe_grouped_swiglu_joint";
    if (shared == nullptr)
        return fp8 ? grouped_swiglu<true>(routed, hidden, phases, call, stream, who) : grouped_swiglu<false>(routed, hidden, phases, call, stream, who);
    return fp8 ? grouped_swiglu_joint<true>(routed, *shared, hidden, phases, call, stream, who)
               : grouped_swiglu_joint<false>(routed, *shared, hidden, phases, call, stream, who);
}

}  // namespace

bool layer_may_combine(int32_t n_experts, int32_t n_rows, bool shared, int32_t hidden) {
    return thin_down_narrow(thin_down_waves(n_experts, n_rows, shared, hidden));
}

bool layer_shared_first(const moe_mlp_group& routed, const moe_mlp_group& shared, int32_t hidden) {
    if (hidden < (routed.fp8 ? 6144 : 2048)) return false;
    if (router_shared_front(routed.n_experts) + shared_first_blocks(shared.inter) > cu_count()) return false;
    return shared.n_rows > 0 && check_group(routed, hidden, routed.fp8, "moe_layer_forward") == MOE_OK &&
           check_group(shared, hidden, shared.fp8, "moe_layer_forward") == MOE_OK && joins(routed, shared, hidden) &&
           joint_thin(gate_up_args(routed, hidden), routed.n_rows, row_bound(routed), gate_up_args(shared, hidden), shared.n_rows);
}

bool layer_claims(const moe_mlp_group& routed, const moe_mlp_group* shared, int32_t hidden) {
    return both_kinds_of(routed.fp8, routed, hidden) || (shared && both_kinds_of(shared->fp8, *shared, hidden));
}

bool layer_joins(const moe_mlp_group& routed, const moe_mlp_group& shared, int32_t hidden) { return joins(routed, shared, hidden); }

int layer_experts(const moe_mlp_group& routed, const moe_mlp_group* shared, int32_t hidden, int32_t fp8, LayerCall* call, void* stream) {
    return swiglu_groups(routed, shared, hidden, fp8, MOE_PHASE_BOTH, call, stream);
}

}  // namespace moe

extern "C" size_t moe_grouped_workspace_bytes(int32_t, int32_t) { return 256; }

extern "C" int moe_grouped_swiglu_bf16(const void* x, int32_t x_rows, const int32_t* row_map, const void* const* w_gate,
                                       const void* const* w_up, const void* const* w_down, const int32_t* offsets,
                                       int32_t n_rows, int32_t n_experts, int32_t hidden, int32_t inter, void* act,
                                       void* y, int32_t phases, void*, size_t, void* stream) {
    const moe_mlp_group m{x, x_rows, n_rows, row_map, w_gate, w_up, w_down, nullptr, nullptr, nullptr, offsets, n_experts, inter, 0, 0, act, y, nullptr, 0};
    return moe::grouped_swiglu<false>(m, hidden, phases, nullptr, stream, "moe_grouped_swiglu_bf16");
}

extern "C" int moe_grouped_swiglu_w8a16(const void* x, int32_t x_rows, const int32_t* row_map, const void* const* w_gate,
                                        const void* const* w_up, const void* const* w_down,
                                        const float* const* s_gate, const float* const* s_up,
                                        const float* const* s_down, const int32_t* offsets, int32_t n_rows,
                                        int32_t n_experts, int32_t hidden, int32_t inter, void* act, void* y,
                                        int32_t phases, void*, size_t, void* stream) {
    const moe_mlp_group m{x, x_rows, n_rows, row_map, w_gate, w_up, w_down, s_gate, s_up, s_down, offsets, n_experts, inter, 0, 0, act, y, nullptr, 0};
    return moe::grouped_swiglu<true>(m, hidden, phases, nullptr, stream, "moe_grouped_swiglu_w8a16");
}

extern "C" int moe_grouped_swiglu_joint(const moe_mlp_group* routed, const moe_mlp_group* shared, int32_t hidden, int32_t fp8,
                                        int32_t phases, void* stream) {
    using namespace moe;
    MOE_REQUIRE(routed != nullptr, "moe_grouped_swiglu_joint: NULL group");
    return swiglu_groups(*routed, shared, hidden, fp8, phases, nullptr, stream);
}

extern "C" size_t moe_mlp_workspace_bytes(const moe_mlp_group* m, int32_t hidden) {
    using namespace moe;
    if (m == nullptr || !m->fp8 || m->n_experts != 1 || m->n_rows < 1 || hidden < 1) return 0;
    const SplitPlan plan = split_plan(m->n_rows, m->inter, (hidden + 255) / 256);
    return plan.slices > 1 ? (size_t)plan.slices * m->n_rows * hidden * 4 : 0;
}

extern "C" int moe_shared_joins(const moe_mlp_group* routed, const moe_mlp_group* shared, int32_t hidden) {
    return routed && shared && moe::joins(*routed, *shared, hidden) ? 1 : 0;
}

extern "C" int moe_dequant_fp8_block128(const void* q, const float* scale, int32_t rows, int32_t cols, void* out,
                                        void* stream) {
    using namespace moe;
    MOE_REQUIRE(rows >= 0 && cols >= 0, "moe_dequant_fp8_block128: negative shape %d x %d", rows, cols);
    if (rows == 0 || cols == 0) return MOE_OK;
    MOE_REQUIRE(q && scale && out, "moe_dequant_fp8_block128: NULL pointer argument");
    const long chunks = (long)rows * ((cols + 15) / 16);
    hipLaunchKernelGGL(dequant_kernel, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, as_stream(stream),
                       static_cast<const uint8_t*>(q), scale, rows, cols, static_cast<uint16_t*>(out));
    MOE_HIP_CHECK(hipGetLastError());
    return MOE_OK;
}
