// In which order loads into registers and DMA into LDS retire.  Each wave requests cold lines one way and hot lines the other
// way behind them, waits until only the younger operations may be in flight, and compares what has arrived.  The cold
// buffer (1 GiB) holds in every word its index; every access stays inside it or inside the hot 4 KiB.
//   build/vmem_order
#include <cstdint>
#include <cstdio>

#include <hip/hip_runtime.h>

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) uint8_t* lds_u8;

#define CHECK(x)                                                                                  \
    do {                                                                                          \
        const hipError_t rc = (x);                                                                \
        if (rc != hipSuccess) { printf("%s: %s\n", #x, hipGetErrorString(rc)); return 1; }         \
    } while (0)

constexpr uint32_t COLD_BYTES = 1u << 30, HOT_BYTES = 4096, BLOCKS = COLD_BYTES / 4096, STALE = 0xdead;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, 0x00020000);
}
// a 4 KiB block of the cold buffer for every id
__device__ __forceinline__ uint32_t cold_block(uint64_t id) { return (uint32_t)((id * 2654435761ull >> 3) % BLOCKS) * 4096u; }

// a cold register load, four hot DMA behind it
__global__ __launch_bounds__(512) void register_load_first(const uint32_t* cold, const uint32_t* hot, uint32_t* missing, int iters) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[8 * 4096];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const auto rc = rsrc(cold, COLD_BYTES), rh = rsrc(hot, HOT_BYTES);
    uint32_t bad = 0;
    for (int it = 0; it < iters; ++it) {
        const uint32_t off = cold_block(((uint64_t)blockIdx.x * 8 + wave) * iters + it) + lane * 16u;
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        uint32_t v = __builtin_amdgcn_raw_buffer_load_b32(rc, off, 0, 2);
        __builtin_amdgcn_sched_barrier(0);
        for (int i = 0; i < 4; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rh, (lds_u8)(lds + wave * 4096 + i * 1024), 16, i * 1024 + lane * 16, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(4)" : "+v"(v));
        bad += v != off / 4;
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    }
    if (bad) atomicAdd(missing, bad);
}

// four cold DMA of 8 gathered rows each, four hot register loads of one address each behind them.  WAIT 4: the DMA must have
// landed; 8: nothing is waited for, a check that the program sees a DMA in flight (what it reads is its own stale LDS).
template <int WAIT>
__global__ __launch_bounds__(512) void dma_first(const uint32_t* cold, const uint32_t* hot, uint32_t* missing, int iters) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[8 * 4096];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const auto rc = rsrc(cold, COLD_BYTES), rh = rsrc(hot, HOT_BYTES);
    uint32_t bad = 0, sink = 0;
    for (int it = 0; it < iters; ++it) {
        uint32_t off[4], r[4];
        for (int i = 0; i < 4; ++i) {
            off[i] = cold_block((((uint64_t)blockIdx.x * 8 + wave) * iters + it) * 32 + i * 8 + (lane >> 3)) + (lane & 7) * 16u;
            *reinterpret_cast<u32x4*>(lds + wave * 4096 + i * 1024 + lane * 16) = u32x4{STALE, STALE, STALE, STALE};
        }
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        for (int i = 0; i < 4; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rc, (lds_u8)(lds + wave * 4096 + i * 1024), 16, off[i], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_raw_buffer_load_b32(rh, 0, i * 1024, 0);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(WAIT) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        for (int i = 0; i < 4; ++i) {
            uint32_t first, last;       // (by hand: the compiler would wait for the DMA in front of a read of its own)
            asm volatile("ds_read_b32 %0, %2\n ds_read_b32 %1, %2 offset:12\n s_waitcnt lgkmcnt(0)"
                         : "=&v"(first), "=&v"(last)
                         : "v"((uint32_t)(uintptr_t)(lds_u8)lds + wave * 4096u + i * 1024u + lane * 16u)
                         : "memory");
            bad += first != off[i] / 4 || last != off[i] / 4 + 3;
        }
        __builtin_amdgcn_sched_barrier(0);          // (a use of the hot loads further up would be waited for there)
        for (int i = 0; i < 4; ++i) sink += r[i];
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    }
    if (bad) atomicAdd(missing, bad);
    if (sink == 1) atomicAdd(missing + 1, 1);       // (keeps the hot loads)
}

__global__ void fill(uint32_t* p, uint32_t n, uint32_t first) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = first + i;
}

int main() {
    uint32_t *cold, *hot, *missing;
    CHECK(hipMalloc(&cold, COLD_BYTES));
    CHECK(hipMalloc(&hot, HOT_BYTES));
    CHECK(hipMalloc(&missing, 8));
    fill<<<4, 256>>>(hot, HOT_BYTES / 4, 0xabcd0000u);
    const char* what[] = {"register load, then 4 DMA, vmcnt(4)", "4 DMA, then 4 register loads, vmcnt(4)", "4 DMA, then 4 register loads, vmcnt(8)"};
    for (int form = 0; form < 3; ++form)
        for (int groups : {1, 256, 1024}) {
            const int iters = groups == 1 ? 2048 : 256;
            uint32_t n[2] = {0, 0};
            fill<<<4096, 256>>>(cold, COLD_BYTES / 4, 0);
            CHECK(hipMemcpy(missing, n, 8, hipMemcpyHostToDevice));
            if (form == 0) register_load_first<<<groups, 512>>>(cold, hot, missing, iters);
            else if (form == 1) dma_first<4><<<groups, 512>>>(cold, hot, missing, iters);
            else dma_first<8><<<groups, 512>>>(cold, hot, missing, iters);
            CHECK(hipGetLastError());
            CHECK(hipDeviceSynchronize());
            CHECK(hipMemcpy(n, missing, 8, hipMemcpyDeviceToHost));
            printf("%s, %d workgroups of 8 waves: %u of %lld lane results not there\n", what[form], groups, n[0],
                   512ll * groups * iters * (form ? 4 : 1));
            fflush(stdout);
        }
    CHECK(hipFree(cold));
    CHECK(hipFree(hot));
    CHECK(hipFree(missing));
    return 0;
}
