// Internal helpers shared by the gfx950 kernels of libminf_hip.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "../../include/minf_hip.h"

#define MINF_WAVE 64

static inline int minf_hip_status(hipError_t e) {
    return e == hipSuccess ? MINF_OK : MINF_ERR_HIP_BASE - (int)e;
}

// Status of the launch that was just enqueued on `stream` (does not synchronise).
static inline int minf_launch_status() { return minf_hip_status(hipGetLastError()); }

__device__ __forceinline__ int minf_lane() { return (int)(threadIdx.x & 63); }

__device__ __forceinline__ uint64_t minf_lanemask_lt() {
    return (1ull << minf_lane()) - 1ull;
}

// Value of `x` in lane `src` (src must be wave-uniform).
__device__ __forceinline__ int minf_readlane(int x, int src) {
    return __builtin_amdgcn_readlane(x, __builtin_amdgcn_readfirstlane(src));
}

// 16 bytes per lane from its own global address into LDS at a wave-uniform base (lane i -> base +
// 16 i).  Written as assembly because the compiler counts the builtin's instruction as a "flat" access,
// which may touch the LDS counter out of order: one of them on any path through a loop turns every wait
// for a fragment read into a wait for ALL outstanding reads (lgkmcnt(0): in the attention walk the first PV
// MFMA waited for the whole V tile, every second k-step for the reads issued just before it).  The copies
// are counted by vmcnt alone, and the callers wait for vmcnt(0) before each barrier.  Attention: 16001-token
// vertical-slash layer 1.68 -> 1.66 ms, dense 16384 tokens on all-zero operands 1.52 -> 1.50; nothing beyond noise
// at 131072 tokens: a SIMD's other wave filled most of those waits, and the chip holds a lower clock on live
// data whatever the schedule.
__device__ __forceinline__ void copy16_to_lds(const char *src, char *dst) {
    const int lds = (int)(unsigned)(unsigned long long)(__attribute__((address_space(3))) char *)dst;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds), "v"(src) : "memory", "m0");
}

// n / d for n < 2^31 by a multiplication and a shift (round-up method: m = ceil(2^(31+bits) / d) fits 32 bits, its
// excess times n stays below 2^(31+bits) / d).  A 32-bit division takes some forty dependent instructions here, and
// every workgroup of the attention kernels made five of them before it could ask for its first byte: 1.2 -> 0.7 us;
// A-shape, 16 heads of 64, 49152 tokens, window 128 125.3 -> 122.4 us, of 128 218.7 -> 216.9; nothing beyond noise
// on walks of 50 steps.
struct FastDiv {
    unsigned d, m, shift;
};
inline FastDiv fast_div(unsigned d) {
    unsigned bits = 0;
    while ((1ull << bits) < d) ++bits;
    if (bits == 0) return FastDiv{1u, 0x80000000u, 31u};
    return FastDiv{d, (unsigned)(((1ull << (31 + bits)) + d - 1) / d), 31u + bits};
}
__device__ __forceinline__ unsigned fast_quot(unsigned n, const FastDiv &f) { return (unsigned)(((unsigned long long)n * f.m) >> f.shift); }
