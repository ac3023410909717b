// Device code shared by the batched prompt phase's kernels (q4_gemm.hip,
// prefill.hip).

#pragma once

#include "cw_internal.hpp"

namespace cwi {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kT = 256;

__device__ __forceinline__ float2 add(float2 a, float2 b) {
    return make_float2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ float4 add(float4 a, float4 b) {
    return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

// The sum in order of the S >= 1 partials at(0), at(1), ...: four requested
// at a time, so that no load waits for another's sum.
template <typename At>
__device__ __forceinline__ auto sum_parts(int S, At at) {
    auto v = at(0);
    int s = 1;
    for (; s + 4 <= S; s += 4) {
        const auto a = at(s), b = at(s + 1), c = at(s + 2), d = at(s + 3);
        v = add(add(add(add(v, a), b), c), d);
    }
    if (s + 3 == S) {
        const auto a = at(s), b = at(s + 1), c = at(s + 2);
        return add(add(add(v, a), b), c);
    }
    if (s + 2 == S) {
        const auto a = at(s), b = at(s + 1);
        return add(add(v, a), b);
    }
    return s < S ? add(v, at(s)) : v;
}

typedef __attribute__((address_space(3))) unsigned char lds_u8;

// 64-lane global -> LDS DMAs of 16 bytes per lane: lane i's bytes land at
// lds_dst + 16 i; lds_dst is wave-uniform (M0, set by the compiler through the
// operand constraint), the source a uniform base plus a lane offset, or an
// address per lane.  Written as asm so the compiler's wait-count pass does not track
// them and adds no wait before the LDS reads of another buffer; the kernel
// orders them itself with counted vmcnt waits and a barrier.
__device__ __forceinline__ uint32_t lds_off(unsigned char *p) {
    return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_u8 *)p);
}
__device__ __forceinline__ void dma16(const void *base, uint32_t off, unsigned char *lds_dst) {
    asm volatile("global_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(off), "s"(base), "{m0}"(lds_off(lds_dst))
                 : "memory");
}

}  // namespace cwi
