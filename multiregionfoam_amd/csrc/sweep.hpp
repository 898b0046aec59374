// Device helpers shared by the DILU sweep kernels (dilu.hip, dilu_box.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "dilu.hpp"

namespace mrfg {

template <typename T>
struct Bits;
template <>
struct Bits<double> {
    using U = unsigned long long;
    static constexpr U kSent = kHaloSentinel64;
    __device__ static U to(double v) { return (U)__double_as_longlong(v); }
    __device__ static double from(U u) { return __longlong_as_double((long long)u); }
};
template <>
struct Bits<float> {
    using U = unsigned int;
    static constexpr U kSent = kHaloSentinel32;
    __device__ static U to(float v) { return (U)__float_as_uint(v); }
    __device__ static float from(U u) { return __uint_as_float(u); }
};

template <typename U>
__device__ inline U haloLoad(const U *h, int slot)
{
    return __hip_atomic_load(&h[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline double elem(const double2 &v, int i) { return i == 0 ? v.x : v.y; }
__device__ inline float elem(const float4 &v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }
__device__ inline int elem(const int4 &v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// Value type of a record chunk for sweep mode MODE over values T.
template <typename T, int MODE>
struct RecordOf {
    using V = typename Pack<T>::V;
    static constexpr int N = Pack<T>::N;
};
template <typename T>
struct RecordOf<T, kDiluFactor> {
    using V = double2;
    static constexpr int N = 2;
};

// Raw buffer access (gfx9 buffer resource: base, byte size, 32-bit
// offsets).  Every address of the sweeps' fast paths is a wave-uniform
// resource plus a scalar step offset plus a per-lane constant, so a step
// spends no instructions on 64-bit address arithmetic.  A lane offset of kNoLane lies
// beyond every resource: the hardware drops such a store, which replaces the
// per-step exec-mask juggling of conditional stores.
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
constexpr int kRawBufferWord3 = 0x00020000;   // 32-bit data format, no swizzle, no index stride
constexpr int kSysCoherent = 16;              // sc1: the policy of the agent-scope relaxed atomics
constexpr unsigned kNoLane = 0x80000000u;

// (the arguments are wave-uniform; readfirstlane states it, so the resource
// lives in scalar registers)
__device__ inline __amdgpu_buffer_rsrc_t rawBuffer(const void *base, size_t bytes)
{
    const unsigned long long a = (unsigned long long)base;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
    int n = __builtin_amdgcn_readfirstlane((int)bytes);
    int w3 = kRawBufferWord3;
    // every resource keeps its own size and flag registers: two resources
    // sharing one would be reassembled before each use
    asm volatile("" : "+s"(n), "+s"(w3));
    return __builtin_amdgcn_make_buffer_rsrc((void *)(((unsigned long long)hi << 32) | lo), (short)0, n, w3);
}

template <typename X, int aux>
__device__ inline X bufLoad(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff)
{
    if constexpr (sizeof(X) == 16) return __builtin_bit_cast(X, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, aux));
    else if constexpr (sizeof(X) == 8) return __builtin_bit_cast(X, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, aux));
    else return __builtin_bit_cast(X, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, aux));
}

template <typename X, int aux>
__device__ inline void bufStore(X v, __amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff)
{
    if constexpr (sizeof(X) == 8) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, voff, soff, aux);
    else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, voff, soff, aux);
}

}  // namespace mrfg
