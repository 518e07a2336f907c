// int4 weights as f16 MFMA fragments: what the several-token decode kernels
// (i4mm.hip, i4xs.hpp) share. (The prefill GEMM's conversion multiplies by the
// scale as well and stays its own.)
#pragma once
#include <hip/hip_runtime.h>

namespace st {
namespace i4 {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// v_and_or_b32 with both constants in registers (a VOP3 takes no literal).
__device__ __forceinline__ unsigned and_or(unsigned a, unsigned m, unsigned c) {
    unsigned r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(m), "v"(c));
    return r;
}

// GPTQ word (nibbles n0..n7 = k0..k7) -> (n0 - z, n4 - z), (n1 - z, n5 - z),
// (n2 - z, n6 - z), (n3 - z, n7 - z) in f16, exactly: 1024 + n - (1024 + z),
// or (1024 + 16 n) / 16 - (64 + z) for the odd nibbles.
__device__ __forceinline__ half8 word_to_b(unsigned w, half2_t zlo, half2_t zhi) {
    const unsigned m_lo = 0x000F000Fu, m_hi = 0x00F000F0u, bias = 0x64006400u;
    const half2_t sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
    const unsigned w8 = w >> 8;
    const half2_t h0 = __builtin_bit_cast(half2_t, and_or(w, m_lo, bias)) - zlo;
    const half2_t h1 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, and_or(w, m_hi, bias)), sixteenth, zhi);
    const half2_t h2 = __builtin_bit_cast(half2_t, and_or(w8, m_lo, bias)) - zlo;
    const half2_t h3 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, and_or(w8, m_hi, bias)), sixteenth, zhi);
    const u32x4 r = {__builtin_bit_cast(unsigned, h0), __builtin_bit_cast(unsigned, h1), __builtin_bit_cast(unsigned, h2),
                     __builtin_bit_cast(unsigned, h3)};
    return __builtin_bit_cast(half8, r);
}

// 8 halves (k0..k7, as 4 dwords) -> the order of word_to_b: k0,k4,k1,k5,k2,k6,k3,k7.
__device__ __forceinline__ u32x4 to_b_order(u32x4 a) {
    u32x4 r;
    r.x = __builtin_amdgcn_perm(a.z, a.x, 0x05040100u);
    r.y = __builtin_amdgcn_perm(a.z, a.x, 0x07060302u);
    r.z = __builtin_amdgcn_perm(a.w, a.y, 0x05040100u);
    r.w = __builtin_amdgcn_perm(a.w, a.y, 0x07060302u);
    return r;
}

__device__ __forceinline__ float silu_f(float v) { return __fdividef(v, 1.0f + __expf(-v)); }

// (not __syncthreads(), whose fence would wait for the loads in flight)
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace i4
}  // namespace st
