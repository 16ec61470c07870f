// eimp_device.h -- wave-level helpers shared by the device code.
#pragma once

#include <type_traits>

#include "eimp_internal.h"

namespace eimp {

// ---------------------------------------------------------------------------
// wave helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

// Pointers read out of device structs are generic, so accesses through them
// compile to FLAT instructions, which count in the LDS counter as well: the
// next s_waitcnt for an LDS result then also waits for a FLAT store to be
// acknowledged by memory.  Inside loops that mix LDS traffic with global
// stores the pointers are cast to the global address space first.
template <class T>
using gptr_t = __attribute__((address_space(1))) T *;
template <class T>
__device__ __forceinline__ gptr_t<T> gmem(T *p) {
    return (gptr_t<T>)p;
}
// Arrays that no kernel running at the same time writes, read at wave-uniform
// addresses through the constant address space: scalar loads.
template <class T>
using cptr_t = const __attribute__((address_space(4))) T *;
template <class T>
__device__ __forceinline__ cptr_t<T> cmem(const T *p) {
    return (cptr_t<T>)p;
}
// LDS (address space 3) pointers: 32-bit byte addresses
template <class T>
using lds_ptr_t = __attribute__((address_space(3))) T *;
// compile-time loop: f(std::integral_constant<int, I>) for I in [B, E)
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// clang vector types: assignable through global-address-space pointers
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t mbcnt(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

__device__ __forceinline__ uint64_t lanemask_lt() {
    uint32_t l = lane_id();
    return l == 0 ? 0ull : (~0ull >> (64 - l));
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
__device__ __forceinline__ uint64_t wave_sum64(uint64_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor(v, o));
    return v;
}
// inclusive scan over the wave
__device__ __forceinline__ uint32_t wave_scan_incl(uint32_t v) {
    uint32_t l = lane_id();
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t u = __shfl_up(v, o);
        if (l >= (uint32_t)o) v += u;
    }
    return v;
}

// v_writelane_b32 through the LLVM intrinsic (no clang builtin in this
// toolchain); the compiler sees it, so it inserts the wait states a VALU-written
// SGPR operand needs.
extern "C" __device__ uint32_t eimp_llvm_writelane(uint32_t val, uint32_t lane, uint32_t old)
    __asm("llvm.amdgcn.writelane");

// writes a wave-uniform value into lane L of a VGPR
template <int L>
__device__ __forceinline__ uint32_t writelane(uint32_t old, uint32_t val) {
    return eimp_llvm_writelane(val, (uint32_t)L, old);
}


// Exclusive prefix sum of v over lanes 0..N-1 (other lanes: garbage), by DPP
// row shifts and row broadcasts (no LDS).
template <int N>
__device__ __forceinline__ uint32_t lane_scan_excl(uint32_t v) {
    uint32_t x = v;
    // within rows of 16 lanes: lane i += lane i-1, i-2, i-4, i-8 (zero past the row start)
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xF, 0xF, true);
    if constexpr (N > 2) x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xF, 0xF, true);
    if constexpr (N > 4) x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xF, 0xF, true);
    if constexpr (N > 8) x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xF, 0xF, true);
    // across rows: lane 15 of each row into rows 1 and 3, then lane 31 into rows 2 and 3
    if constexpr (N > 16) x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xA, 0xF, false);
    if constexpr (N > 32) x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xC, 0xF, false);
    return x - v;
}

}  // namespace eimp
