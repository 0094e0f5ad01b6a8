// Loads that go straight into LDS, their waits, and loops unrolled by the compiler: what the products that stage their tiles in LDS share.
#pragma once
#include "common.h"

#include <type_traits>
#include <utility>

// All but the n youngest of the wave's loads have arrived (a wave's loads retire in order).
#define LI_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | 0x0F70)
#define LI_LOAD_TO_LDS(gptr, lptr)                                                                        \
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(gptr),              \
                                     (__attribute__((address_space(3))) void*)(lptr), 16, 0, 0)

// f(std::integral_constant<int, 0>) ... f(std::integral_constant<int, N - 1>)
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// The same load with its address as (scalar base) + (32-bit offset of the lane): no address
// arithmetic in vector registers.  M0 carries the LDS address, as in the compiler's own form.
#define LI_LOAD_TO_LDS_AT(base, voff, lptr)                                                              \
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"                          \
                 :: "s"((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)(lptr)), "v"(voff), "s"(base) : "memory", "m0")

// The same with a 64-bit address a lane: rows that are gathered from a tensor of any size.
#define LI_LOAD_TO_LDS_FROM(vptr, lptr)                                                                  \
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"                         \
                 :: "s"((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)(lptr)), "v"(vptr) : "memory", "m0")
