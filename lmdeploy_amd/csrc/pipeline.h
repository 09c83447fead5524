// The pieces that the kernels' hand-made software pipelines share: loads from inline assembly that are waited for by count,
// LDS addresses and fragment reads, and the packing of partial sums.
#pragma once

#include "w4a16_common.h"

#include <type_traits>

namespace w4a16 {

// Compile-time loop: f(std::integral_constant<int, 0>{}), ..., f(<N-1>); gives inline assembly
// its immediate operands.
template<int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// Loads of the software pipeline.  They are issued from inline assembly, in place ("+v"), with
// a scalar base and a per-thread 32-bit offset, and waited for by count: the compiler would
// drain every load in flight at the loop header, exposing the memory latency once per K step.
template<int OFF>
__device__ __forceinline__ void gload128(u32x4_t& dst, uint32_t voff, const void* sbase)
{
    asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "+v"(dst) : "v"(voff), "s"(sbase), "n"(OFF));
}
template<int OFF>
__device__ __forceinline__ void gload32(uint32_t& dst, uint32_t voff, const void* sbase)
{
    asm volatile("global_load_dword %0, %1, %2 offset:%3" : "+v"(dst) : "v"(voff), "s"(sbase), "n"(OFF));
}
// wait until at most N of this wave's loads are in flight; tied to `v` so that no use of it can
// be scheduled above the wait
template<int N, typename V>
__device__ __forceinline__ void wait_vm(V& v)
{
    asm volatile("s_waitcnt vmcnt(%1)" : "+v"(v) : "n"(N));
}

// The byte address of something in LDS, as the direct-to-LDS loads take it: lane l's 16 bytes land at the address in M0 plus
// 16 l.  They are written in assembly (rather than through the builtin) so that the memory address is a scalar base plus a
// 32-bit lane offset instead of a 64-bit lane address, which costs a register pair and an add per request.  They count
// in vmcnt like any other load and are complete there when the data is in LDS.
__device__ __forceinline__ uint32_t lds_addr(const void* p)
{
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)(p);
}
// LDS fragment read from inline assembly (byte address + immediate).  Left to the compiler, each activation fragment was
// read right before the MFMAs that use it, which then waited a full LDS latency; and any compiler-visible LDS read after a
// direct-to-LDS load would be preceded by a wait for ALL loads in flight.
template<int OFF>
__device__ __forceinline__ void lds_read128(half8_t& dst, uint32_t addr)
{
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}

__device__ __forceinline__ uint64_t pack2(float a, float b)
{
    return (uint64_t)__builtin_bit_cast(uint32_t, a) | ((uint64_t)__builtin_bit_cast(uint32_t, b) << 32);
}
__device__ __forceinline__ float lo_float(uint64_t v) { return __builtin_bit_cast(float, (uint32_t)v); }
__device__ __forceinline__ float hi_float(uint64_t v) { return __builtin_bit_cast(float, (uint32_t)(v >> 32)); }

}  // namespace w4a16
