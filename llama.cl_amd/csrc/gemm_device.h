// Device helpers shared by the prefill product kernels: vector types, the constants of the convert-free fold and
// asynchronous global -> LDS copies.
#pragma once
#include "common.h"

namespace llmops {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kFoldBiasBits = 0x4B400000;  // the float 1.5 * 2^23 ...
constexpr float kFoldBias = 12582912.0f;   // ... whose low mantissa bits count in units of 1

__device__ __forceinline__ uint32_t lo4(uint32_t w) { return w & 0x0F0F0F0Fu; }
__device__ __forceinline__ uint32_t hi4(uint32_t w) { return (w >> 4) & 0x0F0F0F0Fu; }

__device__ __forceinline__ uint32_t lds_off(const void* p) {
    return (uint32_t)(uintptr_t)((const __attribute__((address_space(3))) void*)p);
}
// a value / pointer that is the same for the whole wave, in scalar registers
__device__ __forceinline__ uint32_t uniform_u32(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ const void* uniform_ptr(const void* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return reinterpret_cast<const void*>(((uint64_t)hi << 32) | lo);
}
// lane i's 16 (4) bytes at base + off (base the same for the whole wave, off a byte offset per lane)
// land at lds_base + 16*i (4*i); counts in vmcnt like any load.  (uniform_u32 belongs to the callers whose lds_base the
// compiler does not see to be uniform)
__device__ __forceinline__ void copy16_to_lds(const void* base, uint32_t off, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(lds_base) : "memory", "m0");
}
__device__ __forceinline__ void copy4_to_lds(const void* base, uint32_t off, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" : : "v"(off), "s"(base), "s"(lds_base) : "memory", "m0");
}
// the same with byte offsets of 64 bits
__device__ __forceinline__ void copy16_to_lds(const void* base, uint64_t off, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(reinterpret_cast<uint64_t>(base) + off), "s"(lds_base) : "memory", "m0");
}
__device__ __forceinline__ void copy4_to_lds(const void* base, uint64_t off, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(reinterpret_cast<uint64_t>(base) + off), "s"(lds_base) : "memory", "m0");
}

}  // namespace llmops
