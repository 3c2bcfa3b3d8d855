// What the resident decode kernels (decode_persistent.hip, decode_ahead.hip) share: accesses that say which memory they mean, the tagged
// elements that carry values between workgroups, and the argmax's order.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_utils.h"

namespace fh {

// ---- plain global accesses -------------------------------------------------------------------------------
// Pointers that reach the kernel through descriptors in memory have lost their address space; a load through
// them would be a FLAT instruction, whose completion the compiler can only order with a full wait.  These
// say "global" explicitly.
typedef uint32_t res_u32x4 __attribute__((ext_vector_type(4)));
template <typename T>
__device__ __forceinline__ T ldg(const T* p) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (sizeof(T) == 16) {
        const res_u32x4 v = *(const __attribute__((address_space(1))) res_u32x4*)(uintptr_t)p;
        T r;
        __builtin_memcpy(&r, &v, 16);
        return r;
    } else {
        static_assert(sizeof(T) <= 8, "ldg: scalar or 16-byte types only");
        return *(const __attribute__((address_space(1))) T*)(uintptr_t)p;
    }
#else
    return *p;
#endif
}
template <typename T>
__device__ __forceinline__ void stg(T* p, T v) {
#if defined(__HIP_DEVICE_COMPILE__)
    *(__attribute__((address_space(1))) T*)(uintptr_t)p = v;
#else
    *p = v;
#endif
}

// ---- coherent (agent-scope, L2-bypassing) accesses ----------------------------------------------------
__device__ __forceinline__ uint64_t ldc64(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void stc64(uint64_t* p, uint32_t tag, uint32_t payload) {
    __hip_atomic_store(p, ((uint64_t)tag << 32) | payload, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int dot16(int4 w, int4 a, int acc) {
    acc = __builtin_amdgcn_sdot4(w.x, a.x, acc, false);
    acc = __builtin_amdgcn_sdot4(w.y, a.y, acc, false);
    acc = __builtin_amdgcn_sdot4(w.z, a.z, acc, false);
    acc = __builtin_amdgcn_sdot4(w.w, a.w, acc, false);
    return acc;
}

struct ArgPair { float v; uint32_t i; };
__device__ __forceinline__ ArgPair arg_better(ArgPair a, ArgPair b) {
    const bool take_b = (b.v > a.v) || (b.v == a.v && b.i > a.i);
    return take_b ? b : a;
}

}  // namespace fh
