// What the resident decode kernels (decode_persistent.hip, decode_ahead.hip) share: accesses that say which memory they mean, the tagged
// elements that carry values between workgroups, and the argmax's order.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

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

// A workgroup that takes part in hand-overs.
struct PollCtx {
    uint32_t tid, lane, wave, wg, G, spin_limit;
    uint32_t* sh_abort;      // LDS
    uint32_t* abort_flag;    // global
};

// N elements a thread takes, re-read together until all carry their tags; bounded.  Every load of a round trip is issued before any is looked at, and
// without a condition: a branch around one of them would put a wait behind it.  (A thread without an element of its own takes one that another has.)
// LATER: an element of a later phase will do; nothing is handed out.
template <int N, bool LATER = false, typename Addr, typename Tag>
__device__ __forceinline__ void poll_tagged(Addr addr, Tag tag, uint32_t* out, const PollCtx& cx) {
    uint64_t w[N];
    uint32_t spins = 0;
    for (;;) {
#pragma unroll
        for (int i = 0; i < N; i++) w[i] = ldc64(addr(i));
        uint32_t off = 0;
#pragma unroll
        for (int i = 0; i < N; i++) off |= LATER ? ((uint32_t)(w[i] >> 32) - tag(i)) >> 31 : (uint32_t)(w[i] >> 32) ^ tag(i);
        if (!off) break;
        ++spins;
        if (spins > cx.spin_limit ||
            ((spins & 1023u) == 0 && __hip_atomic_load(cx.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
            *cx.sh_abort = 1;
            __hip_atomic_store(cx.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    if constexpr (LATER) return;
#pragma unroll
    for (int i = 0; i < N; i++) out[i] = (uint32_t)w[i];
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

// One workgroup's part of an argmax: the LAST index among equal maxima (project.rs:501-503).
template <uint32_t WAVES>
__device__ __forceinline__ ArgPair best_of_workgroup(ArgPair v, ArgPair* sh, const PollCtx& cx) {
    auto fold = [&](auto O) { v = arg_better(v, ArgPair{lane_xor<O.value>(v.v), lane_xor<O.value>(v.i)}); };
    fold(std::integral_constant<int, 32>{}); fold(std::integral_constant<int, 16>{}); fold(std::integral_constant<int, 8>{});
    fold(std::integral_constant<int, 4>{}); fold(std::integral_constant<int, 2>{}); fold(std::integral_constant<int, 1>{});
    __syncthreads();
    if (cx.lane == 0) sh[cx.wave] = v;
    __syncthreads();
    ArgPair r = sh[0];
    for (uint32_t w = 1; w < WAVES; w++) r = arg_better(r, sh[w]);
    return r;
}

}  // namespace fh
