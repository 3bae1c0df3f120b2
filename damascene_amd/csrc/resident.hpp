// resident.hpp -- launches whose blocks all stay on the device and hand each
// other values while they run (the plain Lanczos steps and the block filter).
#pragma once
#include <hip/hip_runtime.h>

#include "resident_gate.hpp"

namespace dmsc {

namespace resident {

// Values that other blocks of the running grid write or read: accesses at
// device scope, which go past the per-XCD caches.
template <typename T>
__device__ __forceinline__ T shared_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void shared_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// base[off / sizeof(T)] by a byte offset below 4 GiB: a scalar base and one
// register of address.
template <typename T>
__device__ __forceinline__ T* at_byte(T* base, unsigned off) {
  return (T*)((char*)base + off);
}
template <typename T>
__device__ __forceinline__ const T* at_byte(const T* base, unsigned off) {
  return (const T*)((const char*)base + off);
}

// A copy the compiler knows nothing about: what is computed from it stays in
// the loop that computes it instead of holding registers across it.
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Every memory access this wave issued has completed.
__device__ __forceinline__ void drain_memory() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Up to N values at byte offsets at[u] of base, each awaited until its block
// has written it (kEmpty before that): at most `polls` rounds of reads; then,
// or once another block gave up, *stalled is set and false returned.  live:
// bit u set where v[u] is wanted.
template <int N, typename T>
__device__ __forceinline__ bool await(const T* base, const unsigned (&at)[N], unsigned live, T kEmpty, int* stalled,
                                      int polls, T (&v)[N]) {
  for (int i = 0;; i++) {
    bool all = true;
#pragma unroll
    for (int u = 0; u < N; u++)
      if (live >> u & 1) v[u] = shared_load(at_byte(base, at[u]));
#pragma unroll
    for (int u = 0; u < N; u++)
      if ((live >> u & 1) && v[u] == kEmpty) all = false;
    if (all) return true;
    if (i >= polls || ((i & 63) == 63 && shared_load(stalled))) {
      shared_store(stalled, 1);
      return false;
    }
    __builtin_amdgcn_s_sleep(1);
  }
}

}  // namespace resident
}  // namespace dmsc
