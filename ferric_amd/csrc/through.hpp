// Stores to pinned host memory that a host thread polls (transfer.hip, dequant.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fhip {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// a store that goes through to memory: behind s_waitcnt vmcnt(0) it has arrived
template <class U>
__device__ __forceinline__ void store_through(U* p, U v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }
template <>
__device__ __forceinline__ void store_through(u32x4* p, u32x4 v) { asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" : : "v"(p), "v"(v) : "memory"); }

}  // namespace fhip
