// Global-memory store helpers shared by the kernels.
//
// Outputs that are far larger than the caches are written with non-temporal
// stores: a streaming kernel that reads 128 B and writes 256 B per pixel runs
// 25-30 % faster on MI355X when its output lines do not linger in L2 / Infinity
// Cache waiting to be evicted.  Small outputs keep the default policy so that the
// next layer finds them in cache.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
// the same and a dword at any address
typedef v4i v4i_u __attribute__((aligned(1)));
typedef v2i v2i_u __attribute__((aligned(1)));
typedef int i32_u __attribute__((aligned(1)));

// Outputs at least this large are streamed past the caches.
#define PULPNN_NT_BYTES (32ll << 20)

// The policy is a template parameter on purpose: with a run-time flag
// ("if (nt) non-temporal store; else store;") the optimiser merges the two stores into
// one and drops the non-temporal hint.  Callers keep one copy of their store code per
// policy and branch between the copies.
template <bool NT>
__device__ __forceinline__ void store16(void *p, v4i v)
{
  if constexpr (NT) __builtin_nontemporal_store(v, (v4i *)p);
  else *(v4i *)p = v;
}
template <bool NT>
__device__ __forceinline__ void store8(void *p, v2i v)
{
  if constexpr (NT) __builtin_nontemporal_store(v, (v2i *)p);
  else *(v2i *)p = v;
}
template <bool NT>
__device__ __forceinline__ void store4(void *p, int v)
{
  if constexpr (NT) __builtin_nontemporal_store(v, (int *)p);
  else *(int *)p = v;
}

// bytes [0, n) of a dword, n clamped to [0, 4]
__device__ __forceinline__ unsigned low_bytes(int n)
{
  const int m = min(n, 4);
  return m <= 0 ? 0u : __builtin_amdgcn_alignbit(0u, 0xffffffffu, 32 - 8 * m);  // (4 bytes: a shift by 0)
}
// bits [0, n) of a dword, n clamped to [0, 32], and all but them: three instructions each
__device__ __forceinline__ unsigned low_bits(int n) { return (unsigned)((0xffffffffull << min(max(n, 0), 32)) >> 32); }
__device__ __forceinline__ unsigned high_bits(int n) { return (unsigned)(0xffffffffull << min(max(n, 0), 32)); }
