// Device helpers shared by the fused cell kernels (apply_kernel.hpp) and the
// chain kernels (apply_chain.hpp).
#pragma once

#include "common.hpp"

namespace femtc
{

// A geometry piece: two elements, 16 bytes for FP64 and 8 for FP32.  A
// cell's G block (6 Q^3 elements, always a multiple of two) is 16-byte
// aligned for FP64 and 8-byte aligned for FP32.
template <typename T>
using Piece = T __attribute__((ext_vector_type(2)));

__device__ inline void atomic_add(double* p, double v)
{
  unsafeAtomicAdd(p, v);
}
__device__ inline void atomic_add(float* p, float v) { unsafeAtomicAdd(p, v); }

// Atomic add into LDS (ds_add_f64 / ds_add_f32): lanes of one instruction
// that hit the same address all count.
template <typename T>
__device__ inline void lds_add(T* p, T v)
{
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <typename T>
__device__ inline T stream_load(const T* p)
{
  return __builtin_nontemporal_load(p);
}

// e[k] = v[k] + v[K-1-k], o[k] = v[k] - v[K-1-k], e[K/2] = v[K/2] (odd K)
template <int K, typename T>
__device__ inline void eo_split(const T (&v)[K], T (&e)[(K + 1) / 2],
                                T (&o)[K / 2])
{
#pragma unroll
  for (int k = 0; k < K / 2; ++k)
  {
    e[k] = v[k] + v[K - 1 - k];
    o[k] = v[k] - v[K - 1 - k];
  }
  if constexpr (K % 2)
    e[K / 2] = v[K / 2];
}

// out[m] = ev[m] + od[m], out[M-1-m] = ev[m] - od[m], out[M/2] = ev[M/2]
template <int M, typename T>
__device__ inline void eo_join(const T (&ev)[(M + 1) / 2], const T (&od)[M / 2],
                               T (&out)[M])
{
#pragma unroll
  for (int m = 0; m < M / 2; ++m)
  {
    out[m] = ev[m] + od[m];
    out[M - 1 - m] = ev[m] - od[m];
  }
  if constexpr (M % 2)
    out[M / 2] = ev[M / 2];
}

// The geometry block is staged through LDS in two halves of qa-planes:
// planes [0, QA1) and [QA1, Q).
template <int Q>
constexpr int geometry_split()
{
  return (Q + 1) / 2;
}

// Synchronisation between the contraction stages.  A one-wave workgroup (or
// a multi-wave one whose cells span waves) uses the workgroup barrier; in
// the blocked scatter every wave owns whole cells and its own LDS work area,
// so a stage only has to order the wave's own LDS accesses: LDS operations of
// one wave execute in issue order, and the fences plus wave barrier keep the
// compiler from moving accesses across the stage boundary.
template <bool WAVE_LOCAL>
__device__ inline void stage_sync()
{
  if constexpr (WAVE_LOCAL)
  {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  else
    __syncthreads();
}

// LDS-only workgroup barrier: orders the LDS accesses of the workgroup
// without waiting for its outstanding global stores and atomics.
__device__ __forceinline__ void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

} // namespace femtc
