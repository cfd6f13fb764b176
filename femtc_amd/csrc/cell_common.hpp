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

template <typename T>
__device__ inline T stream_load(const T* p)
{
  return __builtin_nontemporal_load(p);
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
