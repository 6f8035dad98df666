// Device-side building blocks shared by every kernel of the solver path.
//
// Conventions:
//  * one workgroup owns one clade row of S state columns; row loads and stores
//    are coalesced (thread t: columns t, t + NT, t + 2*NT, ...);
//  * the species tree is held as int32 tables over preorder positions
//    (kb_rowops.hpp) with -1 meaning "no node".
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define KB_NEG_INF (-__builtin_inff())

namespace kb {

__device__ __forceinline__ float fsafe(float m) { return m == KB_NEG_INF ? 0.0f : m; }

// 2^x by the hardware instruction: the same as exp2f for x >= -126 and 0 below
// (where exp2f returns a denormal).  For terms whose size next to the others
// of their sum or product makes such values negligible.
__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }

// log2 x by the hardware instruction: the same as log2f for x >= 2^-126 and
// for 0; for the sums of max-shifted terms, which are 0 or at least 1.
__device__ __forceinline__ float log2_hw(float x) { return __builtin_amdgcn_logf(x); }

// 1/x by the hardware reciprocal (1 ulp) instead of a correctly rounded division.
__device__ __forceinline__ float rcp_hw(float x) { return __builtin_amdgcn_rcpf(x); }

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

template <typename T>
__device__ __forceinline__ T wave_max(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    T u = __shfl_xor(v, o, 64);
    v = u > v ? u : v;
  }
  return v;
}

// Block-wide reductions. `red` is LDS scratch of at least NT/64 elements.
// Every thread returns the full result. Two barriers (reuse-safe).
template <int NT, typename T>
__device__ __forceinline__ T block_sum(T v, T* red) {
  constexpr int NW = NT / 64;
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) red[w] = v;
  __syncthreads();
  T r = red[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) r += red[i];
  __syncthreads();
  return r;
}

template <int NT, typename T>
__device__ __forceinline__ T block_max(T v, T* red) {
  constexpr int NW = NT / 64;
  v = wave_max(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) red[w] = v;
  __syncthreads();
  T r = red[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) r = red[i] > r ? red[i] : r;
  __syncthreads();
  return r;
}

// Online merge of a (max, scaled-sum) pair into an accumulator.
__device__ __forceinline__ void lse_merge(float& m, float& acc, float m2, float s2) {
  float nm = fmaxf(m, m2);
  float nms = fsafe(nm);
  float a = (m == KB_NEG_INF) ? 0.0f : acc * exp2_hw(m - nms);
  float b = (m2 == KB_NEG_INF) ? 0.0f : s2 * exp2_hw(m2 - nms);
  acc = a + b;
  m = nm;
}

}  // namespace kb
