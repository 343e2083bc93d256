// End of a reducing lattice pass: the last workgroup to finish sums the partial rows and runs the background update
// that would otherwise be a launch of its own (k_update), in the same order and with the same bits.
//
// The update's launch cost every step 6-8 us (the gap between dependent kernels, its start, its serial chain). Here a
// workgroup writes its row through the coherence point (agent scope), waits for its own stores and counts itself in;
// the one that completes the count reads all rows through the coherence point.  Nothing is written back or
// invalidated: device-scope fences, which flush the L2s' dirty lines, cost about 100 us a pass.  Measured, a leapfrog
// step by passes with the update's launch / with this: 32^3 FP64 10.9 / 9.1 us, 64^3 FP64 12.9 / 11.7, 128^3 FP32-bulk
// 30.8 / 29.7 (velocity Verlet 32.9 / 30.2), 200^3 FP64 118.9 / 118.2; without any update 4.8, 6.4, 24, 111.
// The full-row and plane-chunk passes have it. In the charged-scalar + U(1) pass it gained nothing (100^3 9.0 / 9.1 ms
// the 100 steps) and in the one-site passes its registers (114 where 60 do) would halve the wavefronts in flight.
#pragma once

#include "update_device.hpp"

namespace clmi {

template <int NT>
__device__ __forceinline__ void finish_pass(const PassTail &t)
{
  if (!t.on) return;
  constexpr int VT = 512;  // the update kernel's threads, whose order of summation this keeps
  __shared__ double wsum[VT / 64][kNumRed];
  __shared__ double tot[kNumRed];
  __shared__ DevState S;
  __shared__ int last;
  static_assert(NT >= 128, "the second wave copies the state");
  constexpr int nS = sizeof(DevState) / 8;
  static_assert(sizeof(DevState) % 8 == 0 && nS <= 64, "one wave copies the state");
  const int tid = threadIdx.x;
  if (tid < 64) {
    __builtin_amdgcn_s_waitcnt(0);  // this wave stored the workgroup's rows
    if (tid == 0)
      last = __hip_atomic_fetch_add(t.count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == gridDim.x;
  }
  __syncthreads();
  if (!last) return;
  if (tid >= 64 && tid < 64 + nS) ((uint64_t *)&S)[tid - 64] = ((const uint64_t *)t.st)[tid - 64];
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const int rows = t.rows;
  const auto P = __builtin_amdgcn_make_buffer_rsrc((void *)t.partials, 0, rows * (int)(kNumRed * sizeof(double)), 0x00020000);
  // virtual thread vt adds rows vt, vt + VT, ... in that order; thread tid stands for vt = tid + j NT and has U rows in
  // flight (rows beyond the last read zeros, which are not added)
  constexpr int VPT = NT < VT ? VT / NT : 1, U = VPT > 2 ? VPT : 2;
  static_assert(VT % NT == 0 || NT % VT == 0, "whole virtual threads");
  static_assert(U % VPT == 0, "a batch of rows goes round the virtual threads");
  if (tid < VT) {
    double v[VPT][kNumRed];
#pragma unroll
    for (int j = 0; j < VPT; ++j)
#pragma unroll
      for (int k = 0; k < kNumRed; ++k) v[j][k] = 0.0;
    constexpr int ST = NT < VT ? NT : VT;
    for (int r0 = tid; r0 < rows; r0 += U * ST) {
      u4 q[U][kNumRed / 2];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int k = 0; k < kNumRed / 2; ++k)
          q[u][k] = __builtin_amdgcn_raw_buffer_load_b128(P, (r0 + u * ST) * (int)(kNumRed * sizeof(double)) + 16 * k, 0, 16);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (r0 + u * ST < rows)
#pragma unroll
          for (int k = 0; k < kNumRed / 2; ++k) {
            const uint64_t lo = q[u][k].x | (uint64_t)q[u][k].y << 32, hi = q[u][k].z | (uint64_t)q[u][k].w << 32;
            v[u % VPT][2 * k] += __builtin_bit_cast(double, lo);
            v[u % VPT][2 * k + 1] += __builtin_bit_cast(double, hi);
          }
    }
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
#pragma unroll
      for (int k = 0; k < kNumRed; ++k) v[j][k] = wave_sum(v[j][k]);
      if ((tid & 63) == 0)
#pragma unroll
        for (int k = 0; k < kNumRed; ++k) wsum[(tid + j * NT) >> 6][k] = v[j][k];
    }
  }
  __syncthreads();
  if (tid < kNumRed) {
    double s = 0.0;
    for (int w = 0; w < VT / 64; ++w) s += wsum[w][tid];
    tot[tid] = s * t.mc.invV;
    S.red[tid] = s * t.mc.invV;
  }
  __syncthreads();
  if (tid == 0) {
    apply_update<true>(&S, tot, t.mc, t.ops);
    __hip_atomic_store(t.count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (tid < nS) ((uint64_t *)t.st)[tid] = ((const uint64_t *)&S)[tid];
}

}  // namespace clmi
