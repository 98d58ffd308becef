// esp_wave.h - exchanges and fixed-order sums inside a 64-lane wave by DPP and
// lane reads, shared by the kernels of both engines.
#pragma once

#include <hip/hip_runtime.h>

// v of the lane that the DPP control CTRL names (zero past the row's ends), and v of
// lane l of the wave
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v)
{
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffll), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ __forceinline__ double lane_value(double v, int l)
{
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// Sum over the wave in a fixed order, the same value in every lane: pairs within
// the rows of 16 lanes by DPP (a few cycles a step where a shuffle through LDS
// takes a hundred), then the four rows.  Every lane of the wave must be active.
__device__ __forceinline__ double wave_sum(double v)
{
  v = v + dpp_move<0xB1>(v);   // lanes 1,0,3,2 of every four
  v = v + dpp_move<0x4E>(v);   // lanes 2,3,0,1
  v = v + dpp_move<0x141>(v);  // mirrored within 8 lanes
  v = v + dpp_move<0x140>(v);  // mirrored within 16 lanes
  return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

// The value lane `q` of this lane's group of four holds
template <int G>
__device__ __forceinline__ double group_value(double v, int q)
{
  static_assert(G == 4, "a quad");
  return q == 0   ? dpp_move<0x00>(v)
         : q == 1 ? dpp_move<0x55>(v)
         : q == 2 ? dpp_move<0xAA>(v)
                  : dpp_move<0xFF>(v);
}

// acc[c] += the value v[c] of lane 0, 1, ... G - 1 of this lane's group (4 or 16
// lanes), one after the other
template <int G, int NS, int K = 0>
__device__ __forceinline__ void add_in_order(double (&acc)[NS], const double (&v)[NS])
{
  static_assert(G == 4 || G == 16, "a quad or a row");
  if constexpr (K < G) {
#pragma unroll
    for (int c = 0; c < NS; c++)
      acc[c] = acc[c] + dpp_move<G == 4 ? 0x55 * K : 0x150 + K>(v[c]);
    add_in_order<G, NS, K + 1>(acc, v);
  }
}

// In the first quad of a row (one quad: NQ = 1): acc[c] += v[c] of the same lane of
// quad 0, 1, ... NQ - 1, one after the other; the other quads' sums mean nothing
template <int NQ, int NS, int K = 0>
__device__ __forceinline__ void add_quads(double (&acc)[NS], const double (&v)[NS])
{
  if constexpr (K < NQ) {
#pragma unroll
    for (int c = 0; c < NS; c++) {
      if constexpr (K == 0) acc[c] = acc[c] + v[c];
      else acc[c] = acc[c] + dpp_move<0x100 + 4 * K>(v[c]);  // the lane 4 K above
    }
    add_quads<NQ, NS, K + 1>(acc, v);
  }
}
