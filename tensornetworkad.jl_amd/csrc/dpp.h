// Sums across the lanes of a wavefront by DPP lane moves (no LDS), for doubles.
#pragma once
#include <hip/hip_runtime.h>

namespace tnad {
namespace {

// DPP lane move of a double (its two 32-bit halves); lanes outside row_mask keep x.  With every row enabled
// no old value is needed, so the move writes a fresh register (no copy of x ahead of it).
template <int CTRL, int ROWMASK = 0xF>
__device__ __forceinline__ double dpp_d(double x) {
  const long long b = __double_as_longlong(x);
  int lo, hi;
  if constexpr (ROWMASK == 0xF) {
    lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, false);
    hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, false);
  } else {
    lo = __builtin_amdgcn_update_dpp((int)b, (int)b, CTRL, ROWMASK, 0xF, false);
    hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), CTRL, ROWMASK, 0xF, false);
  }
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// sums over each row of 16 lanes of N values at once, stage by stage (the lane moves of different
// values interleave); butterflies, so every lane of a row ends with the same bits
template <int N>
__device__ __forceinline__ void row16_sums(double (&x)[N]) {
#pragma unroll
  for (int a = 0; a < N; ++a) x[a] += dpp_d<0xB1>(x[a]);    // quad_perm (1, 0, 3, 2)
#pragma unroll
  for (int a = 0; a < N; ++a) x[a] += dpp_d<0x4E>(x[a]);    // quad_perm (2, 3, 0, 1)
#pragma unroll
  for (int a = 0; a < N; ++a) x[a] += dpp_d<0x141>(x[a]);   // row_half_mirror
#pragma unroll
  for (int a = 0; a < N; ++a) x[a] += dpp_d<0x140>(x[a]);   // row_mirror
}

// totals of N values over the wavefront, in every lane (the N butterflies interleave)
template <int N>
__device__ __forceinline__ void wave_sums(double (&x)[N]) {
  row16_sums<N>(x);
#pragma unroll
  for (int k = 0; k < N; ++k) x[k] += dpp_d<0x142, 0xA>(x[k]);
#pragma unroll
  for (int k = 0; k < N; ++k) x[k] += dpp_d<0x143, 0x8>(x[k]);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const long long b = __double_as_longlong(x[k]);
    const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
    x[k] = __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
  }
}

// sum over the wavefront, the same value in every lane
__device__ __forceinline__ double wave_sum(double x) {
  double v[1] = {x};
  row16_sums<1>(v);
  x = v[0];
  x += dpp_d<0x142, 0xA>(x);   // row_bcast15: row 1 += row 0, row 3 += row 2
  x += dpp_d<0x143, 0x8>(x);   // row_bcast31: row 3 += lane 31; lane 63 holds the total
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

}  // namespace
}  // namespace tnad
