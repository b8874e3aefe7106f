// Exchanges between the lanes of a wave: sums of several values with few moves,
// and the order of LDS accesses.
#pragma once

#include <hip/hip_runtime.h>

namespace nkx {

// LDS accesses of one wave stay in order across it: needed between the writes of
// some lanes and the reads of others, which the compiler takes for unrelated
// where the addresses of one lane differ.  Costs no instruction (a wave's LDS
// accesses are carried out in order).
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sum of each of 16 values over the 16 lanes of a row; lane l of the row
// returns the total of value bitrev4(l).  Fifteen exchanges: each halves the
// values held.
__device__ __forceinline__ double row_sum16(double (&v)[16], int l16) {
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int half = 8 >> b;
    const bool up = (l16 >> b) & 1;
#pragma unroll
    for (int i = 0; i < half; ++i) {
      const double lo = v[i], hi = v[i + half];
      v[i] = (up ? hi : lo) + __shfl_xor(up ? lo : hi, 1 << b);
    }
  }
  return v[0];
}

__device__ __forceinline__ int bitrev4(int l) {
  return ((l & 1) << 3) | ((l & 2) << 1) | ((l & 4) >> 1) | ((l & 8) >> 3);
}

// DPP move of a double (both halves) from the lane that CTRL selects inside the
// same row of 16 lanes; every lane must be active.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xF, 0xF, false);
  const unsigned hi =
      (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Value of lane l (uniform) of a wave, in scalar registers.
__device__ __forceinline__ int lane_int(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ double lane_double(double v, int l) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Sum over the 64 lanes of a wave; every lane must be active, and every lane
// receives the same value.  Inside each row of 16 lanes by DPP moves (quad
// permutations for lane ^ 1 and lane ^ 2, then the half-row and row mirrors):
// each step adds the same two partial sums in every lane (a + b and b + a are
// the same double), so all lanes of a row hold the same row sum.  The four row
// sums are read out of lanes 0, 16, 32 and 48 and added in a fixed order.
// No LDS instruction is involved (lane shuffles through ds_bpermute would
// put twelve dependent LDS round trips in every sum).
__device__ __forceinline__ double wave_sum(double v) {
  v += dpp_move<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_move<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_move<0x141>(v);  // row_half_mirror: lane 7 - i of each 8
  v += dpp_move<0x140>(v);  // row_mirror: lane 15 - i of each 16
  return (lane_double(v, 0) + lane_double(v, 16)) + (lane_double(v, 32) + lane_double(v, 48));
}

}  // namespace nkx
