// Morton order of points and functions: the code of a place in a box, on the host
// and on the device alike, and the box of a point set.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

namespace nkx {

// 21 bits with two zero bits between each
__host__ __device__ inline uint64_t spread21(uint64_t v) {
  v &= 0x1fffff;
  v = (v | v << 32) & 0x1f00000000ffffull;
  v = (v | v << 16) & 0x1f0000ff0000ffull;
  v = (v | v << 8) & 0x100f00f00f00f00full;
  v = (v | v << 4) & 0x10c30c30c30c30c3ull;
  v = (v | v << 2) & 0x1249249249249249ull;
  return v;
}

// 63-bit code of p's place in the box lo .. hi, 21 bits per axis; x in the lowest
// bit of each triple, or (XHIGH) in the highest.  Products and sums rounded one by
// one, so that it does not depend on where it is formed.
template <bool XHIGH>
__host__ __device__ inline uint64_t morton_code(const double *p, const double *lo,
                                                const double *hi) {
#pragma clang fp contract(off)
  uint64_t code = 0;
  for (int d = 0; d < 3; ++d) {
    const double ext = fmax(hi[d] - lo[d], 1e-12);
    const double t = fmin(fmax((p[d] - lo[d]) / ext, 0.0), 1.0);
    code |= spread21((uint64_t)(t * 2097151.0)) << (XHIGH ? 2 - d : d);
  }
  return code;
}

#ifdef __HIPCC__
constexpr int kBoxThreads = 256;

// Minimum and maximum of six values per thread over the workgroup (lo xyz, hi
// xyz); thread k < 6 returns value k.
__device__ __forceinline__ double box_reduce(double v[6], double (*s)[kBoxThreads]) {
  for (int k = 0; k < 6; ++k) s[k][threadIdx.x] = v[k];
  __syncthreads();
  for (int h = kBoxThreads / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h)
      for (int k = 0; k < 6; ++k) {
        const double o = s[k][threadIdx.x + h];
        s[k][threadIdx.x] = k < 3 ? fmin(s[k][threadIdx.x], o) : fmax(s[k][threadIdx.x], o);
      }
    __syncthreads();
  }
  return threadIdx.x < 6 ? s[threadIdx.x][0] : 0.0;
}

// box of the points, per workgroup
static __global__ void __launch_bounds__(kBoxThreads) points_box(int64_t n,
                                                                 const double *__restrict__ pts,
                                                                 double *__restrict__ part) {
  __shared__ double s[6][kBoxThreads];
  double v[6] = {HUGE_VAL, HUGE_VAL, HUGE_VAL, -HUGE_VAL, -HUGE_VAL, -HUGE_VAL};
  for (int64_t i = (int64_t)blockIdx.x * kBoxThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBoxThreads)
    for (int d = 0; d < 3; ++d) {
      const double x = pts[3 * i + d];
      v[d] = fmin(v[d], x);
      v[3 + d] = fmax(v[3 + d], x);
    }
  const double r = box_reduce(v, s);
  if (threadIdx.x < 6) part[6 * blockIdx.x + threadIdx.x] = r;
}

// nparts partial boxes into one, by one workgroup
[[maybe_unused]] static __global__ void __launch_bounds__(kBoxThreads) points_box_final(
    int nparts, const double *__restrict__ part, double *__restrict__ bb) {
  __shared__ double s[6][kBoxThreads];
  double v[6] = {HUGE_VAL, HUGE_VAL, HUGE_VAL, -HUGE_VAL, -HUGE_VAL, -HUGE_VAL};
  for (int i = threadIdx.x; i < nparts; i += kBoxThreads)
    for (int k = 0; k < 6; ++k)
      v[k] = k < 3 ? fmin(v[k], part[6 * i + k]) : fmax(v[k], part[6 * i + k]);
  const double r = box_reduce(v, s);
  if (threadIdx.x < 6) bb[threadIdx.x] = r;
}

// Codes (and indices) of the points in the box of nparts partial ones, which every
// workgroup reduces again: at most kBoxParts of them (one launch less than with
// points_box_final, which 6.3 M points are better served by: 43 us for 1024 parts
// and 34 for the codes, 207 and 116 with 64 parts).
constexpr int kBoxParts = 64;
template <bool XHIGH>
__global__ void __launch_bounds__(kBoxThreads) points_keys(int64_t n, int nparts,
                                                           const double *__restrict__ pts,
                                                           const double *__restrict__ part,
                                                           uint64_t *__restrict__ key,
                                                           int *__restrict__ idx) {
  __shared__ double bb[6];
  if (threadIdx.x < 6) {
    double r = part[threadIdx.x];
    for (int i = 1; i < nparts; ++i)
      r = threadIdx.x < 3 ? fmin(r, part[6 * i + threadIdx.x]) : fmax(r, part[6 * i + threadIdx.x]);
    bb[threadIdx.x] = r;
  }
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * kBoxThreads + threadIdx.x;
  if (i >= n) return;
  key[i] = morton_code<XHIGH>(pts + 3 * i, bb, bb + 3);
  idx[i] = (int)i;
}
#endif  // __HIPCC__

}  // namespace nkx
