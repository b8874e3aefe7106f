// int8 slice form shared by the mixed-precision kernels (V_xc build and
// nuclear gradient): tile layout, slicing, the ten-product tile contraction
// on v_mfma_i32_16x16x64_i8 and the direct global -> LDS section copy.
//
// integer MFMA accumulation.
//
// Every operand tile of the two contractions (P blocks, collocation values,
// Z) is stored as four int8 slices with one power-of-two scale per tile row
// (an Ozaki-type splitting; Ozaki, Ogita & Oishi, Numer. Algorithms 2012):
//   x = 2^(e-6) (a0 + 2^-7 a1 + 2^-14 a2 + 2^-21 a3),   |a_s| <= 64,
// e = the exponent of the row's largest |x| (|x| < 2^e), each slice rounded
// to nearest from the exact FP64 remainder, so |x - sum| <= 2^(e-28) with
// random sign.  A tile product is
//   sum_k x_ik y_kj = 2^(eA_i + eB_j - 12) sum_d 2^(-7d) sum_(s+t=d) sum_k a_s,ik b_t,kj
// and every inner sum runs on v_mfma_i32_16x16x64_i8 in exact int32
// arithmetic (|sum| <= 4 * 64^3 < 2^31).  The ten slice products with
// s + t <= 3 are kept; the dropped ones are below 2^-28 of the row-times-
// column scale, of random sign.  The int32 sums are combined and scaled in
// FP64 per exponent group of KG 64-function blocks (density: the P row and Pm
// point exponents are shared over the group, the sums run across its steps)
// and per 64-point batch (V).  The functional, rho, grad rho, E_xc, N_el and the V
// accumulation are FP64; collocation gradients are FP32 (rounded once from
// FP64).  Exact accumulation is the point of the integer form:
// v_mfma_f32_*_bf16 rounds its FP32 sums relative to the largest term with a
// mean pulled toward zero, a bias that shows up in N_el on large grids.
//
// Tile layout: a 64 x 64 tile T[row][k] is four row fragments of 16 rows;
// lane l of fragment rt holds T[16 rt + l % 16][16 (l / 16) + e], e = 0..15,
// as 16 consecutive bytes -- the A-operand order of v_mfma_i32_16x16x64_i8,
// and, read as B[k][j] with j the row of T, its B-operand order.  A section
// is the four slice planes (4 KB each) followed by the 64 row exponents.
//
// Per live slot (bytes):   F   Phi, rows = functions, k = points   16.25 KB
//                          Pm  Phi, rows = points, k = functions   16.25 KB
//                          Z   Z,   rows = functions, k = points   16.25 KB
//                          G   dPhi/dx, dy, dz, FP32 [f][p]         48 KB (GGA)
// P is gathered into one section per 64 x 64 block pair (rows mu, k = nu).
#pragma once
#include "nkx_internal.hpp"

namespace nkx {

typedef int v4i __attribute__((ext_vector_type(4)));

// v_mfma_i32_16x16x64_i8 lane layout (checked by tests/gpu_probe): lane l
// supplies A[l%16][16(l/16) .. +15] and B[16(l/16) .. +15][l%16]; result
// register r of lane l holds D[4(l/16) + r][l%16].

namespace {
constexpr int FB = 64;
constexpr int PT = 64;
constexpr int TILE = FB * PT;
constexpr int PLANE = TILE;                  // bytes per slice plane
constexpr int SEC = 4 * PLANE + 256;         // section: 4 planes + exponents (padded)
constexpr int OFF_F = 0, OFF_PM = SEC, OFF_Z = 2 * SEC, OFF_G = 3 * SEC;
constexpr int MAXNFB = 1024;
// function blocks per exponent group: the P sections of blocks (fm, fk) with
// the same fk / KG share row exponents, and a batch's Pm sections of blocks
// with the same local index / KG share point exponents
constexpr int KG = 4;

__host__ __device__ inline int64_t slot_bytes_i8(int gga) {
  return 3 * (int64_t)SEC + (gga ? 3 * (int64_t)TILE * 4 : 0);
}

// byte offset of T[row][k] inside one plane
__device__ __forceinline__ int frag8(int row, int k) {
  return (((row >> 4) * 64) + (row & 15) + 16 * (k >> 4)) * 16 + (k & 15);
}

// exponent e with max < 2^e; rows whose largest |x| is below 2^-120 are
// stored as zero
__device__ __forceinline__ int row_exp(double m) {
  if (!(m >= 0x1p-120)) return -127;
  int e;
  (void)frexp(m, &e);
  return e;
}

// 2^e as a double, e in the normal range
__device__ __forceinline__ double pow2(int e) {
  return __longlong_as_double((long long)(e + 1023) << 52);
}
// 2^e, or 0 for the zero-row exponent marker -127
__device__ __forceinline__ double pow2_or_zero(int e) { return e == -127 ? 0.0 : pow2(e); }

// Byte 0 of a .. d as one word
__device__ __forceinline__ int bytes4(unsigned a, unsigned b, unsigned c, unsigned d) {
  return (int)(__builtin_amdgcn_perm(b, a, 0x0c0c0400u) |
               __builtin_amdgcn_perm(d, c, 0x04000c0cu));
}

// Slices of 16 elements |x| < 2^e, none NaN (e = -127: all zero): four roundings
// half to even, each of the exact remainder of the one before.  A rounding is one
// FMA onto 1.5 2^52, whose low byte is the slice: thirteen instructions an element
// with the packing, where ldexp, rint, conversions and byte stores took 24.
__device__ __forceinline__ void slice16(const double (&x)[16], int e, v4i (&out)[4]) {
  const double sc = e == -127 ? 0.0 : pow2(6 - e);
  constexpr double M = 0x1.8p52;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    unsigned d[4][4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      double t = fma(x[4 * w + k], sc, M);
      double r = fma(x[4 * w + k], sc, M - t);  // exact, |r| <= 1/2
      d[0][k] = (unsigned)__double2loint(t);
#pragma unroll
      for (int p = 1; p < 4; ++p) {
        t = fma(r, 128.0, M);
        if (p < 3) r = fma(r, 128.0, M - t);
        d[p][k] = (unsigned)__double2loint(t);
      }
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) out[p][w] = bytes4(d[p][0], d[p][1], d[p][2], d[p][3]);
  }
}

// The four planes of 16 integers |V| <= 2^27 as balanced base-128 digits: V =
// a0 2^21 + a1 2^14 + a2 2^7 + a3, a1 .. a3 in [-64, 63].  With V + kDigitBias
// given (element e in byte e of a plane) the lower digits are seven-bit fields
// a + 64; b - 64 for the four fields of a word at once is (b | 80) - 40, top bits
// flipped.
constexpr int kDigitBias = 64 * (1 + (1 << 7) + (1 << 14));
__device__ __forceinline__ void pack16(const unsigned (&U)[16], v4i (&out)[4]) {
#pragma unroll
  for (int w = 0; w < 4; ++w)
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int sh = 21 - 7 * p;
      const unsigned b = (unsigned)bytes4(U[4 * w] >> sh, U[4 * w + 1] >> sh, U[4 * w + 2] >> sh,
                                          U[4 * w + 3] >> sh);
      out[p][w] = p == 0 ? (int)b : (int)(((b | 0x80808080u) - 0x40404040u) ^ 0x80808080u);
    }
}

// High words of the largest |x| of 16; elements that are not finite are set to
// zero first
__device__ __forceinline__ unsigned max_hi(double (&x)[16]) {
  auto top = [&]() {
    unsigned m = 0;
#pragma unroll
    for (int e = 0; e < 16; ++e) m = max(m, (unsigned)__double2hiint(x[e]) & 0x7fffffffu);
    return m;
  };
  unsigned m = top();
  if (m >= 0x7ff00000u) {
#pragma unroll
    for (int e = 0; e < 16; ++e)
      if (!isfinite(x[e])) x[e] = 0.0;
    m = top();
  }
  return m;
}

// Element e of 16 packed ones: its integer V, and all of them times `scale`
// (2^(exponent - 27), or zero for a row stored as zero): exact.
__device__ __forceinline__ int unslice_int(const v4i (&w)[4], int e) {
  const int sh = 24 - 8 * (e & 3);
  auto d = [&](int p) { return (int)((unsigned)w[p][e >> 2] << sh) >> 24; };
  return (d(0) << 21) + (d(1) << 14) + (d(2) << 7) + d(3);
}
__device__ __forceinline__ double unslice_scale(int e) { return e == -127 ? 0.0 : pow2(e - 27); }

__device__ __forceinline__ v4i ld16(const signed char *p) {
  return *reinterpret_cast<const v4i *>(p);
}

// The ten slice products of one 16 x 16 x 64 tile product, combined into the
// FP64 value scaled by 2^(e - 19), e = eA + eB: hi = 128 d0 + d1,
// lo = 128 d2 + d3, value = hi + 2^-14 lo.
__device__ __forceinline__ void tile_product(const v4i *A, const v4i *B, int hi[4], int lo[4]) {
  const v4i z = {0, 0, 0, 0};
  v4i d0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[0], B[0], z, 0, 0, 0);
  v4i d1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[0], B[1], z, 0, 0, 0);
  d1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[1], B[0], d1, 0, 0, 0);
  v4i d2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[0], B[2], z, 0, 0, 0);
  d2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[1], B[1], d2, 0, 0, 0);
  d2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[2], B[0], d2, 0, 0, 0);
  v4i d3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[0], B[3], z, 0, 0, 0);
  d3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[1], B[2], d3, 0, 0, 0);
  d3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[2], B[1], d3, 0, 0, 0);
  d3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[3], B[0], d3, 0, 0, 0);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    hi[r] = d0[r] * 128 + d1[r];
    lo[r] = d2[r] * 128 + d3[r];
  }
}

// The same ten slice products added to running sums hi, lo of earlier tile
// products with the same row and column exponents: the d1 and d3 chains start
// from hi and lo, so hi = 128 d0 + d1 and lo = 128 d2 + d3 stay exact int32
// sums.  Over n products |hi| <= n (128 + 2) 2^18 and |lo| <= n (3 * 128 + 4)
// 2^18, both below 2^31 for n <= 16.
__device__ __forceinline__ void tile_product_acc(const v4i *A, const v4i *B, v4i &hi, v4i &lo) {
  const v4i z = {0, 0, 0, 0};
  const v4i d0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[0], B[0], z, 0, 0, 0);
  v4i d1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[0], B[1], hi, 0, 0, 0);
  d1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[1], B[0], d1, 0, 0, 0);
  v4i d2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[0], B[2], z, 0, 0, 0);
  d2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[1], B[1], d2, 0, 0, 0);
  d2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[2], B[0], d2, 0, 0, 0);
  v4i d3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[0], B[3], lo, 0, 0, 0);
  d3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[1], B[2], d3, 0, 0, 0);
  d3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[2], B[1], d3, 0, 0, 0);
  d3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[3], B[0], d3, 0, 0, 0);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    hi[r] = d0[r] * 128 + d1[r];
    lo[r] = d2[r] * 128 + d3[r];
  }
}

// Z = a phi + bx dphi/dx + by dphi/dy + bz dphi/dz, in one fixed order of
// roundings (every kernel that forms Z uses this)
__device__ __forceinline__ double z_value(double ph, double gx, double gy, double gz, double a,
                                          double bx, double by, double bz) {
  return fma(bz, gz, fma(by, gy, fma(bx, gx, a * ph)));
}

// Item t of a 64 x 64 FP64 tile held in LDS (v[row][k], row stride 65; TR: the
// tile read transposed, v[k][row]): row 16 (t / 64) + t % 16, k 16 ((t % 64) /
// 16) .. +15.  Conflict-free in both orders.
template <bool TR>
__device__ __forceinline__ void tile_item(const double (*v)[65], double (&x)[16]) {
  const int l = threadIdx.x & 63;
  const int row = 16 * (threadIdx.x >> 6) + (l & 15), k0 = 16 * (l >> 4);
#pragma unroll
  for (int e = 0; e < 16; ++e) x[e] = TR ? v[k0 + e][row] : v[row][k0 + e];
}

// Item t sliced with its row's exponent ex into a section at dst (fragment
// order), 256 threads.
__device__ __forceinline__ void store_item(const double (&x)[16], int ex, signed char *dst) {
  const int t = threadIdx.x, l = t & 63;
  v4i out[4];
  slice16(x, ex, out);
#pragma unroll
  for (int p = 0; p < 4; ++p) *reinterpret_cast<v4i *>(dst + p * PLANE + t * 16) = out[p];
  if (l < 16) dst[4 * PLANE + 16 * (t >> 6) + l] = (signed char)ex;
}

// row_exp of the four items of a row (lanes l, l ^ 16, l ^ 32, l ^ 48); elements
// that are not finite are set to zero.  The high word of the largest magnitude
// holds its exponent.
__device__ __forceinline__ int item_row_exp(double (&x)[16]) {
  unsigned m = max_hi(x);
  m = max(m, (unsigned)__shfl_xor((int)m, 16));
  m = max(m, (unsigned)__shfl_xor((int)m, 32));
  const int e = (int)(m >> 20) - 1022;
  return e < -119 ? -127 : e;
}

// Direct global -> LDS copy of one section (4 planes + the 256-byte exponent
// area) by the NW waves of a workgroup, this one taking pieces w0, w0 + NW,
// ...: 16 pieces of 1 KB (global_load_lds_dwordx4: lane l writes its 16 bytes
// at dst + 16 l) and one of 256 bytes (dword form).  The fixed trip count
// keeps the copies straight-line code, so the compiler's waits after them
// stay exact.  The copies are tracked by vmcnt only; the consumer waits with
// wait_vm0() before the barrier that publishes the LDS.
template <int NW>
__device__ __forceinline__ void dma_section(const signed char *src, signed char *dst_lds, int w0,
                                            int lane) {
#pragma unroll
  for (int k = 0; k < (17 + NW - 1) / NW; ++k) {
    const int pc = w0 + k * NW;
    if (pc < 16)
      __builtin_amdgcn_global_load_lds(src + pc * 1024 + lane * 16, dst_lds + pc * 1024, 16, 0,
                                       0);
    else if (pc == 16)
      __builtin_amdgcn_global_load_lds(src + 16384 + lane * 4, dst_lds + 16384, 4, 0, 0);
  }
}
// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima)
__device__ __forceinline__ void wait_vm0() { __builtin_amdgcn_s_waitcnt(0x0F70); }

}  // namespace
}  // namespace nkx
