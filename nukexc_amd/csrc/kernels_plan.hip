// Launch plan of the batched build on the device: Morton order of a molecule's
// points into padded 64-point batches, the batches' boxes, and the screening of
// (function block, batch) pairs.  Every comparison and rounding is that of a
// plain host loop (products and sums rounded one by one), so the plan does not
// depend on where it is built.
// Bound by launches and the radix sort's passes up to about 100 k points
// (0.19 ms for the whole plan of 121 k points, 6.6 ms in host loops).
#include <hipcub/hipcub.hpp>

#include "morton.hpp"
#include "nkx_internal.hpp"
#include "vxc_kernels.hpp"

namespace nkx {

namespace {

constexpr int NT = kBoxThreads;
constexpr int PT = 64;
constexpr int FB = 64;

// One wave per batch: its 64 points in sorted order (past the end: copies of
// the last one, weight 0, index -1) and their box.
__global__ void __launch_bounds__(NT) plan_gather(int64_t n, int64_t nb,
                                                  const int *__restrict__ perm,
                                                  const double *__restrict__ pts,
                                                  const double *__restrict__ w,
                                                  double *__restrict__ px, double *__restrict__ py,
                                                  double *__restrict__ pz, double *__restrict__ pw,
                                                  int *__restrict__ pidx,
                                                  double *__restrict__ boxes) {
  const int64_t sp = (int64_t)blockIdx.x * NT + threadIdx.x, b = sp / PT;
  if (b >= nb) return;  // whole waves
  const int64_t src = perm[sp < n ? sp : n - 1];
  double lo[3], hi[3];
  for (int d = 0; d < 3; ++d) lo[d] = hi[d] = pts[3 * src + d];
  px[sp] = lo[0];
  py[sp] = lo[1];
  pz[sp] = lo[2];
  pw[sp] = sp < n ? w[src] : 0.0;
  pidx[sp] = sp < n ? (int)src : -1;
  for (int o = 32; o > 0; o >>= 1)
    for (int d = 0; d < 3; ++d) {
      lo[d] = fmin(lo[d], __shfl_xor(lo[d], o));
      hi[d] = fmax(hi[d], __shfl_xor(hi[d], o));
    }
  if ((threadIdx.x & (PT - 1)) == 0)
    for (int d = 0; d < 3; ++d) {
      boxes[6 * b + d] = lo[d];
      boxes[6 * b + 3 + d] = hi[d];
    }
}

// Block f of functions (centre, radius; 4 doubles each, sorted order) reaches
// the box: some distance is below the radius; one lane per function.
__device__ __forceinline__ bool reaches(const double *box, const double *fn, int nbf, int f) {
#pragma clang fp contract(off)
  const int k = f * FB + (threadIdx.x & 63);
  bool hit = false;
  if (k < nbf) {
    const double *c = fn + 4 * (int64_t)k;
    double d2 = 0.0;
    for (int d = 0; d < 3; ++d) {
      double e = 0.0;
      if (c[d] < box[d]) e = box[d] - c[d];
      else if (c[d] > box[3 + d]) e = c[d] - box[3 + d];
      d2 = d2 + e * e;
    }
    hit = d2 < c[3] * c[3];
  }
  return __ballot(hit) != 0;
}

// One wave per batch: live[b * nfb + f], the number of live blocks and of
// functions in them, of pairs of blocks (2a, 2a + 1) with a live one, and whether
// the last block of an odd number is live.
__global__ void __launch_bounds__(NT) plan_screen(int64_t nb, int nbf, int nfb,
                                                  const double *__restrict__ boxes,
                                                  const double *__restrict__ fn,
                                                  unsigned char *__restrict__ live,
                                                  int2 *__restrict__ count) {
  const int64_t b = (int64_t)blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
  if (b >= nb) return;
  double box[6];
  for (int k = 0; k < 6; ++k) box[k] = boxes[6 * b + k];
  int nblk = 0, nfun = 0, ntwo = 0;
  bool even = false;  // of the even block before
  for (int f = 0; f < nfb; ++f) {
    const bool hit = reaches(box, fn, nbf, f);
    if (f & 1) ntwo += hit || even;
    else even = hit;
    if (hit) {
      ++nblk;
      nfun += min(nbf, (f + 1) * FB) - f * FB;
    }
    if ((threadIdx.x & 63) == 0) live[b * nfb + f] = hit ? 1 : 0;
  }
  if ((threadIdx.x & 63) == 0) count[b] = make_int2(plan_count(nblk, ntwo, (nfb & 1) && even), nfun);
}

// One wave per batch: its live blocks in ascending order from slot b_off[b],
// the slots' batch, the molecule's table [block][batch] -> slot or -1, and the
// block pairs that share a batch.
__global__ void __launch_bounds__(NT) plan_fill(int64_t nb, int nfb, int blk0, int64_t b0,
                                                const unsigned char *__restrict__ live,
                                                const int *__restrict__ b_off,
                                                int *__restrict__ b_fbl, int *__restrict__ slot_b,
                                                int *__restrict__ tile_slot,
                                                int *__restrict__ pairs) {
  const int64_t b = (int64_t)blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
  if (b >= nb) return;
  const int lane = threadIdx.x & 63;
  const unsigned char *lv = live + b * nfb;
  int at = b_off[b0 + b];
  for (int f0 = 0; f0 < nfb; f0 += 64) {
    const int f = f0 + lane;
    const bool on = f < nfb && lv[f];
    const unsigned long long m = __ballot(on);
    const int slot = at + __popcll(m & ((1ull << lane) - 1ull));
    if (on) {
      b_fbl[slot] = blk0 + f;
      slot_b[slot] = (int)(b0 + b);
    }
    if (f < nfb) tile_slot[(int64_t)f * nb + b] = on ? slot : -1;
    at += __popcll(m);
  }
  for (int i = 0; i < nfb; ++i) {
    if (!lv[i]) continue;
    for (int j = i + lane; j < nfb; j += 64)
      if (lv[j] && !pairs[i * nfb + j]) pairs[i * nfb + j] = 1;
  }
}

__global__ void __launch_bounds__(NT) plan_zero(int64_t n, int *__restrict__ x) {
  const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (i < n) x[i] = 0;
}

unsigned nblocks(int64_t n, int per = NT) { return (unsigned)((n + per - 1) / per); }

}  // namespace

void vk_plan_points(hipStream_t s, PlanScratch &sc, int64_t npts, const double *pts,
                    const double *w, double *px, double *py, double *pz, double *pw, int *pidx,
                    double *boxes) {
  NKX_REQUIRE(npts > 0 && npts < INT32_MAX, NKX_ERR_UNSUPPORTED,
              "a molecule's plan takes 1 .. 2^31 - 2 points");
  const int nparts = (int)std::min<int64_t>(kBoxParts, (npts + NT - 1) / NT);
  size_t bytes = 0;
  NKX_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (uint64_t *)nullptr,
                                                   (uint64_t *)nullptr, (int *)nullptr,
                                                   (int *)nullptr, (int)npts, 0, 63, s));
  sc.part.reserve((size_t)6 * kBoxParts);
  sc.key.reserve((size_t)2 * npts);
  sc.idx.reserve((size_t)2 * npts);
  sc.tmp.reserve(bytes);
  uint64_t *k0 = sc.key.p, *k1 = k0 + npts;
  int *i0 = sc.idx.p, *i1 = i0 + npts;
  hipLaunchKernelGGL(points_box, dim3(nparts), dim3(NT), 0, s, npts, pts, sc.part.p);
  hipLaunchKernelGGL(points_keys<false>, dim3(nblocks(npts)), dim3(NT), 0, s, npts, nparts, pts,
                     sc.part.p, k0, i0);
  NKX_HIP_CHECK(hipGetLastError());
  // stable: points with equal codes stay in the grid's order
  NKX_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(sc.tmp.p, bytes, k0, k1, i0, i1, (int)npts, 0,
                                                   63, s));
  const int64_t nb = (npts + PT - 1) / PT;
  hipLaunchKernelGGL(plan_gather, dim3(nblocks(nb * PT)), dim3(NT), 0, s, npts, nb, i1, pts, w,
                     px, py, pz, pw, pidx, boxes);
  NKX_HIP_CHECK(hipGetLastError());
}

void vk_plan_screen(hipStream_t s, int64_t nb, int nbf, int nfb, const double *boxes,
                    const double *fn, unsigned char *live, int *count) {
  if (nb <= 0) return;
  hipLaunchKernelGGL(plan_screen, dim3(nblocks(nb, NT / 64)), dim3(NT), 0, s, nb, nbf, nfb, boxes,
                     fn, live, reinterpret_cast<int2 *>(count));
  NKX_HIP_CHECK(hipGetLastError());
}

void vk_plan_fill(hipStream_t s, int64_t nb, int nfb, int blk0, int64_t b0,
                  const unsigned char *live, const int *b_off, int *b_fbl, int *slot_b,
                  int *tile_slot, int *pairs) {
  if (nb <= 0) return;
  const int64_t np = (int64_t)nfb * nfb;
  hipLaunchKernelGGL(plan_zero, dim3(nblocks(np)), dim3(NT), 0, s, np, pairs);
  hipLaunchKernelGGL(plan_fill, dim3(nblocks(nb, NT / 64)), dim3(NT), 0, s, nb, nfb, blk0, b0,
                     live, b_off, b_fbl, slot_b, tile_slot, pairs);
  NKX_HIP_CHECK(hipGetLastError());
}

}  // namespace nkx
