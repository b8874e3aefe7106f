// Grid partition, compaction, reference-shaped collocation, functionals.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "nkx_internal.hpp"
#include "sto_run.hpp"
#include "xc_functionals.hpp"
#include "xc_polarized.hpp"

namespace nkx {

// ---------------------------------------------------------------------------
// Becke partition (partitioning.hpp:44-55, :63-120, :126-213), one thread per
// point:
//   w_g *= P_own / sum_i P_i,  P_i = prod_(j != i) s(mu_ij),
//   mu_ij = clamp((r_i - r_j) / R~_ij, -1, 1),  s = (1 - p(p(p(mu)))) / 2,
// with R~ = min(R_ij, 5) in the capped form.  Every product runs over j in
// index order and the sum over i in index order, as the reference's loops.
//
// Capped form, exact screening: with R~ <= 5 every atom i whose distance
// exceeds the nearest atom's by >= 5 bohr has mu_(i,nearest) >= 1, so s = 0
// and P_i = 0 exactly; every j farther than r_i + 5 has mu_ij <= -1 and
// contributes the factor s(-1) = 1 exactly (p(+-1) = +-1 in FP64).  Skipping
// those factors and terms leaves every product and sum bit-identical (the
// unscreened mode, BECKE_NO_SCREEN, evaluates all of them and is compared
// with the screened one bit for bit by the tests).
//
// Work per point: distances are compared squared first, so a square root is
// taken only for atoms near enough to matter (the nearest distance is the
// root of the smallest square: the rounded root is monotonic).  Candidates i
// (at most BK_NC per pass, in index order) are held in registers; one sweep
// over j in index order multiplies every candidate's product by its factor,
// so each r_j is formed once per pass rather than once per (i, j).  The
// capped (or plain) inter-atomic distances come from a table (becke_rtab).
// ---------------------------------------------------------------------------
// The factor's polynomial and the distances are formed with rounded products
// and sums in the order written (no contraction into FMAs), the reference's
// compute_p / compute_s (partitioning.hpp:51-55) with x^3 = (x x) x: near
// mu = 1, 1 - p(p(p(mu))) keeps no digits below 2^-53, so which points end
// with exactly zero weight depends on this rounding, and fixing it makes the
// partition (and the compacted point set) reproducible bit for bit by a host
// loop with the same order.
__device__ __forceinline__ double becke_p(double x) {
#pragma clang fp contract(off)
  return (1.5 * x) - (0.5 * (x * x * x));
}

__device__ __forceinline__ double becke_s(double mu) {
#pragma clang fp contract(off)
  return 0.5 * (1.0 - becke_p(becke_p(becke_p(mu))));
}

// squared distance ((dx dx + dy dy) + dz dz), rounded at every step
__device__ __forceinline__ double bdist2(double px, double py, double pz, const double *c) {
#pragma clang fp contract(off)
  const double dx = px - c[0], dy = py - c[1], dz = pz - c[2];
  return dx * dx + dy * dy + dz * dz;
}

// R~_ij (capped) or R_ij (plain) for all pairs, row-major natoms x natoms
__global__ void __launch_bounds__(256) becke_rtab(int natoms, const double *__restrict__ C,
                                                  int capped, double *__restrict__ rt) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)natoms * natoms) return;
  const int i = (int)(e / natoms), j = (int)(e % natoms);
  double R = sqrt(bdist2(C[3 * i], C[3 * i + 1], C[3 * i + 2], C + 3 * j));
  if (capped) R = fmin(R, 5.0);
  rt[e] = R;
}

constexpr int BK_NC = 16;

__global__ void __launch_bounds__(256) becke_kernel(int natoms, const double *__restrict__ C,
                                                    const double *__restrict__ rt, int64_t npts,
                                                    const double *__restrict__ pts,
                                                    const int *__restrict__ owner,
                                                    double *__restrict__ w, int mode) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= npts) return;
  const bool capped = (mode & BECKE_CAPPED) != 0;
  const bool screen = capped && !(mode & BECKE_NO_SCREEN);
  const double px = pts[3 * g], py = pts[3 * g + 1], pz = pts[3 * g + 2];
  const int own = owner[g];
  double rmin = 0.0, lim_i2 = 0.0;
  if (screen) {
    double d2min = 1e300;
    for (int j = 0; j < natoms; ++j) d2min = fmin(d2min, bdist2(px, py, pz, C + 3 * j));
    rmin = sqrt(d2min);
    // beyond this square, r_i - r_min > 5 for sure (margin 1e-3 bohr)
    lim_i2 = (rmin + 5.001) * (rmin + 5.001);
  }
  double norm = 0.0, pown = 0.0;
  int next = 0;
  while (next < natoms) {
    double ri[BK_NC], Pi[BK_NC];
    int ii[BK_NC];
#pragma unroll
    for (int k = 0; k < BK_NC; ++k) {
      ri[k] = 0.0;
      Pi[k] = 1.0;
      ii[k] = -1;
    }
    int nc = 0;
    double rmax = 0.0;
    for (; next < natoms && nc < BK_NC; ++next) {
      const double d2 = bdist2(px, py, pz, C + 3 * next);
      if (screen && d2 > lim_i2) continue;
      const double r = sqrt(d2);
      if (screen && r - rmin >= 5.0) continue;  // P_i == 0 exactly
#pragma unroll
      for (int k = 0; k < BK_NC; ++k)
        if (k == nc) {
          ri[k] = r;
          ii[k] = next;
        }
      rmax = fmax(rmax, r);
      ++nc;
    }
    if (nc == 0) break;
    // beyond this square, r_i - r_j < -5 for every candidate i
    const double lim_j2 = (rmax + 5.001) * (rmax + 5.001);
    for (int j = 0; j < natoms; ++j) {
      const double d2 = bdist2(px, py, pz, C + 3 * j);
      if (screen && d2 > lim_j2) continue;  // every factor == 1 exactly
      const double rj = sqrt(d2);
#pragma unroll
      for (int k = 0; k < BK_NC; ++k) {
        const int i = ii[k];
        if (i < 0 || i == j) continue;
        // factor == 1 exactly, or the product already exactly zero
        if (screen && (ri[k] - rj <= -5.0 || Pi[k] == 0.0)) continue;
        double mu = (ri[k] - rj) / rt[(int64_t)i * natoms + j];
        mu = mu > 1.0 ? 1.0 : (mu < -1.0 ? -1.0 : mu);
        Pi[k] *= becke_s(mu);
      }
    }
#pragma unroll
    for (int k = 0; k < BK_NC; ++k) {
      if (ii[k] < 0) continue;
      if (ii[k] == own) pown = Pi[k];
      norm += Pi[k];
    }
  }
  w[g] *= pown / norm;
}

// Atom-centred product grid on the device, one workgroup per radial shell:
// shell q of atom sh_atom[q] at radius sh_r[q] (radial weight sh_w[q]) takes
// angular rule sh_rule[q] (points ang[4 (rule_off[k] + j) ..]) and writes
// its points from sh_poff[q]: centre + r u_j with weight w_r w_j.  Rounded
// products and sums, no contraction (the pragma: HIP's __dmul_rn is a plain
// product that may be fused into the following sum): bit-identical to a
// host loop.
__global__ void __launch_bounds__(256) grid_shells_kernel(
    const int *__restrict__ sh_atom, const double *__restrict__ sh_r,
    const double *__restrict__ sh_w, const int *__restrict__ sh_rule,
    const int64_t *__restrict__ sh_poff, const int *__restrict__ rule_off,
    const int *__restrict__ rule_n, const double *__restrict__ xyz,
    const double *__restrict__ ang, double *__restrict__ P, double *__restrict__ W,
    int *__restrict__ O) {
#pragma clang fp contract(off)
  const int q = blockIdx.x, a = sh_atom[q], k = sh_rule[q];
  const double r = sh_r[q], wr = sh_w[q];
  const double *u = ang + 4 * (int64_t)rule_off[k];
  for (int j = threadIdx.x; j < rule_n[k]; j += 256) {
    const int64_t g = sh_poff[q] + j;
    for (int d = 0; d < 3; ++d) P[3 * g + d] = xyz[3 * a + d] + r * u[4 * j + d];
    W[g] = wr * u[4 * j + 3];
    O[g] = a;
  }
}

void launch_grid_shells(hipStream_t s, int nshell, const int *sh_atom, const double *sh_r,
                        const double *sh_w, const int *sh_rule, const int64_t *sh_poff,
                        const int *rule_off, const int *rule_n, const double *xyz,
                        const double *ang, double *P, double *W, int *O) {
  if (nshell <= 0) return;
  hipLaunchKernelGGL(grid_shells_kernel, dim3((unsigned)nshell), dim3(256), 0, s, sh_atom, sh_r,
                     sh_w, sh_rule, sh_poff, rule_off, rule_n, xyz, ang, P, W, O);
  NKX_HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Workspace of the allocation-free Becke partition (nkx_becke_noalloc): the
// pair-distance table in a file-scope device array, BECKE_SCRATCH_ATOMS^2
// doubles (2 MiB), one copy per GPU held until the process ends.  Host code
// never passes the array's name to a kernel: its device address is resolved
// once per device (becke_scratch_init, from nkx_create with that device
// current) and kept per device.
static __device__ __align__(256) double scratch[BECKE_SCRATCH_ATOMS * BECKE_SCRATCH_ATOMS];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch_ptr[kMaxDevices] = {};
}  // namespace

void becke_scratch_init(int device) {
  NKX_REQUIRE(device >= 0 && device < kMaxDevices, NKX_ERR_INVALID_ARGUMENT,
              "device index beyond the scratch table");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[device]) return;
  void *p = nullptr;
  NKX_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  g_scratch_ptr[device] = static_cast<double *>(p);
}

double *becke_scratch(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return g_scratch_ptr[device];
}

void launch_becke(hipStream_t s, int natoms, const double *centers, int64_t npts,
                  const double *pts, const int *owner, double *w, int mode, double *rtab) {
  if (npts == 0) return;
  const int64_t npair = (int64_t)natoms * natoms;
  hipLaunchKernelGGL(becke_rtab, dim3((unsigned)((npair + 255) / 256)), dim3(256), 0, s, natoms,
                     centers, mode & BECKE_CAPPED, rtab);
  NKX_HIP_CHECK(hipGetLastError());
  const int64_t blocks = (npts + 255) / 256;
  hipLaunchKernelGGL(becke_kernel, dim3((unsigned)blocks), dim3(256), 0, s, natoms, centers, rtab,
                     npts, pts, owner, w, mode);
  NKX_HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Order-preserving compaction of (point, weight, owner) with w > thr.  The
// reference compacts with an atomic counter, so its surviving order is
// nondeterministic (grid.hpp:329-338); this keeps generation order.
// ---------------------------------------------------------------------------
constexpr int kCompactBlock = 1024;

__global__ void __launch_bounds__(kCompactBlock) compact_count(int64_t n, double thr,
                                                               const double *__restrict__ w,
                                                               int64_t *__restrict__ counts) {
  __shared__ int part[kCompactBlock / 64];
  const int64_t g = (int64_t)blockIdx.x * kCompactBlock + threadIdx.x;
  const bool keep = g < n && w[g] > thr;
  const unsigned long long mask = __ballot(keep);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = __popcll(mask);
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t s = 0;
    for (int i = 0; i < kCompactBlock / 64; ++i) s += part[i];
    counts[blockIdx.x] = s;
  }
}

__global__ void __launch_bounds__(kCompactBlock) compact_scatter(
    int64_t n, double thr, const double *__restrict__ pin, const double *__restrict__ win,
    const int *__restrict__ oin, const int64_t *__restrict__ offs, double *__restrict__ pout,
    double *__restrict__ wout, int *__restrict__ oout) {
  __shared__ int part[kCompactBlock / 64];
  const int64_t g = (int64_t)blockIdx.x * kCompactBlock + threadIdx.x;
  const bool keep = g < n && win[g] > thr;
  const unsigned long long mask = __ballot(keep);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0) part[wv] = __popcll(mask);
  __syncthreads();
  int before = 0;
  for (int i = 0; i < wv; ++i) before += part[i];
  const unsigned long long lower = lane ? (mask & ((1ull << lane) - 1ull)) : 0ull;
  if (keep) {
    const int64_t d = offs[blockIdx.x] + before + __popcll(lower);
    pout[3 * d] = pin[3 * g];
    pout[3 * d + 1] = pin[3 * g + 1];
    pout[3 * d + 2] = pin[3 * g + 2];
    wout[d] = win[g];
    oout[d] = oin[g];
  }
}

// Exclusive sums of the block counts in place; their total to page-locked memory.
__global__ void __launch_bounds__(kCompactBlock) compact_scan(int64_t nb,
                                                              int64_t *__restrict__ counts,
                                                              int64_t *__restrict__ total) {
  __shared__ int64_t part[kCompactBlock / 64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int64_t run = 0;
  for (int64_t i0 = 0; i0 < nb; i0 += kCompactBlock) {
    const int64_t i = i0 + threadIdx.x;
    const int64_t c = i < nb ? counts[i] : 0;
    int64_t v = c;
    for (int o = 1; o < 64; o <<= 1) {
      const int64_t u = __shfl_up(v, o);
      if (lane >= o) v += u;
    }
    if (lane == 63) part[wv] = v;
    __syncthreads();
    int64_t before = run;
    for (int k = 0; k < kCompactBlock / 64; ++k) {
      if (k < wv) before += part[k];
      run += part[k];
    }
    if (i < nb) counts[i] = before + v - c;
    __syncthreads();
  }
  if (threadIdx.x == 0) *total = run;
}

int64_t compact_points(hipStream_t s, int64_t n, double thr, const double *pin,
                       const double *win, const int *oin, double *pout, double *wout,
                       int *oout, int64_t *counts, int64_t *total) {
  if (n == 0) return 0;
  const int64_t nb = (n + kCompactBlock - 1) / kCompactBlock;
  hipLaunchKernelGGL(compact_count, dim3((unsigned)nb), dim3(kCompactBlock), 0, s, n, thr, win,
                     counts);
  NKX_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(compact_scan, dim3(1), dim3(kCompactBlock), 0, s, nb, counts, total);
  NKX_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(compact_scatter, dim3((unsigned)nb), dim3(kCompactBlock), 0, s, n, thr, pin,
                     win, oin, counts, pout, wout, oout);
  NKX_HIP_CHECK(hipGetLastError());
  NKX_HIP_CHECK(hipStreamSynchronize(s));
  return *total;
}

// ---------------------------------------------------------------------------
// Collocation in the reference layout: LayoutLeft (N_bf, N_pts), element
// (mu, g) at mu + g * N_bf (stobasis.hpp:494-584).  One workgroup per 64
// points, 4 FW functions at a time: a wave takes FW consecutive functions, a
// point per lane (sto_run.hpp), into LDS tiles of 64 points x 4 FW functions
// whose rows go out as runs of 4 FW doubles.
//
// Bound by its writes with the gradient (3.4 TB/s), by those and FP64 VALU issue
// without; by the chain of one wave's functions on small grids.  One thread per
// element, functions fastest, loads a function record per element and evaluates
// every exponential, root and quotient again: 375 us per call on benzene (120
// functions, 342 144 points); now 110 us for the values and 292 us for the three
// gradients.
template <bool VAL, bool GRAD, int FW>
__global__ void __launch_bounds__(256) colloc_ref_kernel(int nbf, const FuncRec *__restrict__ F,
                                                         const HarmTerm *__restrict__ T,
                                                         int64_t npts,
                                                         const double *__restrict__ pts,
                                                         double *phi, double *gx, double *gy,
                                                         double *gz) {
  constexpr int NARR = (VAL ? 1 : 0) + (GRAD ? 3 : 0), G0 = VAL ? 1 : 0;
  constexpr int CR_F = 4 * FW, CR_LD = CR_F + 1;
  __shared__ double t[NARR][64][CR_LD];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t g0 = (int64_t)blockIdx.x * 64;
  const int64_t g = g0 + lane < npts ? g0 + lane : npts - 1;
  const double x = pts[3 * g], y = pts[3 * g + 1], z = pts[3 * g + 2];
  double *const out[4] = {VAL ? phi : gx, VAL ? gx : gy, VAL ? gy : gz, gz};
  const int c = threadIdx.x & (CR_F - 1);
  for (int m0 = blockIdx.y * CR_F; m0 < nbf; m0 += gridDim.y * CR_F) {
    // the functions of a short last tile are dealt to all four waves
    const int q = (min(CR_F, nbf - m0) + 3) >> 2, i0 = q * wv;
    const int f0 = m0 + i0, n = min(q, nbf - f0);
    StoRun run;
#pragma unroll 1
    for (int i = 0; i < n; ++i) {
      const FuncRec *fr = F + f0 + i;
      double v, gr[3];
      run.eval<GRAD, false>(fr[0], fr[i ? -1 : 0], i == 0, T, x, y, z, v, gr);
      if (VAL) t[0][lane][i0 + i] = v;
      if (GRAD) {
#pragma unroll
        for (int k = 0; k < 3; ++k) t[(G0 + k) % NARR][lane][i0 + i] = gr[k];
      }
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < NARR; ++a) {
      for (int r = threadIdx.x / CR_F; r < 64; r += 256 / CR_F)
        if (m0 + c < nbf && g0 + r < npts) out[a][(g0 + r) * nbf + m0 + c] = t[a][r][c];
    }
    __syncthreads();
  }
}

void launch_collocation_ref(hipStream_t s, int nbf, const FuncRec *f, const HarmTerm *t,
                            int64_t npts, const double *pts, double *phi, double *gx,
                            double *gy, double *gz) {
  if (nbf <= 0 || npts <= 0) return;
  const int64_t step = max_workgroups(256) * 64;  // points of a launch
  if (npts > step) {
    auto at = [&](double *p) { return p ? p + step * nbf : p; };
    launch_collocation_ref(s, nbf, f, t, step, pts, phi, gx, gy, gz);
    launch_collocation_ref(s, nbf, f, t, npts - step, pts + 3 * step, at(phi), at(gx), at(gy),
                           at(gz));
    return;
  }
  const int64_t nwg = (npts + 63) / 64;
  // Small outputs: narrow tiles (FW 4, 2 below one workgroup per CU), each a
  // workgroup of its own, for shorter chains and more waves in flight; the lines
  // that two tiles share meet in the last-level cache (256 MB, shared with what
  // else is held).  Larger ones: those lines would go to memory twice, so tiles are
  // 32 functions wide and one workgroup writes all of its points' tiles, or where
  // that makes fewer than 2048 workgroups (eight a CU) every ny-th of them.  Both
  // calls, us (FW 8 in a loop / FW 4 each its own): 9 MB of output 72.3 / 69.6, 71
  // MB 96 / 83, 0.5 GB 269 / 308, 2.2 GB 799 / 1246; FW 2 at 4 MB 64.5 for 67.2.
  // Values and gradients, us (one workgroup / ny by 2048 / a workgroup each tile / FW
  // 4 each its own): 1200 functions at 3 840 points 585 / 213 / 206 / 191, 400 at 28
  // 800 262 / 197 / 183 / 168, 110 at 62 370 155 / 150 / 154 / 168, 110 at 176 418
  // 319 / 320 / 338 / 398.
  const int64_t bytes = (int64_t)8 * nbf * npts * ((phi ? 1 : 0) + (gx ? 3 : 0));
  const int fw = bytes > ((int64_t)1 << 26) ? 8 : nwg < 256 ? 2 : 4;
  const int64_t tiles = (nbf + 4 * fw - 1) / (4 * fw);
  const unsigned ny =
      (unsigned)(fw == 8 ? std::min<int64_t>(tiles, std::max<int64_t>(1, 2048 / nwg)) : tiles);
#define NKX_COLLOC_FW(V, G, W)                                                              \
  hipLaunchKernelGGL((colloc_ref_kernel<V, G, W>), dim3((unsigned)nwg, ny), dim3(256), 0, s, \
                     nbf, f, t, npts, pts, phi, gx, gy, gz)
#define NKX_COLLOC(V, G)                 \
  if (fw == 8) NKX_COLLOC_FW(V, G, 8);   \
  else if (fw == 4) NKX_COLLOC_FW(V, G, 4); \
  else NKX_COLLOC_FW(V, G, 2)
  if (gx && phi) {
    NKX_COLLOC(true, true);
  } else if (gx) {
    NKX_COLLOC(false, true);
  } else {
    NKX_COLLOC(true, false);
  }
#undef NKX_COLLOC_FW
#undef NKX_COLLOC
  NKX_HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Plain device copy with 16-byte vector loads and stores (grid-stride).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) copy16_kernel(int64_t n, const int4 *__restrict__ src,
                                                     int4 *__restrict__ dst) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

void launch_copy16(hipStream_t s, void *dst, const void *src, size_t bytes) {
  const int64_t n = (int64_t)(bytes / 16);
  if (n == 0) return;
  const int64_t blocks = std::min<int64_t>((n + 255) / 256, 256 * 32);
  hipLaunchKernelGGL(copy16_kernel, dim3((unsigned)blocks), dim3(256), 0, s, n,
                     reinterpret_cast<const int4 *>(src), reinterpret_cast<int4 *>(dst));
  NKX_HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Functional evaluation on device arrays.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) functional_kernel(XcList xl, int64_t npts,
                                                         const double *__restrict__ rho,
                                                         const double *__restrict__ sigma,
                                                         double *exc, double *vrho,
                                                         double *vsigma) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= npts) return;
  const double r = rho[g];
  const XcPoint o = xc_eval(xl.n, xl.ids, xl.thr, r, sigma ? sigma[g] : 0.0);
  exc[g] = r > 0.0 ? o.e / r : 0.0;
  vrho[g] = o.vrho;
  if (vsigma) vsigma[g] = o.vsigma;
}

void launch_functional_eval(hipStream_t s, XcList xl, int64_t npts, const double *rho,
                            const double *sigma, double *exc, double *vrho, double *vsigma) {
  if (npts == 0) return;
  hipLaunchKernelGGL(functional_kernel, dim3((unsigned)((npts + 255) / 256)), dim3(256), 0, s, xl,
                     npts, rho, sigma, exc, vrho, vsigma);
  NKX_HIP_CHECK(hipGetLastError());
}

// Spin-polarised evaluation, libxc XC_POLARIZED layout (rho[2g+s],
// sigma[3g+k], vrho[2g+s], vsigma[3g+k]); exc per particle.
__global__ void __launch_bounds__(256) functional_pol_kernel(XcList xl, int64_t npts,
                                                             const double *__restrict__ rho,
                                                             const double *__restrict__ sigma,
                                                             double *exc, double *vrho,
                                                             double *vsigma) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= npts) return;
  const double r[2] = {rho[2 * g], rho[2 * g + 1]};
  const double sg[3] = {sigma ? sigma[3 * g] : 0.0, sigma ? sigma[3 * g + 1] : 0.0,
                        sigma ? sigma[3 * g + 2] : 0.0};
  double e, vr[2], vs[3];
  xc_eval_polarized(xl.n, xl.ids, xl.thr, r, sg, e, vr, vs);
  exc[g] = e;
  vrho[2 * g] = vr[0];
  vrho[2 * g + 1] = vr[1];
  if (vsigma) {
    vsigma[3 * g] = vs[0];
    vsigma[3 * g + 1] = vs[1];
    vsigma[3 * g + 2] = vs[2];
  }
}

void launch_functional_eval_pol(hipStream_t s, XcList xl, int64_t npts, const double *rho,
                                const double *sigma, double *exc, double *vrho,
                                double *vsigma) {
  if (npts == 0) return;
  hipLaunchKernelGGL(functional_pol_kernel, dim3((unsigned)((npts + 255) / 256)), dim3(256), 0,
                     s, xl, npts, rho, sigma, exc, vrho, vsigma);
  NKX_HIP_CHECK(hipGetLastError());
}

}  // namespace nkx
