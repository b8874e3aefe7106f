// Reference-shaped density and XC assembly on collocation matrices that the
// caller holds (density.hpp:150-255, xc_integrals.hpp:73-262, :424-718):
// LayoutLeft (N_bf, N_pts), element (mu, g) at mu + g N_bf, FP64 throughout.
//
//   density_mo   psi_i = sum_mu C(mu, i) Phi(mu, g) and its gradient on FP64
//                MFMA, rho = sum_i f_i psi_i^2, grad rho = 2 sum_i f_i psi_i
//                grad psi_i; then either rho, grad rho, sigma per point or the
//                functional and the Z coefficients of the point
//   zv_ref       Z = a Phi + b . grad Phi formed on the way into LDS and the
//                split-K contraction Vbar = Phi Z^T on FP64 MFMA
//   finish_ref   sum of the split partials, and E (mirror_ref: V = Vbar +
//                Vbar^T where zv_ref did not form it)
//   density_few  rho, grad rho, sigma of up to eight functions
//
// The four matrices are read twice per call (once per contraction) and nothing
// of their size is written.
#include <algorithm>

#include "lane_sums.hpp"
#include "nkx_internal.hpp"
#include "xc_functionals.hpp"
#include "xc_polarized.hpp"

namespace nkx {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
// four doubles at any 8-byte aligned address (rows of an odd N_bf)
typedef double v4u __attribute__((ext_vector_type(4), aligned(8)));

constexpr int MP = 64;  // points per density workgroup, 16 per wave

struct MoSpin {
  int nocc;
  const double *C, *f;  // C LayoutLeft (N_bf, nocc)
};

struct RefGrads {
  const double *a[4];  // Phi, dPhi/dx, dPhi/dy, dPhi/dz
};

struct RhoOut {
  double *rho, *gx, *gy, *gz, *sigma;  // all but rho may be NULL
};

// ---------------------------------------------------------------------------
// One workgroup of four waves per 64 points, a wave per 16.  MFMA rows are
// points, columns orbitals: lane (q, l16) of the wave reads the four functions
// 16 kk + 4 q .. + 3 of point l16 and of orbital l16 (the order of the
// contraction index is free, so that a point's four lanes read one 128-byte
// line), four MFMA steps per load.  Up to four orbital tiles of 16 are held at
// once (of both spins together, so that an open shell reads the matrices
// once); more of them take further passes.  Tail functions are masked to zero and
// columns past nocc never enter a sum, so no value of a neighbouring row
// does.
//
// Bound by reading the four matrices (6.1 TB/s) where one tile is enough, by
// the FP64 MFMA rate (2048 flops per 64 cycles and SIMD) from about three
// tiles on.  A thread per point with a scalar loop over orbitals and
// functions reads each matrix once per orbital, uncoalesced: 41.6 ms per spin
// on benzene (120 functions, 259 200 points, 21 and 20 orbitals), 288 us on
// water (25 functions, 64 800 points, 5 orbitals); this form takes 328 us for
// both spins (3.0 TB/s; 364 us with tiles of each spin's own, four instead of
// three, and the last functions' loads under conditions) and 23 us.
//
// MODE 0 writes rho, grad rho and sigma of one spin; 1 evaluates the
// functional and writes the Z coefficients (w v_rho / 2, 2 w v_sigma grad rho)
// and the energy of the 64 points; 2 (two spins) writes (rho, grad rho) per
// spin into coef for xc_pol_ref, whose functional holds more registers than
// the contraction can spare at two waves per SIMD.
enum MoMode { kMoDensity = 0, kMoXc = 1, kMoSpins = 2 };

// One pass of a wave over the functions with NT tiles of 16 orbitals, t0 .. t0 +
// NT - 1 of the n0 + n1 orbitals of both spins in a row (a tile may hold both);
// row[a]: this lane's point in matrix a.
template <int NARR, int NT, int NS>
__device__ __forceinline__ void mo_pass(int nbf, const double *const (&row)[NARR], int t0,
                                        int n0, int n1, const double *__restrict__ C0,
                                        const double *__restrict__ C1,
                                        const double *__restrict__ f0,
                                        const double *__restrict__ f1, int l16, int q, int wv,
                                        double (*red)[NARR][MP]) {
  const int nfull = nbf / 16;  // whole blocks of functions
  // a lane's four functions of block kk at p (p points at function 4 q)
  auto load = [&](const double *p, int kk) -> v4d {
    const v4u t = *reinterpret_cast<const v4u *>(p + 16 * kk);
    return v4d{t[0], t[1], t[2], t[3]};
  };
  // of the last, partial block; past the end the last function again, and zero
  // for the orbitals (loads under a condition become branches, each with a wait
  // for the loads before it)
  auto load_tail = [&](const double *p) -> v4d {
    v4d t;
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] = p[min(16 * nfull + e, nbf - 1 - 4 * q)];
    return t;
  };
  const double *cp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int n = NS == 2 ? n0 + n1 : n0;
    const int col = min(16 * (t0 + t) + l16, n - 1);
    const bool s1 = NS == 2 && col >= n0;
    cp[t] = (s1 ? C1 : C0) + (int64_t)(s1 ? col - n0 : col) * nbf + 4 * q;
  }
  v4d acc[NT][NARR];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int a = 0; a < NARR; ++a) acc[t][a] = v4d{0.0, 0.0, 0.0, 0.0};
  auto products = [&](const v4d(&A)[NARR], const v4d(&B)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int a = 0; a < NARR; ++a)
          acc[t][a] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[a][e], B[t][e], acc[t][a], 0, 0, 0);
  };
  v4d A[NARR], B[NT];
  if (nfull) {
#pragma unroll
    for (int a = 0; a < NARR; ++a) A[a] = load(row[a], 0);
  }
  // the matrices' fragments one block ahead, the orbitals' (cached) in time
#pragma unroll 1
  for (int kk = 0; kk < nfull; ++kk) {
    v4d An[NARR];
    const int kn = kk + 1 < nfull ? kk + 1 : kk;
#pragma unroll
    for (int t = 0; t < NT; ++t) B[t] = load(cp[t], kk);
    __builtin_amdgcn_sched_barrier(0);  // the products wait for B alone
#pragma unroll
    for (int a = 0; a < NARR; ++a) An[a] = load(row[a], kn);
    products(A, B);
#pragma unroll
    for (int a = 0; a < NARR; ++a) A[a] = An[a];
  }
  if (16 * nfull < nbf) {
#pragma unroll
    for (int a = 0; a < NARR; ++a) A[a] = load_tail(row[a]);
#pragma unroll
    for (int t = 0; t < NT; ++t) B[t] = load_tail(cp[t]);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (16 * nfull + 4 * q + e >= nbf) B[t][e] = 0.0;
    products(A, B);
  }
  // f psi psi_a summed over the pass's orbitals, spin by spin
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    double v[4 * NARR];
#pragma unroll
    for (int k = 0; k < 4 * NARR; ++k) v[k] = 0.0;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int c0 = 16 * (t0 + t) - (s ? n0 : 0), col = c0 + l16;  // of the spin
      if (c0 > -16 && col >= 0 && col < (s ? n1 : n0)) {
        const double f = s ? f1[col] : f0[col];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const double fp = f * acc[t][0][r];
#pragma unroll
          for (int a = 0; a < NARR; ++a) v[4 * a + r] += fp * acc[t][a][r];
        }
      }
    }
    if constexpr (NARR == 4) {
      const double tot = row_sum16(v, l16);
      const int k = bitrev4(l16);
      red[s][k >> 2][16 * wv + 4 * (k & 3) + q] += tot;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        double x = v[r];
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) x += __shfl_xor(x, o);
        if (l16 == r) red[s][0][16 * wv + 4 * r + q] += x;
      }
    }
  }
}

template <int NARR, int MAXT, int MODE>
__global__ void __launch_bounds__(256, MAXT == 1 ? 3 : 2) density_mo(
    int nbf, int64_t npts, RefGrads in, int n0, int n1, const double *__restrict__ C0,
    const double *__restrict__ C1, const double *__restrict__ f0, const double *__restrict__ f1,
    RhoOut out, XcList xl, const double *__restrict__ w, double *__restrict__ coef,
    double *__restrict__ epart) {
  constexpr int NS = MODE == kMoSpins ? 2 : 1;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, q = lane >> 4;
  const int64_t g0 = (int64_t)blockIdx.x * MP;
  const int64_t gr = g0 + 16 * wv + l16;
  const int64_t off = (gr < npts ? gr : npts - 1) * nbf + 4 * q;
  const double *row[NARR];
#pragma unroll
  for (int a = 0; a < NARR; ++a) row[a] = in.a[a] + off;
  const int nt = ((NS == 2 ? n0 + n1 : n0) + 15) / 16;
  // sums over the orbitals; a slot belongs to one wave until the barrier
  __shared__ double red[NS][NARR][MP];
#pragma unroll
  for (int k = 0; k < NS * NARR; ++k)
    if (q == 0) (&red[0][0][0])[k * MP + 16 * wv + l16] = 0.0;
  wave_fence();
#define NKX_PASS(NT, T0) \
  mo_pass<NARR, NT, NS>(nbf, row, T0, n0, n1, C0, C1, f0, f1, l16, q, wv, red)
  if constexpr (MAXT == 1) {
    if (nt) NKX_PASS(1, 0);
  } else {
    int t0 = 0;
    for (; t0 + 4 <= nt; t0 += 4) NKX_PASS(4, t0);
    if (nt - t0 == 1) NKX_PASS(1, t0);
    else if (nt - t0 == 2) NKX_PASS(2, t0);
    else if (nt - t0 == 3) NKX_PASS(3, t0);
  }
#undef NKX_PASS

  __syncthreads();
  if (wv != 0) return;
  const int64_t g = g0 + lane;
  const bool live = g < npts;
  if constexpr (MODE == kMoDensity) {
    if (!live) return;
    out.rho[g] = red[0][0][lane];
    if constexpr (NARR == 4) {
      const double a = red[0][1][lane], b = red[0][2][lane], c = red[0][3][lane];
      if (out.gx) {
        out.gx[g] = 2.0 * a;
        out.gy[g] = 2.0 * b;
        out.gz[g] = 2.0 * c;
      }
      if (out.sigma) out.sigma[g] = 4.0 * (a * a + b * b + c * c);
    }
    return;
  }
  if constexpr (MODE == kMoSpins) {
    if (!live) return;
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int a = 0; a < 4; ++a)
        coef[8 * g + 4 * s + a] = a >= NARR ? 0.0 : (a ? 2.0 : 1.0) * red[s][a % NARR][lane];
    return;
  }
  if constexpr (MODE == kMoXc) {
    double e = 0.0;
    if (live) {
      const double wg = w[g], r = red[0][0][lane];
      double d[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) d[k] = NARR == 4 ? 2.0 * red[0][(k + 1) % NARR][lane] : 0.0;
      const XcPoint o =
          xc_eval(xl.n, xl.ids, xl.thr, r, d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
      const double b = 2.0 * wg * o.vsigma;
      coef[4 * g] = 0.5 * wg * o.vrho;
#pragma unroll
      for (int k = 0; k < 3; ++k) coef[4 * g + 1 + k] = NARR == 4 ? b * d[k] : 0.0;
      e = r > 0.0 ? wg * o.e : 0.0;
    }
    for (int o = 32; o > 0; o >>= 1) e += __shfl_down(e, o);
    if (lane == 0) epart[blockIdx.x] = e;
  }
}

// rho, grad rho and sigma of a basis of NB functions, a point per thread: the
// point's rows are read once, into registers.  Taken to eight functions, where
// density_mo spends more on a workgroup's set-up, exchange and barrier than on its
// 64 points (with the gradient nine take 188 us in both, values gain up to twelve).
// Two million points, call times in us, here and there: 1 function 25 and 75, with
// the gradient 49 and 156; 3 functions 30 and 76, 68 and 162; 8 functions 41 and
// 77, 140 and 195, with 40 orbitals 58 and 180, 151 and 501; 100 000 points 22 and
// 26, 32 and 39.
template <int NARR, int NB>
__global__ void __launch_bounds__(256) density_few(int64_t npts, RefGrads in, int nocc,
                                                   const double *__restrict__ C,
                                                   const double *__restrict__ f, RhoOut out) {
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (g >= npts) return;
  double x[NARR][NB], v[NARR];
#pragma unroll
  for (int a = 0; a < NARR; ++a) {
    v[a] = 0.0;
#pragma unroll
    for (int k = 0; k < NB; ++k) x[a][k] = in.a[a][g * NB + k];
  }
  for (int i = 0; i < nocc; ++i) {
    double psi[NARR];
#pragma unroll
    for (int a = 0; a < NARR; ++a) {
      psi[a] = 0.0;
#pragma unroll
      for (int k = 0; k < NB; ++k) psi[a] = fma(C[i * NB + k], x[a][k], psi[a]);
    }
    const double fp = f[i] * psi[0];
#pragma unroll
    for (int a = 0; a < NARR; ++a) v[a] = fma(fp, psi[a], v[a]);
  }
  out.rho[g] = v[0];
  if constexpr (NARR == 4) {
    if (out.gx) {
      out.gx[g] = 2.0 * v[1];
      out.gy[g] = 2.0 * v[2];
      out.gz[g] = 2.0 * v[3];
    }
    if (out.sigma) out.sigma[g] = 4.0 * (v[1] * v[1] + v[2] * v[2] + v[3] * v[3]);
  }
}

// The polarised functional per point: (rho, grad rho) per spin in coef become
// the Z coefficients (w v_rho_s / 2, w (2 v_sigma_ss grad rho_s + v_sigma_ab
// grad rho_s')); energies per 64 points.
__global__ void __launch_bounds__(64) xc_pol_ref(int64_t npts, int gga, XcList xl,
                                                 const double *__restrict__ w,
                                                 double *__restrict__ coef,
                                                 double *__restrict__ epart) {
  const int64_t g = (int64_t)blockIdx.x * MP + threadIdx.x;
  double e = 0.0;
  if (g < npts) {
    const double wg = w[g];
    double x[2][4];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int a = 0; a < 4; ++a) x[s][a] = coef[8 * g + 4 * s + a];
    const double r2[2] = {x[0][0], x[1][0]};
    const double sg[3] = {x[0][1] * x[0][1] + x[0][2] * x[0][2] + x[0][3] * x[0][3],
                          x[0][1] * x[1][1] + x[0][2] * x[1][2] + x[0][3] * x[1][3],
                          x[1][1] * x[1][1] + x[1][2] * x[1][2] + x[1][3] * x[1][3]};
    double exc, vr[2], vs[3];
    xc_eval_polarized(xl.n, xl.ids, xl.thr, r2, sg, exc, vr, vs);
    const double vab = wg * vs[1];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const double vss = 2.0 * wg * vs[2 * s];
      coef[8 * g + 4 * s] = 0.5 * wg * vr[s];
#pragma unroll
      for (int k = 1; k < 4; ++k)
        coef[8 * g + 4 * s + k] = gga ? vss * x[s][k] + vab * x[1 - s][k] : 0.0;
    }
    e = wg * (r2[0] + r2[1]) * exc;
  }
  for (int o = 32; o > 0; o >>= 1) e += __shfl_down(e, o);
  if (threadIdx.x == 0) epart[blockIdx.x] = e;
}

// ---------------------------------------------------------------------------
// Vbar(mu, nu) = sum_g Phi(mu, g) Z_s(nu, g) on TM x TM tiles, the points of
// one split per workgroup, Z formed from the four matrices on the way into LDS
// (both spins from one read).  KP points per stage, two LDS buffers: the next
// stage's elements (four per thread and matrix) go to registers while the
// current one's products run, one barrier per stage; the Z coefficients run
// one stage further ahead through a ring of three.  Rows of 16 functions are
// dealt to the waves in turn, and those past N_bf are skipped, so that a tile
// that is only partly used keeps its waves level.  TM is 32, 64 or 128: the
// smallest that holds the basis, so that each matrix is read once (a tile of
// 64 reads it twice from 65 functions on); from 129 on tiles of 128.
//
// LDS rows are 16 doubles longer than a multiple of 32, so that the two point
// rows that half a wave reads fall on different banks.
//
// Bound by reading the four matrices up to about 64 functions, by the FP64
// MFMA rate above.  With Z as a matrix of its own and a VALU kernel with
// atomics this took 318 + 772 us per spin on benzene and 81 + 247 us on water;
// now 405 us for both spins (42 TFLOP/s; 450 us with the loads under conditions
// and 510 with every wave forming Z after its products too) and 11.5 us (4.5 TB/s).
template <int TM>
struct ZvShape {
  static constexpr int threads = TM == 128 ? 512 : 256;
  static constexpr int KP = 4 * threads / TM;         // points per stage
  static constexpr int WR = 2, WC = threads / 64 / 2;  // waves over rows, columns
  static constexpr int NI = TM / 16 / WR, NJ = TM / 16 / WC;
  static constexpr int LD = TM + 16;
};

template <int TM, int NARR, int NS>
__global__ void __launch_bounds__(ZvShape<TM>::threads) zv_ref(
    int nbf, int64_t npts, int64_t kchunk, int nsplit, RefGrads in,
    const double *__restrict__ coef, double *__restrict__ part) {
  using S = ZvShape<TM>;
  constexpr int KP = S::KP, LD = S::LD, NI = S::NI, NJ = S::NJ, RPT = S::threads / TM;
  constexpr int SZ = 2 * KP * LD * (1 + NS);  // doubles of both stage buffers
  __shared__ double buf[SZ], cs[3][KP][4 * NS];
  double(*As)[KP][LD] = reinterpret_cast<double(*)[KP][LD]>(buf);
  double(*Zs)[NS][KP][LD] = reinterpret_cast<double(*)[NS][KP][LD]>(buf + 2 * KP * LD);
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, q = lane >> 4;
  const int wr = wv % S::WR, wc = wv / S::WR;
  const int ntile = (nbf + TM - 1) / TM;
  const int tile = blockIdx.x % (ntile * ntile);
  const int split = blockIdx.x / (ntile * ntile);
  const int m0 = (tile / ntile) * TM, n0 = (tile % ntile) * TM;
  const int64_t k0 = (int64_t)split * kchunk;
  const int64_t k1 = k0 + kchunk < npts ? k0 + kchunk : npts;
  const int c = threadIdx.x % TM, r0 = threadIdx.x / TM;
  const bool diag = m0 == n0;
  // functions and points past the end repeat the last one: those functions are
  // not written out, those points have zero coefficients.  (Loads under a
  // condition become branches, each with a wait for the loads before it.)
  const int cm = min(m0 + c, nbf - 1), cz = min(n0 + c, nbf - 1);

  double xa[4], xz[NARR][4];  // a stage's elements of this thread, rows r0 + RPT u
  auto load = [&](int64_t kb) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t e = min(kb + r0 + RPT * u, k1 - 1) * nbf;
#pragma unroll
      for (int a = 0; a < NARR; ++a) xz[a][u] = in.a[a][e + cz];
      if (diag) xa[u] = xz[0][u];  // uniform
    }
    if (!diag) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        xa[u] = in.a[0][min(kb + r0 + RPT * u, k1 - 1) * nbf + cm];
    }
  };
  auto load_coef = [&](int64_t kb) -> double {
    const int64_t e = 4 * NS * kb + threadIdx.x;
    return (int)threadIdx.x < KP * 4 * NS && e < 4 * NS * k1 ? coef[e] : 0.0;
  };
  auto store_coef = [&](int ring, double v) {
    if (threadIdx.x < KP * 4 * NS) (&cs[ring][0][0])[threadIdx.x] = v;
  };
  auto store = [&](int b, int ring) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = r0 + RPT * u;
      As[b][r][c] = xa[u];
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        double z = cs[ring][r][4 * s] * xz[0][u];
#pragma unroll
        for (int a = 1; a < NARR; ++a) z += cs[ring][r][4 * s + a] * xz[a][u];
        Zs[b][s][r][c] = z;
      }
    }
  };
  static_assert(KP * 4 * NS <= S::threads, "one coefficient per thread");

  v4d acc[NS][NI][NJ];
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[s][i][j] = v4d{0.0, 0.0, 0.0, 0.0};

  // this wave's 16-row and 16-column groups with functions in them
  const int ni = min(NI, max(0, ((nbf - m0 + 15) / 16 - wr + S::WR - 1) / S::WR));
  const int nj = min(NJ, max(0, ((nbf - n0 + 15) / 16 - wc + S::WC - 1) / S::WC));
  const int nst = k1 > k0 ? (int)((k1 - k0 + KP - 1) / KP) : 0;
  double cn = 0.0;  // this thread's coefficient of the stage after the next
  if (nst) {
    store_coef(0, load_coef(k0));
    store_coef(1, load_coef(k0 + KP));
    load(k0);
    __syncthreads();
    store(0, 0);
    if (nst > 1) load(k0 + KP);
    cn = load_coef(k0 + 2 * KP);
    __syncthreads();
  }
  // Waves w and w + 4 share a SIMD: one forms Z before its products, the other
  // after them, so that the matrix cores do not wait for both.
  const bool first = TM == 128 && wv < 4;
  int ring = 1;  // of stage s + 1
  for (int s = 0; s < nst; ++s) {
    const bool more = s + 1 < nst;
    const int b = s & 1;
    const int ring2 = ring == 2 ? 0 : ring + 1;
    // the next stage into the other buffer, the coefficients of the one after,
    // and then the loads (nothing after them waits before the next stage)
    auto next = [&]() {
      if (!more) return;
      store(b ^ 1, ring);
      store_coef(ring2, cn);
      if (s + 2 < nst) load(k0 + (int64_t)(s + 2) * KP);
      cn = load_coef(k0 + (int64_t)(s + 3) * KP);
    };
    if (first) next();
    {
#pragma unroll
      for (int ks = 0; ks < KP; ks += 4) {
        double av[NI], zv[NS][NJ];
#pragma unroll
        for (int i = 0; i < NI; ++i) av[i] = As[b][ks + q][16 * (wr + S::WR * i) + l16];
#pragma unroll
        for (int sp = 0; sp < NS; ++sp)
#pragma unroll
          for (int j = 0; j < NJ; ++j) zv[sp][j] = Zs[b][sp][ks + q][16 * (wc + S::WC * j) + l16];
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            if (i < ni && j < nj) {  // uniform
#pragma unroll
              for (int sp = 0; sp < NS; ++sp)
                acc[sp][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i], zv[sp][j],
                                                                     acc[sp][i][j], 0, 0, 0);
            }
      }
    }
    if (!first) next();
    ring = ring2;
    __syncthreads();
  }
  if constexpr (TM < 128) {
    // the basis fits this tile: Vbar + Vbar^T through LDS
    double(*t)[TM + 1] = reinterpret_cast<double(*)[TM + 1]>(buf);
    static_assert(SZ >= TM * (TM + 1), "the tile fits the stage buffers");
#pragma unroll
    for (int sp = 0; sp < NS; ++sp) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            t[16 * (wr + S::WR * i) + 4 * r + q][16 * (wc + S::WC * j) + l16] = acc[sp][i][j][r];
      __syncthreads();
      double *o = part + ((int64_t)sp * nsplit + split) * nbf * nbf;
      for (int mu = r0; mu < nbf; mu += RPT)
        if (c < nbf) o[mu * nbf + c] = t[mu][c] + t[c][mu];
    }
    return;
  }
#pragma unroll
  for (int sp = 0; sp < NS; ++sp) {
    double *o = part + ((int64_t)sp * nsplit + split) * nbf * nbf;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int nu = n0 + 16 * (wc + S::WC * j) + l16;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int mu = m0 + 16 * (wr + S::WR * i) + 4 * r + q;
          if (mu < nbf && nu < nbf) o[(int64_t)mu * nbf + nu] = acc[sp][i][j][r];
        }
      }
  }
}

// ---------------------------------------------------------------------------
// Sum of the split partials, element by element (n of them per spin, out +
// spin * n), and of the density workgroups' energies (the last workgroup).
// A workgroup takes 64 elements; its eight waves take an eighth of the splits
// each, 16 loads in flight, and are added in order.  Bound by the load latency
// for small bases: 9.5 us for 25 functions and 507 splits; tiles of 16 x 16
// summed with their mirror images in one workgroup (37 us) leave three CUs to
// issue all the loads.
__global__ void __launch_bounds__(512) finish_ref(int64_t n, int nsplit, unsigned nwv,
                                                  const double *__restrict__ part,
                                                  double *__restrict__ V0,
                                                  double *__restrict__ V1, int64_t ne,
                                                  const double *__restrict__ epart,
                                                  double *__restrict__ E) {
  __shared__ double sh[512];
  const unsigned wg = blockIdx.y * gridDim.x + blockIdx.x;
  if (wg >= nwv) {
    if (wg > nwv) return;
    double e = 0.0;
    for (int64_t i = threadIdx.x; i < ne; i += 512) e += epart[i];
    sh[threadIdx.x] = e;
    __syncthreads();
    for (int o = 256; o > 0; o >>= 1) {
      if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
      __syncthreads();
    }
    if (threadIdx.x == 0) *E = sh[0];
    return;
  }
  const unsigned per = (unsigned)((n + 63) / 64), sp = wg / per;
  const int64_t i = (int64_t)(wg % per) * 64 + (threadIdx.x & 63);
  const int wv = threadIdx.x >> 6;
  double v = 0.0;
  if (i < n) {
    const double *p = part + (int64_t)sp * nsplit * n + i;
    int s = (int)((int64_t)wv * nsplit / 8);
    const int s1 = (int)((int64_t)(wv + 1) * nsplit / 8);
    for (; s + 16 <= s1; s += 16) {
      double t[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) t[u] = p[(s + u) * n];
#pragma unroll
      for (int u = 0; u < 16; ++u) v += t[u];
    }
    for (; s < s1; ++s) v += p[s * n];
  }
  sh[threadIdx.x] = v;
  __syncthreads();
  if (wv || i >= n) return;
  v = 0.0;
#pragma unroll
  for (int k = 0; k < 8; ++k) v += sh[64 * k + threadIdx.x];
  (sp ? V1 : V0)[i] = v;
}

// V = Vbar + Vbar^T, 32 x 32 tiles (one per workgroup) through LDS
__global__ void __launch_bounds__(256) mirror_ref(int nbf, int64_t n,
                                                  const double *__restrict__ Vb,
                                                  double *__restrict__ V0,
                                                  double *__restrict__ V1) {
  __shared__ double t[32][33];
  const int nt = (nbf + 31) / 32, sp = blockIdx.x / (nt * nt), k = blockIdx.x % (nt * nt);
  const int i0 = 32 * (k / nt), j0 = 32 * (k % nt), c = threadIdx.x & 31;
  const double *src = Vb + sp * n;
  for (int r = threadIdx.x >> 5; r < 32; r += 8)
    if (j0 + r < nbf && i0 + c < nbf) t[r][c] = src[(int64_t)(j0 + r) * nbf + i0 + c];
  __syncthreads();
  for (int r = threadIdx.x >> 5; r < 32; r += 8)
    if (i0 + r < nbf && j0 + c < nbf) {
      const int64_t e = (int64_t)(i0 + r) * nbf + j0 + c;
      (sp ? V1 : V0)[e] = src[e] + t[c][r];
    }
}

template <int NARR, int MODE>
void launch_density_mo(hipStream_t s, int nbf, int64_t npts, const RefGrads &in,
                       const MoSpin &m0, const MoSpin &m1, const RhoOut &out, const XcList &xl,
                       const double *w, double *coef, double *epart) {
  // one tile of orbitals (at most 16 in all): three waves per SIMD instead of
  // two, as the loads are what bounds it (open-shell water 136 us per call with
  // the form for four tiles, 129)
#define NKX_MO(MAXT)                                                                        \
  hipLaunchKernelGGL((density_mo<NARR, MAXT, MODE>), dim3((unsigned)nwg), dim3(256), 0, s,  \
                     nbf, n, x, m0.nocc, m1.nocc, m0.C, m1.C, m0.f, m1.f, o, xl, at(w, g),  \
                     at(coef, (MODE == kMoSpins ? 8 : 4) * g), at(epart, g / MP))
  auto at = [](auto *p, int64_t i) { return p ? p + i : p; };
  const int64_t step = max_workgroups(256) * MP;  // points of a launch
  for (int64_t g = 0; g < npts; g += step) {
    const int64_t n = std::min(step, npts - g), nwg = (n + MP - 1) / MP;
    RefGrads x;
    for (int a = 0; a < 4; ++a) x.a[a] = at(in.a[a], g * nbf);
    const RhoOut o{at(out.rho, g), at(out.gx, g), at(out.gy, g), at(out.gz, g), at(out.sigma, g)};
    if (m0.nocc + (MODE == kMoSpins ? m1.nocc : 0) <= 16) NKX_MO(1);
    else NKX_MO(4);
    NKX_HIP_CHECK(hipGetLastError());
  }
#undef NKX_MO
}

// density_few where nbf is its NB; false: another size
template <int NARR, int NB>
bool launch_density_few(hipStream_t s, int nbf, int64_t npts, const RefGrads &in,
                        const MoSpin &mo, const RhoOut &out) {
  if constexpr (NB == 0) {
    return false;
  } else {
    if (nbf != NB) return launch_density_few<NARR, NB - 1>(s, nbf, npts, in, mo, out);
    const int64_t nwg = (npts + 255) / 256;
    NKX_REQUIRE(nwg <= max_workgroups(256), NKX_ERR_UNSUPPORTED, "too many points");
    hipLaunchKernelGGL((density_few<NARR, NB>), dim3((unsigned)nwg), dim3(256), 0, s, npts, in,
                       mo.nocc, mo.C, mo.f, out);
    NKX_HIP_CHECK(hipGetLastError());
    return true;
  }
}

template <int NARR, int NS>
void launch_zv(hipStream_t s, int nbf, int64_t npts, int64_t kchunk, int nsplit,
               const RefGrads &in, const double *coef, double *part) {
  const int tm = nbf <= 32 ? 32 : (nbf <= 64 ? 64 : 128);
  const int64_t nt = (nbf + tm - 1) / tm;
  const int64_t nwg = nt * nt * nsplit;
  NKX_REQUIRE(nwg <= max_workgroups(512), NKX_ERR_UNSUPPORTED, "V contraction grid too large");
#define NKX_ZV(TM)                                                                            \
  hipLaunchKernelGGL((zv_ref<TM, NARR, NS>), dim3((unsigned)nwg), dim3(ZvShape<TM>::threads), 0, \
                     s, nbf, npts, kchunk, nsplit, in, coef, part)
  if (tm == 32) NKX_ZV(32);
  else if (tm == 64) NKX_ZV(64);
  else NKX_ZV(128);
#undef NKX_ZV
  NKX_HIP_CHECK(hipGetLastError());
}

// Splits of the points of the V contraction: about one workgroup per CU for
// tiles of 128 (one fits at a time), two for the smaller ones, each with at
// least 64 points.  Without points one split of none, which leaves Vbar zero.
int ref_splits(int nbf, int64_t npts, int64_t *kchunk) {
  const int tm = nbf <= 32 ? 32 : (nbf <= 64 ? 64 : 128);
  const int64_t nt = (nbf + tm - 1) / tm;
  const int64_t want = std::max<int64_t>(1, (tm == 128 ? 256 : 512) / (nt * nt));
  const int64_t ns = std::max<int64_t>(1, std::min<int64_t>(want, npts / 64));
  *kchunk = std::max<int64_t>(32, ((npts + ns - 1) / ns + 31) / 32 * 32);
  return (int)std::max<int64_t>(1, (npts + *kchunk - 1) / *kchunk);
}

template <int NS>
void xc_ref(Ctx &c, int nbf, int64_t npts, const RefGrads &in, bool grad, const double *w,
            const MoSpin &m0, const MoSpin &m1, const XcList &xl, double *E, double *V0,
            double *V1) {
  hipStream_t s = c.stream;
  int64_t kchunk = 0;
  const int nsplit = ref_splits(nbf, npts, &kchunk);
  const int64_t ne = (npts + MP - 1) / MP;
  const size_t n_cf = 4 * NS * (size_t)npts, n_pt = (size_t)NS * nsplit * nbf * nbf;
  const size_t n_vb = nbf > 64 ? (size_t)NS * nbf * nbf : 0;
  c.ws.scratch.reserve(n_cf + n_pt + n_vb + ne);
  double *coef = c.ws.scratch.p, *part = coef + n_cf, *vb = part + n_pt, *ep = vb + n_vb;
  double *Ed = c.out_doubles(1);
  const RhoOut none{};
  if (npts > 0) {
    constexpr int mode = NS == 2 ? kMoSpins : kMoXc;
    if (grad)
      launch_density_mo<4, mode>(s, nbf, npts, in, m0, m1, none, xl, w, coef, ep);
    else
      launch_density_mo<1, mode>(s, nbf, npts, in, m0, m1, none, xl, w, coef, ep);
    if (NS == 2) {
      NKX_REQUIRE(ne <= max_workgroups(MP), NKX_ERR_UNSUPPORTED, "too many points");
      hipLaunchKernelGGL(xc_pol_ref, dim3((unsigned)ne), dim3(MP), 0, s, npts, grad ? 1 : 0, xl,
                         w, coef, ep);
      NKX_HIP_CHECK(hipGetLastError());
    }
  }
  if (grad)
    launch_zv<4, NS>(s, nbf, npts, kchunk, nsplit, in, coef, part);
  else
    launch_zv<1, NS>(s, nbf, npts, kchunk, nsplit, in, coef, part);
  // tiles of 128 leave Vbar; the smaller ones Vbar + Vbar^T
  const bool mirror = nbf > 64;
  const int64_t n = (int64_t)nbf * nbf, nwv = NS * ((n + 63) / 64);
  NKX_REQUIRE(nwv + 1 < (int64_t)1 << 31, NKX_ERR_UNSUPPORTED, "too many functions");
  hipLaunchKernelGGL(finish_ref, grid_2d(nwv + 1, 512), dim3(512), 0, s, n, nsplit, (unsigned)nwv,
                     part, mirror ? vb : V0, mirror ? vb + n : V1, ne, ep, Ed);
  NKX_HIP_CHECK(hipGetLastError());
  if (mirror) {
    const int64_t nt = (nbf + 31) / 32;
    NKX_REQUIRE(NS * nt * nt <= max_workgroups(256), NKX_ERR_UNSUPPORTED, "too many functions");
    hipLaunchKernelGGL(mirror_ref, dim3((unsigned)(NS * nt * nt)), dim3(256), 0, s, nbf, n, vb,
                       V0, V1);
    NKX_HIP_CHECK(hipGetLastError());
  }
  NKX_HIP_CHECK(hipStreamSynchronize(s));
  *E = *Ed;
}

}  // namespace

void launch_density_ref(hipStream_t s, int nbf, int64_t npts, const double *phi,
                        const double *gx, const double *gy, const double *gz, int nocc,
                        const double *C, const double *f, double *rho, double *grx,
                        double *gry, double *grz, double *sigma) {
  if (npts == 0) return;
  const RefGrads in{{phi, gx, gy, gz}};
  const MoSpin mo{nocc, C, f};
  const RhoOut out{rho, grx, gry, grz, sigma};
  const XcList none{};
  if (gx ? launch_density_few<4, 8>(s, nbf, npts, in, mo, out)
         : launch_density_few<1, 8>(s, nbf, npts, in, mo, out))
    return;
  if (gx)
    launch_density_mo<4, kMoDensity>(s, nbf, npts, in, mo, mo, out, none, nullptr, nullptr, nullptr);
  else
    launch_density_mo<1, kMoDensity>(s, nbf, npts, in, mo, mo, out, none, nullptr, nullptr, nullptr);
}

void xc_from_collocation_pol(Ctx &c, int nbf, int64_t npts, const double *phi, const double *gx,
                             const double *gy, const double *gz, const double *w, int nocca,
                             const double *Ca, const double *fa, int noccb, const double *Cb,
                             const double *fb, const XcList &xl, bool gga, double *E,
                             double *Va, double *Vb) {
  xc_ref<2>(c, nbf, npts, RefGrads{{phi, gx, gy, gz}}, gga && gx, w, MoSpin{nocca, Ca, fa},
            MoSpin{noccb, Cb, fb}, xl, E, Va, Vb);
}

void xc_from_collocation(Ctx &c, int nbf, int64_t npts, const double *phi, const double *gx,
                         const double *gy, const double *gz, const double *w, int nocc,
                         const double *C, const double *f, const XcList &xl, bool gga,
                         double *E, double *V) {
  const MoSpin mo{std::max(nocc, 0), C, f};  // a negative count: no orbitals
  xc_ref<1>(c, nbf, npts, RefGrads{{phi, gx, gy, gz}}, gga && gx, w, mo, mo, xl, E, V, V);
}

}  // namespace nkx
