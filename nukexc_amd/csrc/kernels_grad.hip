// Nuclear gradient of E_xc at fixed density matrix P (FP64).  The reference
// has no gradient; the terms follow from E = sum_g w_g f(rho_g, sigma_g) with
// basis functions centred on atoms, grid points moving with their owner atom
// and Becke weights w_g = w0_g P_B(r_g) / sum_i P_i(r_g) (B = owner):
//
//  basis-centre term, atom A, function mu on A, per point g:
//    c_mu(g) = -2 [ d phi_mu(g) (P Y)_mu(g) + (H_mu(g) b_g) (P Phi)_mu(g) ]
//    Y_nu(g) = w v_rho phi_nu + b_g . grad phi_nu,   b_g = 2 w v_sigma grad rho
//    (H_mu = Hessian of phi_mu; GGA only)
//  point-motion term: rigid translation of every atom together with the
//    point leaves rho(r_g) unchanged, so the owner receives -sum_mu c_mu(g);
//  weight term: f_g dw_g/dR_A = (w f)_g sum_i ([i == B]/P_B - 1/Z) dP_i/dR_A
//    for A != B, and the owner receives minus their sum (w is invariant under
//    rigid translation of atoms and point).
// Becke derivatives: P_i = prod_j s(mu_ij), mu_ij = (r_i - r_j)/R~_ij,
//   R~ = min(R_ij, 5) (capped) or R_ij, s = (1 - p(p(p(mu))))/2,
//   dmu_ij/dR_i = -u_i/R~ - [R~ = R_ij] mu (R_i - R_j)/R_ij^2,
//   dmu_ij/dR_j = +u_j/R~ + [R~ = R_ij] mu (R_i - R_j)/R_ij^2,
//   u_i = (r - R_i)/r_i; s' = 0 where mu is clamped at +-1.
#include "grad_rows.hpp"
#include "lane_sums.hpp"
#include "nkx_internal.hpp"
#include "vxc_kernels.hpp"

namespace nkx {

typedef double v4d __attribute__((ext_vector_type(4)));

namespace {
constexpr int FB = 64;
constexpr int PT = 64;
constexpr int TILE = FB * PT;
constexpr int GC = FB * 3;  // per-slot partial: 64 functions x 3 components
}  // namespace

// ---------------------------------------------------------------------------
// Basis-centre term: X = P Phi and W = P Y (Y in tile array yarr) for one pair
// of a batch's live blocks, then grad_rows.  One workgroup of four waves per
// (batch, pair of list blocks); a wave holds 32 rows of its block x 64 points
// of both products (16 rows of the only block where the pair has one).  The
// contraction is that of density_fused_f64 (kernels_density.hip) in stages of 16
// functions: Phi and Y of the next stage go straight into the other LDS
// buffer and the next P fragments into the other register set while the
// current stage's products run.  The epilogue passes X and W of a wave through
// its own part of the buffers, eight rows at a time, to a point per lane.
// cpart[(slot - s0) 192 + 3 mu + k]: per function; tpart[(slot - s0) 256 + 64 k +
// point], slot the pair's first: per point, over the pair's functions.
//
// Bound by the FP64 MFMA rate and FP64 VALU issue (grad_rows) in turn; see
// there for what the epilogue took before.
constexpr int GS = 16;           // functions of a stage
constexpr int GSTG = GS * PT;    // doubles of one array's stage

// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima)
__device__ __forceinline__ void wait_vm0() { __builtin_amdgcn_s_waitcnt(0x0F70); }

__global__ void __launch_bounds__(256, 2) grad_basis_f64(
    MolTab mt, const double *__restrict__ Pt, const int *__restrict__ b_off,
    const int *__restrict__ b_fbl, int64_t s0, int64_t b0, int64_t b1, int nmg, int narr,
    int yarr, int gga, const double *__restrict__ tiles, const double *__restrict__ coef,
    const FuncRec *__restrict__ F, const HarmTerm *__restrict__ T,
    const double *__restrict__ px, const double *__restrict__ py,
    const double *__restrict__ pz, double *__restrict__ cpart, double *__restrict__ tpart) {
  // the pairs of a batch run on one XCD (workgroups are dealt to the eight
  // XCDs in turn) and share its L2 for the tiles
  const int xcd = blockIdx.x & 7, rr = blockIdx.x >> 3;
  const int mgi = rr % nmg;
  const int64_t b = b0 + (int64_t)(rr / nmg) * 8 + xcd;
  if (b >= b1) return;
  const int lo = b_off[b], n = b_off[b + 1] - lo;
  if (2 * mgi >= n) return;  // uniform
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, q = lane >> 4;
  // Phi, Y of a stage; two buffers, declared apart so that a copy into one is
  // known not to touch the other
  __shared__ __attribute__((aligned(16))) double bufA[2][GSTG];
  __shared__ __attribute__((aligned(16))) double bufB[2][GSTG];
  __shared__ double red[4][3][PT];
  const bool two = 2 * mgi + 1 < n;
  const int im = lo + 2 * mgi + (two ? wv >> 1 : 0);
  const int fm = __builtin_amdgcn_readfirstlane(b_fbl[im]);
  const int mol = mt.blk_mol[fm], ld = mt.ld[mol];
  const int row0 = two ? 32 * (wv & 1) : 16 * wv;  // of the block
  const int mbase = fm - mt.blk_local[fm];
  const double *prow =
      Pt + mt.P_off[mol] + (int64_t)(mt.blk_local[fm] * FB + row0 + l16) * ld + 4 * q;
  v4d accX[2][4], accW[2][4];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int j = 0; j < 4; ++j) accX[g][j] = accW[g][j] = v4d{0.0, 0.0, 0.0, 0.0};
  auto issue = [&](int s, double (*dst)[GSTG], v4d (&a)[2]) {
    const int ki = lo + (s >> 2), h = s & 3;
    const int fk = __builtin_amdgcn_readfirstlane(b_fbl[ki]);
    const double *p = prow + (fk - mbase) * FB + GS * h;
    a[0] = *reinterpret_cast<const v4d *>(p);
    if (two) a[1] = *reinterpret_cast<const v4d *>(p + (int64_t)16 * ld);
    const double *src = tiles + (int64_t)(ki - s0) * narr * TILE + GSTG * h;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      // rows 2 rp, 2 rp + 1: 16 bytes per lane, halves exchanged in rows with
      // bit 2 set (density_fused_f64)
      const int rp = 2 * wv + u, r = 2 * rp + (lane >> 5);
      const int c = (lane & 31) ^ (((rp >> 1) & 1) << 3);
      const double *g = src + r * PT + 2 * c;
      __builtin_amdgcn_global_load_lds(g, &dst[0][rp * 2 * PT], 16, 0, 0);
      __builtin_amdgcn_global_load_lds(g + (int64_t)yarr * TILE, &dst[1][rp * 2 * PT], 16, 0, 0);
    }
  };
  auto products = [&](const double (*cur)[GSTG], const v4d (&a)[2]) {
    const int col = l16 ^ ((q & 1) << 4);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int op = 0; op < 2; ++op) {
        double bv[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) bv[j] = cur[op][(4 * q + e) * PT + ((16 * j) ^ col)];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          if (g && !two) continue;  // uniform
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            v4d &acc = op ? accW[g][j] : accX[g][j];
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[g][e], bv[j], acc, 0, 0, 0);
          }
        }
      }
  };
  v4d a0[2], a1[2];
  issue(0, bufA, a0);
  for (int s = 0; s < 4 * n; s += 2) {
    wait_vm0();
    __syncthreads();  // bufA complete, bufB free
    issue(s + 1, bufB, a1);
    products(bufA, a0);
    wait_vm0();
    __syncthreads();
    if (s + 2 < 4 * n) issue(s + 2, bufA, a0);
    products(bufB, a1);
  }
  // epilogue: wave w's part of the buffers holds eight rows of X, then of W
  const int64_t gp = b * PT + lane;
  const GradPoint pt{px[gp], py[gp], pz[gp], coef[4 * gp + 1], coef[4 * gp + 2], coef[4 * gp + 3]};
  double tp[3] = {0.0, 0.0, 0.0};
  double *Xs = (wv & 2 ? &bufB[0][0] : &bufA[0][0]) + (wv & 1) * GSTG, *Ws = Xs + 8 * GR_LD;
  static_assert(2 * 8 * GR_LD <= GSTG, "eight rows of X and W per wave");
  __syncthreads();  // the buffers' readers are done
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    if (g && !two) continue;
    GradFuncs gf;
    gf.load(F + (int64_t)fm * FB + row0 + 16 * g, lane);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          Xs[(4 * r + q) * GR_LD + 16 * j + l16] = accX[g][j][2 * h + r];
          Ws[(4 * r + q) * GR_LD + 16 * j + l16] = accW[g][j][2 * h + r];
        }
      wave_fence();
      grad_rows<8>(gf, 8 * h, T, pt, gga, Xs, Ws, lane,
                   cpart + (im - s0) * GC + 3 * (row0 + 16 * g + 8 * h), tp);
      wave_fence();
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) red[wv][k][lane] = tp[k];
  __syncthreads();
  if (threadIdx.x < 3 * PT) {
    const int k = threadIdx.x / PT, g = threadIdx.x % PT;
    tpart[(int64_t)(lo + 2 * mgi - s0) * (4 * PT) + threadIdx.x] =
        ((red[0][k][g] + red[1][k][g]) + red[2][k][g]) + red[3][k][g];
  }
}

// tpt[3 point + k] = -(sum over a batch's block pairs), or that added to tpt
__global__ void __launch_bounds__(192) grad_points_kernel(int64_t s0, int64_t b0,
                                                          const int *__restrict__ b_off,
                                                          const double *__restrict__ tpart,
                                                          int accum, double *__restrict__ tpt) {
  const int64_t b = b0 + blockIdx.x;
  const int k = threadIdx.x / PT, g = threadIdx.x % PT;
  double t = 0.0;
  for (int s = b_off[b]; s < b_off[b + 1]; s += 2) t += tpart[(s - s0) * (4 * PT) + threadIdx.x];
  const int64_t e = 3 * (b * PT + g) + k;
  tpt[e] = (accum ? tpt[e] : 0.0) - t;
}

// gacc[seg][I * 192 + t] += sum over batches of segment seg of cpart of block I
__global__ void __launch_bounds__(256) grad_fold_kernel(int64_t nb, int64_t b0, int64_t b1,
                                                        int64_t s0, int nseg, int nbf_pad,
                                                        const int *__restrict__ tile_slot,
                                                        const double *__restrict__ cpart,
                                                        double *__restrict__ gacc) {
  const int I = blockIdx.x, seg = blockIdx.y;
  const int t = threadIdx.x;
  if (t >= GC) return;
  const int64_t n = b1 - b0;
  const int64_t lo = b0 + n * seg / nseg, hi = b0 + n * (seg + 1) / nseg;
  const int *ts = tile_slot + (int64_t)I * nb;
  double acc = 0.0;
  for (int64_t b = lo; b < hi; ++b) {
    const int sl = ts[b];
    if (sl >= 0) acc += cpart[(sl - s0) * GC + t];
  }
  gacc[(int64_t)seg * nbf_pad * 3 + I * GC + t] += acc;
}

__global__ void __launch_bounds__(256) owners_kernel(int64_t n, const int *__restrict__ pidx,
                                                     const int *__restrict__ owner,
                                                     int *__restrict__ pown) {
  const int64_t sp = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (sp >= n) return;
  const int src = pidx[sp];
  pown[sp] = src >= 0 ? owner[src] : -1;
}

__device__ __forceinline__ double bp(double x) { return 1.5 * x - 0.5 * x * x * x; }
__device__ __forceinline__ double bdp(double x) { return 1.5 * (1.0 - x * x); }

__device__ __forceinline__ double gdist(double x, double y, double z, const double *c) {
  const double dx = x - c[0], dy = y - c[1], dz = z - c[2];
  return sqrt(dx * dx + dy * dy + dz * dz);
}

// Per atom pair (i, j): 1/R~_ij and the factor of the mu (R_i - R_j) term of
// dmu_ij/dR, [R~ = R_ij] / R_ij^2 (zero where the cap applies), with
// R~ = min(R_ij, 5) (capped partition) or R_ij.  One thread per pair.
__global__ void __launch_bounds__(256) pair_table_kernel(int natoms, const double *__restrict__ C,
                                                         int cap, double2 *__restrict__ tab) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= natoms * natoms) return;
  const int i = e / natoms, j = e % natoms;
  const double dx = C[3 * i] - C[3 * j], dy = C[3 * i + 1] - C[3 * j + 1],
               dz = C[3 * i + 2] - C[3 * j + 2];
  const double R = sqrt(dx * dx + dy * dy + dz * dz);
  const bool capped = cap && R >= 5.0;
  tab[e] = i == j ? make_double2(0.0, 0.0)
                  : make_double2(1.0 / (capped ? 5.0 : R), capped ? 0.0 : 1.0 / (R * R));
}

// One thread per sorted point, one wave per workgroup; per-atom sums in LDS
// (3 natoms doubles).  The candidates (atoms whose cell function can be nonzero
// at some point of the wave) are taken WC at a time in registers: one sweep over
// j multiplies their cell functions P_i and adds them to Z = sum P_i, and once Z
// is known a second one adds the derivative terms of all of them, so that r_j is
// formed once per WC candidates and the force on atom j is summed over them
// before it is summed over the wave.  The cell functions of the first WKEEP
// groups stay in LDS in between; those of later ones (more than 16 atoms near a
// wave) are formed again.  Loops over atoms run in step across the wave (lanes
// without a contribution add zero); each per-atom term is summed over the wave
// (wave_sum: every lane active) and added to LDS by lane 0.  With one writer per
// workgroup (no atomics) the sums, and so the gradient, come out the same on
// every run.  The points of a wave are 64 consecutive sorted points (npts_pad
// and the grid stride are multiples of 64), so every lane runs the same trip
// count.  ptab: the atom-pair table of pair_table_kernel.  |mu| >= 1 gives the
// factor 1 or 0 exactly and no derivative.
//
// Bound by FP64 VALU issue.  A 30-atom molecule, 648 000 points: 2267 us with
// one candidate at a time (a square root per pair in both sweeps, three wave
// sums per pair), 1333 with four, 1091 with the cell functions kept and the
// quotient by s_ij through recip; WC = 3 and 6 cost 6 % more (registers).
constexpr int WC = 4;   // candidates in registers
constexpr int WKEEP = 4;  // groups of WC whose cell functions are kept in LDS

// 1 / a, 0 < a normal: the estimate and two Newton steps (within an ulp)
__device__ __forceinline__ double recip(double a) {
  double y = __builtin_amdgcn_rcp(a);
  y = fma(fma(-a, y, 1.0), y, y);
  return fma(fma(-a, y, 1.0), y, y);
}

struct WeightCands {
  int idx[WC];     // wave-uniform atom, -1: none
  bool act[WC];    // the cell function of this lane's point can be nonzero
  double r[WC];    // this lane's distance
};

// The next WC candidates from atom `next` on (at least one lane within 5 bohr of
// its nearest atom's distance, or any lane without the cap); false when none is
// left.
__device__ __forceinline__ bool next_cands(WeightCands &c, int &next, int natoms,
                                           const double *__restrict__ C, double x, double y,
                                           double z, double rmin, bool cap, bool on) {
  int n = 0;
#pragma unroll
  for (int k = 0; k < WC; ++k) {
    c.idx[k] = -1;
    c.act[k] = false;
    c.r[k] = 1.0;
  }
  for (; next < natoms && n < WC; ++next) {
    const double r = gdist(x, y, z, C + 3 * next);
    const bool a = on && !(cap && r - rmin >= 5.0);
    if (!__ballot(a)) continue;
#pragma unroll
    for (int k = 0; k < WC; ++k)
      if (k == n) {
        c.idx[k] = next;
        c.act[k] = a;
        c.r[k] = r;
      }
    ++n;
  }
  return n > 0;
}

// Becke cell functions P of the candidates at this lane's point.
__device__ __forceinline__ void cand_cells(const WeightCands &c, int natoms,
                                           const double *__restrict__ C,
                                           const double2 *__restrict__ tab, double x, double y,
                                           double z, bool cap, double (&P)[WC]) {
  double rmax = 0.0;
#pragma unroll
  for (int k = 0; k < WC; ++k) {
    P[k] = c.act[k] ? 1.0 : 0.0;
    if (c.act[k]) rmax = fmax(rmax, c.r[k]);
  }
  for (int j = 0; j < natoms; ++j) {
    const double rj = gdist(x, y, z, C + 3 * j);
    if (cap && !__ballot(rmax - rj > -5.0)) continue;  // every factor is 1
#pragma unroll
    for (int k = 0; k < WC; ++k) {
      if (c.idx[k] < 0 || c.idx[k] == j) continue;  // uniform
      const double mu =
          fmin(fmax((c.r[k] - rj) * tab[c.idx[k] * natoms + j].x, -1.0), 1.0);
      P[k] *= 0.5 * (1.0 - bp(bp(bp(mu))));
    }
  }
}

__global__ void __launch_bounds__(64) grad_weights_kernel(
    int64_t npts_pad, int natoms, const double *__restrict__ C, const double *__restrict__ px,
    const double *__restrict__ py, const double *__restrict__ pz, const int *__restrict__ pown,
    const double *__restrict__ epoint, const double *__restrict__ tpt, int partition,
    const double2 *__restrict__ ptab, double *__restrict__ wpart) {
  extern __shared__ double acc[];
  __shared__ double Pk[WKEEP * WC * 64];
  for (int e = threadIdx.x; e < 3 * natoms; e += blockDim.x) acc[e] = 0.0;
  __syncthreads();
  const bool cap = partition == 1;
  const int lane = threadIdx.x & 63;
  for (int64_t sp = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; sp < npts_pad;
       sp += (int64_t)gridDim.x * blockDim.x) {
    const int B = pown[sp];
    const bool act = B >= 0 && B < natoms;  // not padding
    double S[3] = {0.0, 0.0, 0.0};          // the owner receives -S
    double x = 0.0, y = 0.0, z = 0.0, wf = 0.0, rmin = 1e300, Z = 0.0, PB = 0.0;
    if (act) {
      for (int k = 0; k < 3; ++k) S[k] = -tpt[3 * sp + k];
      wf = epoint[sp];
      x = px[sp];
      y = py[sp];
      z = pz[sp];
    }
    const bool wact = act && partition != 0 && wf != 0.0;
    if (__ballot(wact)) {
      if (cap)
        for (int i = 0; i < natoms; ++i) rmin = fmin(rmin, gdist(x, y, z, C + 3 * i));
      WeightCands c;
      int g = 0;
      for (int next = 0; next_cands(c, next, natoms, C, x, y, z, rmin, cap, wact); ++g) {
        double P[WC];
        cand_cells(c, natoms, C, ptab, x, y, z, cap, P);
#pragma unroll
        for (int k = 0; k < WC; ++k) {
          if (g < WKEEP) Pk[(g * WC + k) * 64 + lane] = P[k];
          Z += P[k];
          if (c.idx[k] == B) PB = P[k];
        }
      }
    }
    const bool gact = wact && PB > 0.0 && Z > 0.0;
    if (__ballot(gact)) {
      const double iPB = gact ? 1.0 / PB : 0.0, iZ = gact ? 1.0 / Z : 0.0;
      WeightCands c;
      int g = 0;
      for (int next = 0; next_cands(c, next, natoms, C, x, y, z, rmin, cap, wact); ++g) {
        double P[WC];
        if (g < WKEEP) {
#pragma unroll
          for (int k = 0; k < WC; ++k) P[k] = Pk[(g * WC + k) * 64 + lane];
        } else {
          cand_cells(c, natoms, C, ptab, x, y, z, cap, P);
        }
        double coef[WC], ui[WC][3], gi[WC][3];
#pragma unroll
        for (int k = 0; k < WC; ++k) {
          coef[k] = gact && P[k] != 0.0 ? wf * ((c.idx[k] == B ? iPB : 0.0) - iZ) * P[k] : 0.0;
          const double *Ci = C + 3 * max(c.idx[k], 0);
          const double iri = c.r[k] > 0.0 ? 1.0 / c.r[k] : 0.0;  // 0: on the nucleus
          ui[k][0] = (x - Ci[0]) * iri;
          ui[k][1] = (y - Ci[1]) * iri;
          ui[k][2] = (z - Ci[2]) * iri;
          gi[k][0] = gi[k][1] = gi[k][2] = 0.0;
        }
        for (int j = 0; j < natoms; ++j) {
          const double *Cj = C + 3 * j;
          const double dj[3] = {x - Cj[0], y - Cj[1], z - Cj[2]};
          const double rj = gdist(x, y, z, Cj);
          double mu[WC];
          bool in[WC], any = false;
#pragma unroll
          for (int k = 0; k < WC; ++k) {
            mu[k] = c.idx[k] >= 0 ? (c.r[k] - rj) * ptab[c.idx[k] * natoms + j].x : 1.0;
            in[k] = c.idx[k] != j && coef[k] != 0.0 && mu[k] > -1.0 && mu[k] < 1.0;
            any = any || in[k];
          }
          if (!__ballot(any)) continue;
          const double irj = rj > 0.0 ? 1.0 / rj : 0.0;
          double a = 0.0, gj[3] = {0.0, 0.0, 0.0};
#pragma unroll
          for (int k = 0; k < WC; ++k) {
            if (c.idx[k] < 0 || c.idx[k] == j || !__ballot(in[k])) continue;  // uniform
            const double *Ci = C + 3 * c.idx[k];
            const double2 tij = ptab[c.idx[k] * natoms + j];  // 1/R~, [not capped] / R^2
            const double m = mu[k], p1 = bp(m), p2 = bp(p1), p3 = bp(p2);
            const double sv = 0.5 * (1.0 - p3);  // > 0 because P_i > 0
            const double ds = -0.5 * bdp(p2) * bdp(p1) * bdp(m);
            const double f = in[k] ? coef[k] * ds * recip(sv) : 0.0;
            const double fr = f * tij.x, ft = in[k] ? f * m * tij.y : 0.0;
            a += fr;
#pragma unroll
            for (int t = 0; t < 3; ++t) {
              const double e = ft * (Ci[t] - Cj[t]);
              gi[k][t] -= fr * ui[k][t] + e;
              gj[t] += e;
            }
          }
          const bool mine = j == B;
#pragma unroll
          for (int t = 0; t < 3; ++t) {
            const double g = mine ? 0.0 : gj[t] + a * (dj[t] * irj);
            S[t] += g;
            const double v = wave_sum(g);
            if (lane == 0) acc[3 * j + t] += v;
          }
        }
#pragma unroll
        for (int k = 0; k < WC; ++k) {
          if (c.idx[k] < 0) continue;  // uniform
#pragma unroll
          for (int t = 0; t < 3; ++t) {
            const double g = c.idx[k] != B ? gi[k][t] : 0.0;
            S[t] += g;
            const double v = wave_sum(g);
            if (lane == 0) acc[3 * c.idx[k] + t] += v;
          }
        }
      }
    }
    // owner terms, one wave sum per distinct owner among the wave's points
    unsigned long long pend = __ballot(act);
    while (pend) {
      const int src = __ffsll((long long)pend) - 1;
      const int Bs = __shfl(B, src);
      const bool mine = act && B == Bs;
      for (int k = 0; k < 3; ++k) {
        const double v = wave_sum(mine ? -S[k] : 0.0);
        if (lane == 0) acc[3 * Bs + k] += v;
      }
      pend &= ~__ballot(mine);
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 3 * natoms; e += blockDim.x)
    wpart[(int64_t)blockIdx.x * 3 * natoms + e] = acc[e];
}

// out[k] = sum over the rows of in[r][k]; one workgroup per column.  Thread t
// sums the rows r = t (mod 256) in ascending order, then a fixed tree in LDS
// adds the 256 partial sums, so the order of the additions is the same on
// every run.
__global__ void __launch_bounds__(256) colsum_kernel(int nrow, int ncol,
                                                     const double *__restrict__ in,
                                                     double *__restrict__ out) {
  __shared__ double part[256];
  const int k = blockIdx.x, t = threadIdx.x;
  double v = 0.0;
  for (int r = t; r < nrow; r += 256) v += in[(int64_t)r * ncol + k];
  part[t] = v;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (t < h) part[t] += part[t + h];
    __syncthreads();
  }
  if (t == 0) out[k] = part[0];
}

// ---------------------------------------------------------------------------
void vkg_basis(hipStream_t s, int64_t b0, int64_t b1, int64_t s0, const Plan &pl,
               const double *Pt, int narr, int yarr, int gga, const double *tiles,
               const double *coef, bool accum, double *cpart, double *tpart, double *tpt) {
  if (b1 <= b0) return;
  const int nmg = std::max(1, (pl.max_live + 1) / 2);  // of the fullest batch
  const int64_t step = max_workgroups(256) / (8 * nmg) * 8;  // batches of a launch
  for (int64_t b = b0; b < b1; b += step) {
    const int64_t be = std::min(b + step, b1), nwg = (be - b + 7) / 8 * 8 * nmg;
    hipLaunchKernelGGL(grad_basis_f64, dim3((unsigned)nwg), dim3(256), 0, s, pl.tab(), Pt,
                       pl.b_off.p, pl.b_fbl.p, s0, b, be, nmg, narr, yarr, gga, tiles, coef,
                       pl.funcs.p, pl.terms.p, pl.px.p, pl.py.p, pl.pz.p, cpart, tpart);
    NKX_HIP_CHECK(hipGetLastError());
  }
  hipLaunchKernelGGL(grad_points_kernel, dim3((unsigned)(b1 - b0)), dim3(192), 0, s, s0, b0,
                     pl.b_off.p, tpart, accum ? 1 : 0, tpt);
  NKX_HIP_CHECK(hipGetLastError());
}

void vkg_fold(hipStream_t s, int64_t b0, int64_t b1, int64_t s0, const Plan &pl, int nseg,
              const double *cpart, double *gacc) {
  if (b1 <= b0) return;
  hipLaunchKernelGGL(grad_fold_kernel, dim3((unsigned)pl.nfb, (unsigned)nseg), dim3(256), 0, s,
                     pl.nb, b0, b1, s0, nseg, pl.nbf_pad, pl.tile_slot.p, cpart, gacc);
  NKX_HIP_CHECK(hipGetLastError());
}

void vkg_owners(hipStream_t s, const Plan &pl, const int *owner, int *pown) {
  const int64_t n = pl.npts_pad;
  hipLaunchKernelGGL(owners_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n,
                     pl.pidx.p, owner, pown);
  NKX_HIP_CHECK(hipGetLastError());
}

void vkg_weights(hipStream_t s, const Plan &pl, int natoms, const double *centers,
                 const int *pown, const double *epoint, const double *tpt, int partition,
                 int nblk, double *ptab, double *wpart) {
  double2 *tab = reinterpret_cast<double2 *>(ptab);
  const int npair = natoms * natoms;
  hipLaunchKernelGGL(pair_table_kernel, dim3((unsigned)((npair + 255) / 256)), dim3(256), 0, s,
                     natoms, centers, partition == 1 ? 1 : 0, tab);
  NKX_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(grad_weights_kernel, dim3((unsigned)nblk), dim3(64),
                     (size_t)3 * natoms * sizeof(double), s, pl.npts_pad, natoms, centers,
                     pl.px.p, pl.py.p, pl.pz.p, pown, epoint, tpt, partition, tab, wpart);
  NKX_HIP_CHECK(hipGetLastError());
}

void vkg_colsum(hipStream_t s, int nrow, int ncol, const double *in, double *out) {
  if (ncol <= 0) return;
  hipLaunchKernelGGL(colsum_kernel, dim3((unsigned)ncol), dim3(256), 0, s, nrow, ncol, in, out);
  NKX_HIP_CHECK(hipGetLastError());
}

}  // namespace nkx
