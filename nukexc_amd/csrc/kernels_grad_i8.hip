// Nuclear gradient of E_xc at fixed P, mixed form: the two contractions of the
// basis-centre term, X = P Phi and W = P Y, run on int8 slices with exact
// integer MFMA accumulation (the slice form of the V_xc build); the
// functional, the STO derivatives of the epilogue and every sum are FP64.
// The terms and their derivation are those of the FP64 form
// (kernels_grad.hip):
//   c_mu(g) = -2 [ d phi_mu(g) W_mu(g) + (H_mu(g) b_g) X_mu(g) ],
//   Y_nu(g) = w v_rho phi_nu + b_g . grad phi_nu = 2 a_g phi_nu + b_g . grad phi_nu,
// with (a, b) the per-point coefficients of the density stage.  The
// point-motion and Becke weight terms reuse the FP64 kernels unchanged.
//
// Per live slot the store holds the V build's sections; the gradient uses Pm
// (Phi, rows = points, k = functions) and writes Y in the same orientation
// into the Z section, so both are B operands of P[mu][nu] with per-point
// exponents.
#include "grad_rows.hpp"
#include "nkx_internal.hpp"
#include "slices_i8.hpp"
#include "vxc_kernels.hpp"

namespace nkx {

namespace {
constexpr int GC = FB * 3;  // per-slot partial: 64 functions x 3 components
}  // namespace

// Y slices of one live slot, written at yout + (slot - s0) ystride (the
// slot's Z section, or a separate array for the second spin); one workgroup
// per slot.  Thread t owns fragment item t: point 16 (t / 64) + t % 16,
// functions 16 ((t % 64) / 16) .. +15.
// Phi comes from the Pm slices (per-point exponent), grad Phi from the FP32
// planes; the row maximum over the four threads of a point by shuffles.
__global__ void __launch_bounds__(256) y_slots_i8(int64_t s0, const int *__restrict__ slot_b,
                                                  int gga, const double *__restrict__ coef,
                                                  signed char *__restrict__ store,
                                                  signed char *__restrict__ yout,
                                                  int64_t ystride) {
  const int64_t sl = s0 + blockIdx.x;
  const int64_t b = slot_b[sl];
  signed char *tb = store + (int64_t)blockIdx.x * slot_bytes_i8(gga);
  const int t = threadIdx.x, l = t & 63;
  const int g = 16 * (t >> 6) + (l & 15), k0 = 16 * (l >> 4);
  const int64_t gp = b * PT + g;
  const double a2 = 2.0 * coef[4 * gp], bx = coef[4 * gp + 1], by = coef[4 * gp + 2],
               bz = coef[4 * gp + 3];
  v4i fp[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) fp[p] = ld16(tb + OFF_PM + p * PLANE + t * 16);
  const int eP = tb[OFF_PM + 4 * PLANE + g];
  // every load is issued before the first use (a branch between them would
  // make each wait for the one before)
  const float *G = reinterpret_cast<const float *>(tb + OFF_G);
  float gv[3][16];
  if (gga) {
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e) gv[c][e] = G[c * TILE + (k0 + e) * PT + g];
  } else {
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e) gv[c][e] = 0.0f;
  }
  const double sP = unslice_scale(eP);
  double y[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const double ph = (double)unslice_int(fp, e) * sP;
    y[e] = gga ? z_value(ph, (double)gv[0][e], (double)gv[1][e], (double)gv[2][e], a2, bx, by, bz)
               : a2 * ph;
  }
  const int ey = item_row_exp(y);
  store_item(y, ey, yout + (int64_t)blockIdx.x * ystride);
}

// One workgroup (four waves) per batch.  For each live block I of the batch,
// X and W accumulate over the live blocks K: wave w takes rows 16 w .. +15 of
// I (its P fragment of pair (I, K) in registers), every point of the batch
// (four 16-point fragments of the K slot's Pm and Y sections), the ten slice
// products per tile and an FP64 combine per K.  The steps (I, K) run in that
// order; the K slot's Pm and Y sections are copied into LDS once per step for
// the four waves (two buffers: the next step's copies are issued while the
// current step computes; a second register set for the P fragments would
// cost the occupancy).  The epilogue, after the last K of an I, is the FP64
// form's (grad_rows.hpp): per-function sums over the batch's points into cpart,
// per-point sums over functions into tpt (with the sign of the point-motion
// term).
__global__ void __launch_bounds__(256, 2) grad_basis_i8(
    MolTab mt, const signed char *__restrict__ Ps, const int *__restrict__ b_off,
    const int *__restrict__ b_fbl, int64_t s0, int64_t b0, int gga,
    const signed char *__restrict__ store, const double *__restrict__ coef,
    const FuncRec *__restrict__ F, const HarmTerm *__restrict__ T,
    const double *__restrict__ px, const double *__restrict__ py,
    const double *__restrict__ pz, const signed char *__restrict__ ybase, int64_t ystride,
    int accum, double *__restrict__ cpart, double *__restrict__ tpt) {
  const int b = (int)(b0 + blockIdx.x);
  const int lo = b_off[b], hi = b_off[b + 1];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, q = lane >> 4;
  const int64_t sb_bytes = slot_bytes_i8(gga);

  // Pm and Y sections of a step's K slot, two buffers, declared apart so that
  // a copy into one is known not to touch the other
  __shared__ __attribute__((aligned(16))) signed char bufA[2][SEC];
  __shared__ __attribute__((aligned(16))) signed char bufB[2][SEC];
  __shared__ int lbl[MAXNFB];  // local block index of the batch's live blocks
  __shared__ double red[4][3][PT];
  // the epilogue's points (coordinates, b), kept in LDS for their registers
  __shared__ double pts[6][PT];
  for (int e = threadIdx.x; e < 6 * PT; e += 256) {
    const int c = e / PT, g = e % PT;
    const int64_t gp = (int64_t)b * PT + g;
    pts[c][g] = c == 0 ? px[gp] : c == 1 ? py[gp] : c == 2 ? pz[gp] : coef[4 * gp + c - 2];
  }
  // this lane's point: sums over this wave's functions
  double tp[3] = {0.0, 0.0, 0.0};
  const int n = hi - lo;
  for (int k = threadIdx.x; k < n; k += 256) lbl[k] = mt.blk_local[b_fbl[lo + k]];
  __syncthreads();
  if (n > 0) {
    // the batch's blocks are blocks of one molecule
    const int mol = mt.blk_mol[b_fbl[lo]];
    const signed char *pbase = Ps + mt.Ps_off[mol];
    const int nfbm = mt.nfb[mol];
    // the K slot's sections of a step -> LDS buffer dst (direct copies)
    auto issue = [&](int st, signed char (*dst)[SEC]) {
      const int64_t sk = lo + st % n - s0;
      dma_section<4>(store + sk * sb_bytes + OFF_PM, &dst[0][0], wv, lane);
      dma_section<4>(ybase + sk * ystride, &dst[1][0], (wv + 2) & 3, lane);
    };
    double X[4][4], W[4][4];
    // Epilogue of block I = b_fbl[mi] through the two LDS buffers (X and W of
    // 64 rows fit them): wave w takes 16 functions, a point per lane.
    // X and W leave the registers, which the epilogue needs; the next block's
    // first copies wait for its end (the other workgroup of the CU runs
    // meanwhile).  Result register r of lane l holds row 4 (l / 16) + r, point
    // l % 16 of a tile.
    auto epilogue = [&](int mi) {
      GradFuncs gf;
      gf.load(F + (int64_t)__builtin_amdgcn_readfirstlane(b_fbl[mi]) * FB + 16 * wv, lane);
      double *Xs = reinterpret_cast<double *>(&bufA[0][0]);
      double *Ws = reinterpret_cast<double *>(&bufB[0][0]);
      static_assert(sizeof(bufA) >= FB * GR_LD * sizeof(double), "X of a block in a buffer");
      __syncthreads();  // the buffers' readers are done
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          Xs[(16 * wv + 4 * q + r) * GR_LD + 16 * j + l16] = X[j][r];
          Ws[(16 * wv + 4 * q + r) * GR_LD + 16 * j + l16] = W[j][r];
        }
      wave_fence();  // the rows of a wave are the functions that it takes: no barrier
      const GradPoint pt{pts[0][lane], pts[1][lane], pts[2][lane],
                         pts[3][lane], pts[4][lane], pts[5][lane]};
      grad_rows<16>(gf, 0, T, pt, gga, Xs + 16 * wv * GR_LD, Ws + 16 * wv * GR_LD, lane,
                cpart + (mi - s0) * GC + 48 * wv, tp);
      __syncthreads();  // the buffers are free
    };
    auto products = [&](signed char (*cur)[SEC], const v4i (&Ac)[4], int eAc) {
      double sA[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) sA[r] = pow2_or_zero((int)(signed char)(eAc >> (8 * r)));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int op = 0; op < 2; ++op) {
          const signed char *sec = &cur[op][0];
          v4i B[4];
#pragma unroll
          for (int p = 0; p < 4; ++p) B[p] = ld16(sec + p * PLANE + (j * 64 + lane) * 16);
          const int eB = sec[4 * PLANE + 16 * j + l16];
          const double sB = eB == -127 ? 0.0 : pow2(eB - 19);
          int hi4[4], lo4[4];
          tile_product(Ac, B, hi4, lo4);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const double v = fma((double)lo4[r], 0x1p-14, (double)hi4[r]) * (sA[r] * sB);
            if (op)
              W[j][r] += v;
            else
              X[j][r] += v;
          }
        }
      }
    };
    // one step (I, K): its P fragment, wait for its sections, issue the next
    // step's copies (within a block), then the tile products.  (One loop over
    // all steps: as nested loops their addresses become induction variables
    // that cost 80 registers.)
    auto step = [&](int st, signed char (*cur)[SEC], signed char (*nxt)[SEC]) {
      const int ii = st / n, kk = st - ii * n;
      const signed char *pa =
          pbase + ((int64_t)__builtin_amdgcn_readfirstlane(lbl[ii]) * nfbm +
                   __builtin_amdgcn_readfirstlane(lbl[kk])) * SEC;
      v4i A[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) A[p] = ld16(pa + p * PLANE + (wv * 64 + lane) * 16);
      const int eA = *reinterpret_cast<const int *>(pa + 4 * PLANE + 16 * wv + 4 * q);
      wait_vm0();
      __syncthreads();  // buffer cur complete, nxt free
      if (kk + 1 < n) issue(st + 1, nxt);
      products(cur, A, eA);
    };
    const int nsteps = n * n;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) X[j][r] = W[j][r] = 0.0;
    issue(0, bufA);
    for (int st = 0; st < nsteps; ++st) {
      if (st & 1)
        step(st, bufB, bufA);
      else
        step(st, bufA, bufB);
      if ((st + 1) % n == 0) {  // uniform: the last K of block I
        epilogue(lo + st / n);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) X[j][r] = W[j][r] = 0.0;
        if (st + 1 < nsteps) {
          if (st & 1)
            issue(st + 1, bufA);
          else
            issue(st + 1, bufB);
        }
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; ++k) red[wv][k][lane] = tp[k];
  __syncthreads();
  if (threadIdx.x < 3 * PT) {
    const int k = threadIdx.x / PT, g = threadIdx.x % PT;
    const int64_t e = 3 * ((int64_t)b * PT + g) + k;
    const double t = ((red[0][k][g] + red[1][k][g]) + red[2][k][g]) + red[3][k][g];
    tpt[e] = (accum ? tpt[e] : 0.0) - t;
  }
}

// ---------------------------------------------------------------------------
void vkgm_y_slots(hipStream_t s, int64_t s0, int64_t s1, const Plan &pl, int gga,
                  const double *coef, signed char *store, signed char *ystore_b) {
  if (s1 <= s0) return;
  signed char *yout = ystore_b ? ystore_b : store + OFF_Z;
  const int64_t ystride = ystore_b ? (int64_t)SEC : slot_bytes_i8(gga);
  hipLaunchKernelGGL(y_slots_i8, dim3((unsigned)(s1 - s0)), dim3(256), 0, s, s0, pl.slot_b.p,
                     gga, coef, store, yout, ystride);
  NKX_HIP_CHECK(hipGetLastError());
}

void vkgm_basis(hipStream_t s, int64_t b0, int64_t b1, int64_t s0, const Plan &pl,
                const signed char *Ps, int gga, const signed char *store, const double *coef,
                const signed char *ystore_b, bool accum, double *cpart, double *tpt) {
  if (b1 <= b0) return;
  const signed char *ybase = ystore_b ? ystore_b : store + OFF_Z;
  const int64_t ystride = ystore_b ? (int64_t)SEC : slot_bytes_i8(gga);
  hipLaunchKernelGGL(grad_basis_i8, dim3((unsigned)(b1 - b0)), dim3(256), 0, s, pl.tab(), Ps,
                     pl.b_off.p, pl.b_fbl.p, s0, b0, gga, store, coef, pl.funcs.p, pl.terms.p,
                     pl.px.p, pl.py.p, pl.pz.p, ybase, ystride, accum ? 1 : 0, cpart, tpt);
  NKX_HIP_CHECK(hipGetLastError());
}

}  // namespace nkx
