// Epilogue of the basis-centre gradient, both forms: from X = P Phi and W = P Y
// of a few functions at a wave's 64 points,
//   c_mu(g) = -2 [ d phi_mu(g) W_mu(g) + (H_mu(g) b_g) X_mu(g) ]
// summed over the points per function and over the functions per point.
#pragma once

#include "lane_sums.hpp"
#include "nkx_internal.hpp"
#include "sto_run.hpp"

namespace nkx {

constexpr int GR_LD = 64;  // row length of the X and W tiles in LDS

struct GradPoint {
  double x, y, z, bx, by, bz;
};

// S, grad S and (Hessian of S) b from a monomial list (l > 2), added to.
__device__ __forceinline__ void harm_hess(int off, int cnt, const HarmTerm *__restrict__ T,
                                          const double (&d)[3], const double (&b)[3], double &S,
                                          double (&Sg)[3], double (&Sb)[3]) {
#pragma unroll 1
  for (int t = off; t < off + cnt; ++t) {
    const HarmTerm h = T[t];
    const double xa1 = ipow(d[0], h.a > 0 ? h.a - 1 : 0);
    const double yb1 = ipow(d[1], h.b > 0 ? h.b - 1 : 0);
    const double zc1 = ipow(d[2], h.c > 0 ? h.c - 1 : 0);
    const double xa = h.a > 0 ? xa1 * d[0] : 1.0;
    const double yb = h.b > 0 ? yb1 * d[1] : 1.0;
    const double zc = h.c > 0 ? zc1 * d[2] : 1.0;
    const double ca = h.coef * xa, cxa1 = h.coef * h.a * xa1;
    S += ca * yb * zc;
    if (h.a > 0) Sg[0] += cxa1 * yb * zc;
    if (h.b > 0) Sg[1] += ca * (h.b * yb1) * zc;
    if (h.c > 0) Sg[2] += ca * yb * (h.c * zc1);
    if (h.a > 1) Sb[0] += h.coef * (h.a * (h.a - 1)) * ipow(d[0], h.a - 2) * yb * zc * b[0];
    if (h.b > 1) Sb[1] += ca * (h.b * (h.b - 1)) * ipow(d[1], h.b - 2) * zc * b[1];
    if (h.c > 1) Sb[2] += ca * yb * (h.c * (h.c - 1)) * ipow(d[2], h.c - 2) * b[2];
    if (h.a > 0 && h.b > 0) {
      const double s = cxa1 * (h.b * yb1) * zc;
      Sb[0] += s * b[1];
      Sb[1] += s * b[0];
    }
    if (h.a > 0 && h.c > 0) {
      const double s = cxa1 * yb * (h.c * zc1);
      Sb[0] += s * b[2];
      Sb[2] += s * b[0];
    }
    if (h.b > 0 && h.c > 0) {
      const double s = ca * (h.b * yb1) * (h.c * zc1);
      Sb[1] += s * b[2];
      Sb[2] += s * b[1];
    }
  }
}

// The records of 16 functions, lane l holding function l mod 16.
struct GradFuncs {
  FuncRec rec;
  __device__ __forceinline__ void load(const FuncRec *fr, int lane) {
    rec = fr[lane & 15];
  }
};

// Functions l0 .. l0 + NF - 1 of gf at this lane's point; X and W of function i at
// Xs[i GR_LD + lane], Ws[...].  cp[3 i + k]: sums over the 64 points; tp: this
// point's sums, added to.  The sums of a run of functions on one centre are
// written at the run's first function, the others get zero (only the sums per
// atom are used).  A wave takes one function at a time: its record comes
// out of the lane that holds it into scalar registers, the branches on it are
// scalar branches.  Functions are sorted by centre, so runs of
// them share dx, dy, dz, r and 1/r, and those with the same zeta, k and
// normalisation the radial factor and its derivatives.
//
// Bound by FP64 VALU issue: 1.5 of the 3.3 ms of the mixed basis-centre kernel
// on 30 atoms, 0.25 ms for the whole FP64 one on 8 atoms.  With the (function,
// point) pairs in the MFMA result layout a wave held four functions at a time,
// each lane loading its own record and evaluating a whole Hessian: 3.1 of 4.8
// ms, and 0.89 ms.
template <int NF>
__device__ __forceinline__ void grad_rows(const GradFuncs &gf, int l0, const HarmTerm *__restrict__ T,
                                          const GradPoint &p, int gga, const double *Xs,
                                          const double *Ws, int lane, double *__restrict__ cp,
                                          double (&tp)[3]) {
  double mine = 0.0;         // lane 3 i + k: what goes to cp[3 i + k]
  double run[3] = {0.0, 0.0, 0.0};
  int first = 0;             // of the current run
  StoRun st;
  double xb = 0.0, A = 0.0;  // d . b; (R'' - R' / r) / r^2
  const double b[3] = {p.bx, p.by, p.bz};
  double pcx = 0.0, pcy = 0.0, pcz = 0.0, pzeta = 0.0, pnorm = 0.0;  // the one before
  int pk = 0;
  auto flush = [&](int f) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double t = wave_sum(run[k]);
      if (lane == 3 * f + k) mine = t;
      run[k] = 0.0;
    }
  };
#pragma unroll 1  // the body is long: one copy stays in the instruction cache
  for (int i = 0; i < NF; ++i) {
    const double norm = lane_double(gf.rec.norm, l0 + i);
    if (norm != 0.0) {  // else a padding function
      const double cx = lane_double(gf.rec.cx, l0 + i), cy = lane_double(gf.rec.cy, l0 + i),
                   cz = lane_double(gf.rec.cz, l0 + i), zeta = lane_double(gf.rec.zeta, l0 + i);
      const int k0 = lane_int(gf.rec.k, l0 + i);
      const bool newc = pnorm == 0.0 || cx != pcx || cy != pcy || cz != pcz;
      if (newc) {
        if (i > 0) {
          flush(first);
          first = i;
        }
        st.centre(p.x - cx, p.y - cy, p.z - cz);
        xb = st.d[0] * b[0] + st.d[1] * b[1] + st.d[2] * b[2];
      }
      if (newc || zeta != pzeta || k0 != pk || norm != pnorm) {
        st.shell<false>(k0, zeta, norm);
        const double q = fma((double)k0, st.ir, -zeta), ir2 = st.ir * st.ir;
        A = ((q * q - k0 * ir2) * st.R - st.C) * ir2;
      }
      pnorm = norm;
      pcx = cx;
      pcy = cy;
      pcz = cz;
      pzeta = zeta;
      pk = k0;
      // S, grad S and (Hessian of S) b of the solid harmonic
      const double (&d)[3] = st.d;
      const double R = st.R, R1r = st.C;
      double S, Sg[3], Sb[3] = {0.0, 0.0, 0.0};
      const int type = lane_int(gf.rec.type, l0 + i);
      if (type >= 0) {
        st.harmonic<true>(type, 0, 0, T, S, Sg);
        switch (type) {  // (l < 2: none)
          case 4: Sb[0] = kS2 * b[1], Sb[1] = kS2 * b[0]; break;
          case 5: Sb[1] = kS2 * b[2], Sb[2] = kS2 * b[1]; break;
          case 6:
            Sb[0] = -2.0 * kS20 * b[0], Sb[1] = -2.0 * kS20 * b[1], Sb[2] = 4.0 * kS20 * b[2];
            break;
          case 7: Sb[0] = kS2 * b[2], Sb[2] = kS2 * b[0]; break;
          case 8: Sb[0] = 2.0 * kS22 * b[0], Sb[1] = -2.0 * kS22 * b[1]; break;
          default: break;
        }
      } else {
        S = Sg[0] = Sg[1] = Sg[2] = 0.0;
        harm_hess(lane_int(gf.rec.term_off, l0 + i), lane_int(gf.rec.term_cnt, l0 + i), T, d, b, S, Sg, Sb);
      }
      const double w = -2.0 * Ws[i * GR_LD + lane], SR = S * R1r;
      if (gga) {
        const double x = -2.0 * Xs[i * GR_LD + lane];
        const double sgb = R1r * (Sg[0] * b[0] + Sg[1] * b[1] + Sg[2] * b[2]) + S * A * xb;
        const double rxb = R1r * xb;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const double g = R * Sg[k] + SR * d[k];
          const double hb = R * Sb[k] + sgb * d[k] + rxb * Sg[k] + SR * b[k];
          const double c = g * w + hb * x;
          run[k] += c;
          tp[k] += c;
        }
      } else {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const double c = (R * Sg[k] + SR * d[k]) * w;
          run[k] += c;
          tp[k] += c;
        }
      }
    }
  }
  flush(first);
  if (lane < 3 * NF) cp[lane] = mine;
}

}  // namespace nkx
