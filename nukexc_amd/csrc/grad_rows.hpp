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

// The records of 16 functions, lane l holding function l mod 16, and a bit per
// function: nonzero norm; centre other than the one before's; shell (centre,
// zeta, k, norm) other than the one before's.  The first function and one after a
// padding function (norm zero, skipped) count as other in both.
struct GradFuncs {
  FuncRec rec;
  unsigned live, newc, newsh;
  __device__ __forceinline__ void load(const FuncRec *fr, int lane) {
    const int i = lane & 15;
    rec = fr[i];
    const FuncRec prev = fr[i ? i - 1 : 0];
    const bool c = i == 0 || prev.norm == 0.0 || rec.cx != prev.cx || rec.cy != prev.cy ||
                   rec.cz != prev.cz;
    live = (unsigned)__ballot(rec.norm != 0.0) & 0xffffu;
    newc = (unsigned)__ballot(c) & 0xffffu;
    newsh = (unsigned)__ballot(c || rec.zeta != prev.zeta || rec.k != prev.k ||
                               rec.norm != prev.norm) &
            0xffffu;
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
// With S the harmonic, R the radial factor, C = R' / r and A = (R'' - C) / r^2,
//   c = -2 [ (R W + C (d.b) X) grad S + R X (Hess S) b + beta d + delta b ],
//   delta = C S X,  beta = C S W + (C (grad S . b) + A S (d.b)) X:
// beta and delta are summed over a run and multiplied by d and b once, and the
// vector part costs only what the harmonic has: nothing for s, one FMA for p.
//
// Bound by FP64 VALU issue: 1.0 of the 2.75 ms of the mixed basis-centre kernel
// on 30 atoms, 0.22 ms for the whole FP64 one on 8 atoms.  With gradient and
// Hessian formed per function (and the records of both neighbours compared as
// doubles) 1.45 of 3.2 ms and 0.25 ms; with the (function, point) pairs in the
// MFMA result layout, each lane loading its own record, 3.1 of 4.8 ms and 0.89.
template <int NF>
__device__ __forceinline__ void grad_rows(const GradFuncs &gf, int l0, const HarmTerm *__restrict__ T,
                                          const GradPoint &p, int gga, const double *Xs,
                                          const double *Ws, int lane, double *__restrict__ cp,
                                          double (&tp)[3]) {
  double mine = 0.0;         // lane 3 i + k: what goes to cp[3 i + k]
  double v[3] = {0.0, 0.0, 0.0}, beta = 0.0, delta = 0.0;  // of the current run
  int first = 0;             // of the current run
  StoRun st;
  st.d[0] = st.d[1] = st.d[2] = st.R = st.C = 0.0;
  double xb = 0.0, Axb = 0.0, rxb = 0.0;  // d . b; A xb; C xb
  const double b[3] = {gga ? p.bx : 0.0, gga ? p.by : 0.0, gga ? p.bz : 0.0};
  auto flush = [&](int f) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double c = -2.0 * fma(beta, st.d[k], fma(delta, b[k], v[k]));
      tp[k] += c;
      const double t = wave_sum(c);
      if (lane == 3 * f + k) mine = t;
      v[k] = 0.0;
    }
    beta = delta = 0.0;
  };
  const unsigned live = gf.live >> l0, newc = gf.newc >> l0, newsh = gf.newsh >> l0;
#pragma unroll 1  // the body is long: one copy stays in the instruction cache
  for (int i = 0; i < NF; ++i) {
    if ((live >> i) & 1u) {  // else a padding function
      if (i == 0 || ((newsh >> i) & 1u)) {
        if (i == 0 || ((newc >> i) & 1u)) {
          if (i > 0) {
            flush(first);
            first = i;
          }
          st.centre(p.x - lane_double(gf.rec.cx, l0 + i), p.y - lane_double(gf.rec.cy, l0 + i),
                    p.z - lane_double(gf.rec.cz, l0 + i));
          xb = st.d[0] * b[0] + st.d[1] * b[1] + st.d[2] * b[2];
        }
        const double zeta = lane_double(gf.rec.zeta, l0 + i);
        const int k0 = lane_int(gf.rec.k, l0 + i);
        st.shell<false>(k0, zeta, lane_double(gf.rec.norm, l0 + i));
        const double q = fma((double)k0, st.ir, -zeta), ir2 = st.ir * st.ir;
        Axb = ((q * q - k0 * ir2) * st.R - st.C) * ir2 * xb;
        rxb = st.C * xb;
      }
      const double w = Ws[i * GR_LD + lane], x = gga ? Xs[i * GR_LD + lane] : 0.0;
      const double al = fma(rxb, x, st.R * w), ga = st.R * x;
      const double(&d)[3] = st.d;
      double S, sb;  // the harmonic, grad S . b
      const int type = lane_int(gf.rec.type, l0 + i);
      switch (type) {
        case 0:
          S = kS0;
          sb = 0.0;
          break;
        case 1:
          S = kS1 * d[1];
          sb = kS1 * b[1];
          v[1] = fma(kS1, al, v[1]);
          break;
        case 2:
          S = kS1 * d[2];
          sb = kS1 * b[2];
          v[2] = fma(kS1, al, v[2]);
          break;
        case 3:
          S = kS1 * d[0];
          sb = kS1 * b[0];
          v[0] = fma(kS1, al, v[0]);
          break;
        case 4: {  // kS2 x y
          const double a = kS2 * al, g = kS2 * ga;
          S = kS2 * d[0] * d[1];
          sb = kS2 * fma(d[1], b[0], d[0] * b[1]);
          v[0] = fma(d[1], a, fma(b[1], g, v[0]));
          v[1] = fma(d[0], a, fma(b[0], g, v[1]));
          break;
        }
        case 5: {  // kS2 y z
          const double a = kS2 * al, g = kS2 * ga;
          S = kS2 * d[1] * d[2];
          sb = kS2 * fma(d[2], b[1], d[1] * b[2]);
          v[1] = fma(d[2], a, fma(b[2], g, v[1]));
          v[2] = fma(d[1], a, fma(b[1], g, v[2]));
          break;
        }
        case 6: {  // kS20 (2 z^2 - x^2 - y^2)
          const double a = 2.0 * kS20 * al, g = 2.0 * kS20 * ga;
          S = kS20 * fma(2.0 * d[2], d[2], -fma(d[0], d[0], d[1] * d[1]));
          sb = 2.0 * kS20 * fma(2.0 * d[2], b[2], -fma(d[0], b[0], d[1] * b[1]));
          v[0] = fma(-d[0], a, fma(-b[0], g, v[0]));
          v[1] = fma(-d[1], a, fma(-b[1], g, v[1]));
          v[2] = fma(2.0 * d[2], a, fma(2.0 * b[2], g, v[2]));
          break;
        }
        case 7: {  // kS2 x z
          const double a = kS2 * al, g = kS2 * ga;
          S = kS2 * d[0] * d[2];
          sb = kS2 * fma(d[2], b[0], d[0] * b[2]);
          v[0] = fma(d[2], a, fma(b[2], g, v[0]));
          v[2] = fma(d[0], a, fma(b[0], g, v[2]));
          break;
        }
        case 8: {  // kS22 (x^2 - y^2)
          const double a = 2.0 * kS22 * al, g = 2.0 * kS22 * ga;
          S = kS22 * fma(d[0], d[0], -(d[1] * d[1]));
          sb = 2.0 * kS22 * fma(d[0], b[0], -(d[1] * b[1]));
          v[0] = fma(d[0], a, fma(b[0], g, v[0]));
          v[1] = fma(-d[1], a, fma(-b[1], g, v[1]));
          break;
        }
        default: {
          double Sg[3] = {0.0, 0.0, 0.0}, Sb[3] = {0.0, 0.0, 0.0};
          S = 0.0;
          harm_hess(lane_int(gf.rec.term_off, l0 + i), lane_int(gf.rec.term_cnt, l0 + i), T, d, b,
                    S, Sg, Sb);
          sb = Sg[0] * b[0] + Sg[1] * b[1] + Sg[2] * b[2];
#pragma unroll
          for (int k = 0; k < 3; ++k) v[k] = fma(Sg[k], al, fma(Sb[k], ga, v[k]));
          break;
        }
      }
      const double SR = S * st.C;
      beta = fma(SR, w, fma(fma(st.C, sb, S * Axb), x, beta));
      delta = fma(SR, x, delta);
    }
  }
  flush(first);
  if (lane < 3 * NF) cp[lane] = mine;
}

}  // namespace nkx
