// STO values and gradients of a run of wave-uniform functions at a lane's
// point, FP64.  A wave takes one function at a time (a point per lane), so the
// branches on the function are scalar branches; consecutive functions on one
// centre share d = r - R, |d| and 1 / |d|, and those of one shell also the
// radial factor R(r) = N r^k e^{-zeta r} and R'(r) / r (stobasis.hpp:494-584).
#pragma once

#include "nkx_internal.hpp"
#include "sto_eval.hpp"

namespace nkx {

// r = sqrt(a) and ir = 1 / sqrt(a) from one reciprocal square root estimate
// (v_rsq_f64, about 27 bits) and two coupled Newton (Goldschmidt) steps, ir with
// a third: both as close as a square root and a quotient (within an ulp of
// sqrt(a) and of 1 / r).  Fourteen instructions where those take about 30.
__device__ __forceinline__ void sqrt_rsqrt(double a, double &r, double &ir) {
  const double y = __builtin_amdgcn_rsq(a);
  double g = a * y, h = 0.5 * y;
  double e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  e = fma(-h, g, 0.5);
  h = fma(h, e, h);
  r = fma(fma(-g, g, a), h, g);
  ir = h + h;
  ir = fma(ir, fma(-r, ir, 1.0), ir);
  if (!(a > 1e-290 && a < 1e290)) {  // zero, denormal, overflow, NaN
    r = sqrt(a);
    ir = 1.0 / r;
  }
}

// Normalisations of the real solid harmonics to l = 2.
constexpr double kS0 = 0.28209479177387814;   // sqrt(1 / 4 pi)
constexpr double kS1 = 0.48860251190291992;   // sqrt(3 / 4 pi)
constexpr double kS2 = 1.0925484305920792;    // sqrt(15 / 4 pi)
constexpr double kS20 = 0.31539156525252005;  // sqrt(5 / 16 pi)
constexpr double kS22 = 0.54627421529603959;  // sqrt(15 / 16 pi)

// The state of a run of functions at one point.
struct StoRun {
  double d[3], r, ir;  // of the current centre
  double R, C;         // of the current shell: R and R' / r

  __device__ __forceinline__ void centre(double x, double y, double z) {
    d[0] = x;
    d[1] = y;
    d[2] = z;
    sqrt_rsqrt(x * x + y * y + z * z, r, ir);
  }
  template <bool MIXED>
  __device__ __forceinline__ void shell(int k, double zeta, double norm) {
    const double e = MIXED ? exp_neg_mixed(zeta * r) : exp(-zeta * r);
    R = norm * ipow(r, k) * e;
    C = fma((double)k, ir, -zeta) * R * ir;
  }
  // The solid harmonic and (GRAD) its gradient: closed forms to l = 2 (type l l
  // + l + m), the monomial list beyond (type -1)
  template <bool GRAD>
  __device__ __forceinline__ void harmonic(int type, int off, int cnt,
                                           const HarmTerm *__restrict__ T, double &S,
                                           double (&g)[3]) const {
    const double x = d[0], y = d[1], z = d[2];
    g[0] = g[1] = g[2] = 0.0;
    switch (type) {
      case 0:
        S = kS0;
        return;
      case 1:
        S = kS1 * y;
        if (GRAD) g[1] = kS1;
        return;
      case 2:
        S = kS1 * z;
        if (GRAD) g[2] = kS1;
        return;
      case 3:
        S = kS1 * x;
        if (GRAD) g[0] = kS1;
        return;
      case 4: {
        const double cx = kS2 * x, cy = kS2 * y;
        S = cx * y;
        if (GRAD) g[0] = cy, g[1] = cx;
        return;
      }
      case 5: {
        const double cy = kS2 * y, cz = kS2 * z;
        S = cy * z;
        if (GRAD) g[1] = cz, g[2] = cy;
        return;
      }
      case 6: {
        S = kS20 * fma(2.0 * z, z, -fma(x, x, y * y));
        if (GRAD) g[0] = -2.0 * kS20 * x, g[1] = -2.0 * kS20 * y, g[2] = 4.0 * kS20 * z;
        return;
      }
      case 7: {
        const double cx = kS2 * x, cz = kS2 * z;
        S = cx * z;
        if (GRAD) g[0] = cz, g[2] = cx;
        return;
      }
      case 8: {
        S = kS22 * fma(x, x, -(y * y));
        if (GRAD) g[0] = 2.0 * kS22 * x, g[1] = -2.0 * kS22 * y;
        return;
      }
      default: break;
    }
    S = 0.0;
    for (int t = off; t < off + cnt; ++t) {
      const HarmTerm h = T[t];
      const double xa1 = ipow(x, h.a > 0 ? h.a - 1 : 0);
      const double yb1 = ipow(y, h.b > 0 ? h.b - 1 : 0);
      const double zc1 = ipow(z, h.c > 0 ? h.c - 1 : 0);
      const double xa = h.a > 0 ? xa1 * x : 1.0;
      const double yb = h.b > 0 ? yb1 * y : 1.0;
      const double zc = h.c > 0 ? zc1 * z : 1.0;
      S += h.coef * xa * yb * zc;
      if (GRAD) {
        if (h.a > 0) g[0] += h.coef * h.a * xa1 * yb * zc;
        if (h.b > 0) g[1] += h.coef * h.b * xa * yb1 * zc;
        if (h.c > 0) g[2] += h.coef * h.c * xa * yb * zc1;
      }
    }
  }
  // Function f of a run; prev: the one before (first: none).  Value and (GRAD)
  // gradient.
  template <bool GRAD, bool MIXED>
  __device__ __forceinline__ void eval(const FuncRec &f, const FuncRec &prev, bool first,
                                       const HarmTerm *__restrict__ T, double x, double y,
                                       double z, double &v, double (&gr)[3]) {
    // bit patterns compared: scalar instructions on uniform records, no chain of
    // branches
    auto diff = [](double a, double b) { return __double_as_longlong(a) ^ __double_as_longlong(b); };
    const bool newc =
        first || (diff(f.cx, prev.cx) | diff(f.cy, prev.cy) | diff(f.cz, prev.cz)) != 0;
    const bool news = (diff(f.zeta, prev.zeta) | diff(f.norm, prev.norm) | (f.k ^ prev.k)) != 0;
    if (newc) centre(x - f.cx, y - f.cy, z - f.cz);
    if (newc || news)
      shell<MIXED>(f.k, f.zeta, f.norm);
    double S, g[3];
    harmonic<GRAD>(f.type, f.term_off, f.term_cnt, T, S, g);
    v = R * S;
    if (GRAD) {
#pragma unroll
      for (int k = 0; k < 3; ++k) gr[k] = fma(S, d[k] * C, R * g[k]);
    }
  }
};

}  // namespace nkx
