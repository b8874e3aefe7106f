// FP64 density stage of the batched build (gfx950): the contraction X = P Phi
// with its column sums (density_x_f64) and the Z arrays (z_slots_f64); the
// per-batch functional between them is the one of the int8 form.
#include <algorithm>

#include "nkx_internal.hpp"
#include "vxc_kernels.hpp"

namespace nkx {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int FB = 64;          // functions per block
constexpr int PT = 64;          // points per batch
constexpr int TILE = FB * PT;
constexpr int KS = 32;          // functions of a stage (half a block)
constexpr int STG = KS * PT;    // doubles of a stage

// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima)
__device__ __forceinline__ void wait_vm0() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// ---------------------------------------------------------------------------
// X = P Phi for one pair of a batch's live blocks and, per block, the column
// sums over its 64 functions of Phi X, d/dx Phi X, d/dy Phi X, d/dz Phi X.
//
// One workgroup of four waves per (group of consecutive batches, spin, pair
// of list blocks), batch after batch.  A wave holds 32 rows of its block x 64
// points (16 rows of the only block where the pair has one), so that each Phi
// fragment read from LDS feeds two products.  The contraction runs in stages
// of 32 functions: Phi of the next stage is copied straight into the other
// LDS buffer and the next P fragments are loaded into the other register set
// while the current stage's products run (one wait and one barrier per
// stage).  P rows are read by the wave that owns them, from the cache
// hierarchy; the contraction index is dealt to lanes in runs of four, so that
// a lane loads 32 contiguous bytes of its row (Pt is the gathered transpose
// of P: row mu holds P(nu, mu)).  Points are exchanged between the two halves
// of an LDS row of 64 for rows with bit 2 set, so that the two rows that half
// a wave reads fall on different banks.
//
// Bound by the FP64 MFMA rate (64 cycles per 16 x 16 x 4 product and SIMD): 16
// waters (400 functions, 1.04 M points) take 9.7 ms, 43 TFLOP/s on the padded
// blocks.  One workgroup per batch group with the P block and the Phi tile
// staged through VGPRs, two barriers per step and 94 KB of LDS (one workgroup
// per CU), took 22.1 ms together with the Z stage (3.4 ms now).
__global__ void __launch_bounds__(256, 2) density_x_f64(
    MolTab mt, int64_t pspin, int nspin, int group, const double *__restrict__ Pt,
    const int *__restrict__ b_off, const int *__restrict__ b_fbl, int64_t s0, int64_t b0,
    int64_t b1, int nmg, int narr, int gga, const double *__restrict__ tiles, int64_t pstride,
    double *__restrict__ part) {
  // the pairs and spins of a batch group run on one XCD (workgroups are dealt
  // to the eight XCDs in turn) and share its L2 for the Phi tiles
  const int xcd = blockIdx.x & 7, rr = blockIdx.x >> 3;
  const int inner = nmg * nspin;
  const int mgi = (rr % inner) / nspin, sp = rr % nspin;
  const int64_t bg = b0 + ((int64_t)(rr / inner) * 8 + xcd) * group;
  const int64_t bge = bg + group < b1 ? bg + group : b1;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, q = lane >> 4;
  // two buffers, declared apart so that a copy into one is known not to touch
  // the other
  __shared__ __attribute__((aligned(16))) double bufA[STG];
  __shared__ __attribute__((aligned(16))) double bufB[STG];
  __shared__ double red[4][4][PT];
  const double *Psp = Pt + (int64_t)sp * pspin;
  part += (int64_t)sp * pstride;

  for (int64_t b = bg; b < bge; ++b) {
    const int lo = b_off[b], n = b_off[b + 1] - lo;
    if (2 * mgi >= n) continue;  // uniform
    const bool two = 2 * mgi + 1 < n;
    const int im = lo + 2 * mgi + (two ? wv >> 1 : 0);
    const int fm = __builtin_amdgcn_readfirstlane(b_fbl[im]);
    const int mol = mt.blk_mol[fm], ld = mt.ld[mol];
    const int row0 = two ? 32 * (wv & 1) : 16 * wv;  // of the block
    // this lane's P row of row group 0, at its run of four
    const double *prow =
        Psp + mt.P_off[mol] + (int64_t)(mt.blk_local[fm] * FB + row0 + l16) * ld + 4 * q;
    const int mbase = fm - mt.blk_local[fm];
    v4d acc[2][4];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[g][j] = v4d{0.0, 0.0, 0.0, 0.0};
    struct AFrag {
      v4d v[2][2];  // row group, run of 16 functions
    };
    const int nst = 2 * n;
    auto issue = [&](int s, double *dst, AFrag &a) {
      const int ki = lo + (s >> 1), h = s & 1;
      const int fk = __builtin_amdgcn_readfirstlane(b_fbl[ki]);
      const double *p = prow + (fk - mbase) * FB + KS * h;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        a.v[0][k] = *reinterpret_cast<const v4d *>(p + 16 * k);
        if (two) a.v[1][k] = *reinterpret_cast<const v4d *>(p + (int64_t)16 * ld + 16 * k);
      }
      const double *src = tiles + (int64_t)(ki - s0) * narr * TILE + STG * h;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        // rows 2 rp, 2 rp + 1: 16 bytes per lane
        const int rp = 4 * wv + u, r = 2 * rp + (lane >> 5);
        const int c = (lane & 31) ^ (((rp >> 1) & 1) << 3);
        __builtin_amdgcn_global_load_lds(src + r * PT + 2 * c, dst + rp * 2 * PT, 16, 0, 0);
      }
    };
    auto products = [&](const double *cur, const AFrag &a) {
      const int col = l16 ^ ((q & 1) << 4);
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          double bv[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) bv[j] = cur[(16 * k + 4 * q + e) * PT + ((16 * j) ^ col)];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[0][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.v[0][k][e], bv[j], acc[0][j], 0, 0,
                                                             0);
          if (two) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              acc[1][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.v[1][k][e], bv[j], acc[1][j], 0,
                                                               0, 0);
          }
        }
    };
    AFrag a0, a1;
    __syncthreads();  // the previous batch is done with the buffers
    issue(0, bufA, a0);
    for (int s = 0; s < nst; s += 2) {  // nst is even
      wait_vm0();
      __syncthreads();  // bufA complete, bufB free
      issue(s + 1, bufB, a1);
      products(bufA, a0);
      wait_vm0();
      __syncthreads();
      if (s + 2 < nst) issue(s + 2, bufA, a0);
      products(bufB, a1);
    }
    // column sums: this lane's rows, then the q lanes, then the block's waves
    const double *tb = tiles + (int64_t)(im - s0) * narr * TILE + (row0 + q) * PT + l16;
    double sum[4][4];  // quantity, point group
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[c][j] = 0.0;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      if (g == 1 && !two) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double *t = tb + (16 * g + 4 * r) * PT;
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[0][j] += t[16 * j] * acc[g][j][r];
        if (gga) {
#pragma unroll
          for (int c = 1; c < 4; ++c)
#pragma unroll
            for (int j = 0; j < 4; ++j) sum[c][j] += t[c * TILE + 16 * j] * acc[g][j][r];
        }
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        double v = sum[c][j];
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        if (q == 0) red[wv][c][16 * j + l16] = v;
      }
    __syncthreads();
    {
      const int c = threadIdx.x >> 6, g = threadIdx.x & 63;
      double *o = part + (int64_t)(lo + 2 * mgi - s0) * (4 * PT) + c * PT + g;
      const double v0 = red[0][c][g] + red[1][c][g], v1 = red[2][c][g] + red[3][c][g];
      if (two) {
        o[0] = v0;
        o[4 * PT] = v1;
      } else {
        o[0] = v0 + v1;
      }
    }
  }
}

// Z_s = ascale a_s Phi + b_s . grad Phi per live slot, array narr - nspin + s of
// the slot; coef[s] + 4 point.  Two points per thread, both spins from one read.
// Bound by its bytes: 128 KB read and 32 KB written per slot and spin (GGA),
// 5.3 TB/s on 16 waters.
__global__ void __launch_bounds__(256) z_slots_f64(int64_t s0, const int *__restrict__ slot_b,
                                                   int narr, int nspin, int gga,
                                                   const double *__restrict__ coef,
                                                   int64_t cspin, double ascale,
                                                   double *__restrict__ tiles) {
  const int64_t b = slot_b[s0 + blockIdx.x];
  double *tb = tiles + (int64_t)blockIdx.x * narr * TILE;
  const int c = 2 * (threadIdx.x & 31), r0 = threadIdx.x >> 5;
  double2 k[2][4];
#pragma unroll
  for (int s = 0; s < 2; ++s)
    if (s < nspin) {
      const double *p = coef + s * cspin + 4 * (b * PT + c);
#pragma unroll
      for (int a = 0; a < 4; ++a) k[s][a] = make_double2(p[a], p[4 + a]);
      k[s][0].x *= ascale;
      k[s][0].y *= ascale;
    }
#pragma unroll 4
  for (int r = r0; r < FB; r += 8) {
    const double *t = tb + r * PT + c;
    double2 v[4];
    v[0] = *reinterpret_cast<const double2 *>(t);
    if (gga) {
#pragma unroll
      for (int a = 1; a < 4; ++a) v[a] = *reinterpret_cast<const double2 *>(t + a * TILE);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
      if (s < nspin) {
        double2 z = make_double2(k[s][0].x * v[0].x, k[s][0].y * v[0].y);
        if (gga) {
#pragma unroll
          for (int a = 1; a < 4; ++a) {
            z.x += k[s][a].x * v[a].x;
            z.y += k[s][a].y * v[a].y;
          }
        }
        *reinterpret_cast<double2 *>(tb + (narr - nspin + s) * TILE + r * PT + c) = z;
      }
  }
}

}  // namespace

void vk_density(hipStream_t s, int nspin, int group, int64_t b0, int64_t b1, int64_t s0,
                const Plan &pl, const double *Pt, int narr, int gga, const double *tiles,
                double *part, int64_t pstride) {
  if (b1 <= b0) return;
  NKX_REQUIRE(pl.nfb <= 1024, NKX_ERR_UNSUPPORTED,
              "more than 1024 function blocks (65536 functions)");
  const int g0 = group == 66 ? 2 : (group >= 65 ? 1 : group);  // the int8 form's codes
  const int g = g0 == 1 || g0 == 2 ? g0 : 4;
  const int nmg = (pl.max_mol_nfb + 1) / 2;
  const int64_t ng = ((b1 - b0 + g - 1) / g + 7) / 8 * 8;
  const int64_t nwg = ng * nmg * nspin;
  NKX_REQUIRE(nwg < (int64_t)1 << 31, NKX_ERR_UNSUPPORTED, "density grid too large");
  hipLaunchKernelGGL(density_x_f64, dim3((unsigned)nwg), dim3(256), 0, s, pl.tab(), pl.P_total,
                     nspin, g, Pt, pl.b_off.p, pl.b_fbl.p, s0, b0, b1, nmg, narr, gga, tiles,
                     pstride, part);
  NKX_HIP_CHECK(hipGetLastError());
}

void vk_z_slots(hipStream_t s, int64_t s0, int64_t s1, const Plan &pl, int narr, int nspin,
                int gga, double ascale, const double *coef, double *tiles) {
  if (s1 <= s0) return;
  hipLaunchKernelGGL(z_slots_f64, dim3((unsigned)(s1 - s0)), dim3(256), 0, s, s0, pl.slot_b.p,
                     narr, nspin, gga, coef, (int64_t)4 * pl.npts_pad, ascale, tiles);
  NKX_HIP_CHECK(hipGetLastError());
}

}  // namespace nkx
