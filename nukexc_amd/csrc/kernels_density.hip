// FP64 density stage of the batched build (gfx950): the contraction X = P Phi
// with its column sums (density_fused_f64) and the Z arrays (z_slots_f64); the
// per-batch functional between them is the one of the int8 form.
#include <algorithm>

#include "lane_sums.hpp"
#include "nkx_internal.hpp"
#include "sto_run.hpp"
#include "vxc_kernels.hpp"

namespace nkx {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int FB = 64;          // functions per block
constexpr int PT = 64;          // points per batch
constexpr int TILE = FB * PT;
constexpr int KS = 16;          // functions of a stage
constexpr int STG = KS * PT;    // doubles of a stage

// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima)
__device__ __forceinline__ void wait_vm0() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// ---------------------------------------------------------------------------
// X = P Phi for one pair of a batch's live blocks and, per block, the column
// sums over its 64 functions of Phi X and (GGA) d/dx Phi X, d/dy Phi X,
// d/dz Phi X.
//
// One workgroup of four waves per (group of consecutive batches, spin, pair
// of list blocks), batch after batch.  A wave holds 32 rows of its block x 64
// points (16 rows of the only block where the pair has one), so that each Phi
// fragment read from LDS feeds two products.  The contraction runs in stages
// of 16 functions: Phi of the next stage is copied straight into the other
// LDS buffer and the next P fragments are loaded into the other register set
// while the current stage's products run (one wait and one barrier per
// stage).  P rows are read by the wave that owns them, from the cache
// hierarchy; the contraction index is dealt to lanes in runs of four, so that
// a lane loads 32 contiguous bytes of its row (Pt is the gathered transpose
// of P: row mu holds P(nu, mu)).  Points are exchanged between the two halves
// of an LDS row of 64 for rows with bit 2 set, so that the two rows that half
// a wave reads fall on different banks.  With the gradient the functions are
// evaluated again for the column sums, a point per lane and a function at a
// time (sto_run.hpp), so that no gradient array is kept: its reads (128 KB per
// block) were a quarter of the kernel's time.
//
// Bound by the FP64 MFMA rate (64 cycles per 16 x 16 x 4 product and SIMD): 16
// waters (400 functions, 1.04 M points) take 9.1 ms, 45 TFLOP/s on the padded
// blocks, with 1.1 and 1.3 ms in the collocation and the Z stage.  Stages of 32
// functions fit two workgroups per CU and not three: 9.7 ms; reading the stored
// gradient, 9.0 ms (three workgroups) with 2.75 and 3.4 ms in the other two.  One
// workgroup per batch group with the P block and the Phi tile staged through
// VGPRs, two barriers per step and 94 KB of LDS took 22.1 ms together with the
// Z stage.
template <bool GGA>
__global__ void __launch_bounds__(256, 3) density_fused_f64(
    MolTab mt, int64_t pspin, int nspin, int group, const double *__restrict__ Pt,
    const int *__restrict__ b_off, const int *__restrict__ b_fbl, int64_t s0, int64_t b0,
    int64_t b1, int nmg, int narr, const FuncRec *__restrict__ F,
    const HarmTerm *__restrict__ T, const double *__restrict__ px,
    const double *__restrict__ py, const double *__restrict__ pz,
    const double *__restrict__ tiles, int64_t pstride, double *__restrict__ part) {
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
      v4d v[2];  // row group
    };
    const int nst = 4 * n;
    auto issue = [&](int s, double *dst, AFrag &a) {
      const int ki = lo + (s >> 2), h = s & 3;
      const int fk = __builtin_amdgcn_readfirstlane(b_fbl[ki]);
      const double *p = prow + (fk - mbase) * FB + KS * h;
      a.v[0] = *reinterpret_cast<const v4d *>(p);
      if (two) a.v[1] = *reinterpret_cast<const v4d *>(p + (int64_t)16 * ld);
      const double *src = tiles + (int64_t)(ki - s0) * narr * TILE + STG * h;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        // rows 2 rp, 2 rp + 1: 16 bytes per lane
        const int rp = 2 * wv + u, r = 2 * rp + (lane >> 5);
        const int c = (lane & 31) ^ (((rp >> 1) & 1) << 3);
        __builtin_amdgcn_global_load_lds(src + r * PT + 2 * c, dst + rp * 2 * PT, 16, 0, 0);
      }
    };
    auto products = [&](const double *cur, const AFrag &a) {
      const int col = l16 ^ ((q & 1) << 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        double bv[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) bv[j] = cur[(4 * q + e) * PT + ((16 * j) ^ col)];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[0][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.v[0][e], bv[j], acc[0][j], 0, 0, 0);
        if (two) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[1][j] =
                __builtin_amdgcn_mfma_f64_16x16x4f64(a.v[1][e], bv[j], acc[1][j], 0, 0, 0);
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
    if (GGA) {
      // column sums, a point per lane: eight rows of X at a time through the
      // wave's part of the buffers (columns exchanged by the row's low bits, so
      // that the four rows of a write fall on different banks)
      __syncthreads();  // every wave is done with the buffers
      double *xw = (wv & 2 ? bufB : bufA) + (wv & 1) * (STG / 2);
      const FuncRec *fr = F + (int64_t)fm * FB + row0;
      const int64_t gp = b * PT + lane;
      const double x = px[gp], y = py[gp], z = pz[gp];
      double sum[4] = {0.0, 0.0, 0.0, 0.0};
      StoRun run;
      const int nrow = two ? 32 : 16;
#pragma unroll 1
      for (int i = 0; i < nrow; ++i) {
        if ((i & 7) == 0) {
          wave_fence();
          auto put = [&](const v4d(&c)[4], int h) {
#pragma unroll
            for (int rr = 0; rr < 2; ++rr)
#pragma unroll
              for (int j = 0; j < 4; ++j)
                xw[(4 * rr + q) * PT + ((16 * j + l16) ^ (4 * q))] = h ? c[j][2 + rr] : c[j][rr];
          };
          if (i == 0) put(acc[0], 0);
          if (i == 8) put(acc[0], 1);
          if (i == 16) put(acc[1], 0);
          if (i == 24) put(acc[1], 1);
          wave_fence();
        }
        double v, gr[3];
        run.eval<true, false>(fr[i], fr[i ? i - 1 : 0], i == 0, T, x, y, z, v, gr);
        const double X = xw[(i & 7) * PT + (lane ^ (4 * (i & 3)))];
        sum[0] = fma(v, X, sum[0]);
#pragma unroll
        for (int c = 0; c < 3; ++c) sum[c + 1] = fma(gr[c], X, sum[c + 1]);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) red[wv][c][lane] = sum[c];
    } else {
      // column sum: this lane's rows, then the q lanes
      const double *tb = tiles + (int64_t)(im - s0) * narr * TILE + (row0 + q) * PT + l16;
      double sum[4] = {0.0, 0.0, 0.0, 0.0};  // point group
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        if (g == 1 && !two) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            sum[j] += tb[(16 * g + 4 * r) * PT + 16 * j] * acc[g][j][r];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        double v = sum[j];
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        if (q == 0) red[wv][0][16 * j + l16] = v;
      }
#pragma unroll
      for (int c = 1; c < 4; ++c) red[wv][c][lane] = 0.0;
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
// the slot; coef[s] + 4 point.  With the gradient the functions are evaluated
// here (thread t: functions 16 (t / 64) .. +15 at point t % 64, both spins from
// one evaluation), without it Z is a multiple of the stored Phi.
//
// Bound by FP64 VALU issue with the gradient: 1.3 ms on 16 waters; writing the
// gradient with Phi and reading both back (128 KB per slot) took 1.7 ms more in
// the collocation and 3.4 ms here.
template <bool GGA>
__global__ void __launch_bounds__(256) z_slots_f64(
    int64_t s0, const int *__restrict__ slot_b, const int *__restrict__ b_fbl,
    const FuncRec *__restrict__ F, const HarmTerm *__restrict__ T,
    const double *__restrict__ px, const double *__restrict__ py,
    const double *__restrict__ pz, int narr, int nspin, const double *__restrict__ coef,
    int64_t cspin, double ascale, double *__restrict__ tiles) {
  const int64_t slot = s0 + blockIdx.x, b = slot_b[slot];
  const int f0 = 16 * __builtin_amdgcn_readfirstlane(threadIdx.x / PT), g = threadIdx.x & (PT - 1);
  const int64_t gp = b * PT + g;
  const double *phi = tiles + (int64_t)blockIdx.x * narr * TILE + f0 * PT + g;
  double *zt = tiles + ((int64_t)blockIdx.x * narr + narr - nspin) * TILE + f0 * PT + g;
  double k[2][4];
#pragma unroll
  for (int s = 0; s < 2; ++s)
    if (s < nspin) {
      const double *p = coef + s * cspin + 4 * gp;
      k[s][0] = ascale * p[0];
#pragma unroll
      for (int a = 1; a < 4; ++a) k[s][a] = GGA ? p[a] : 0.0;
    }
  if (GGA) {
    const FuncRec *fr = F + (int64_t)b_fbl[slot] * FB + f0;
    const double x = px[gp], y = py[gp], z = pz[gp];
    StoRun run;
#pragma unroll 1
    for (int i = 0; i < 16; ++i) {
      double v, gr[3];
      run.eval<true, false>(fr[i], fr[i ? i - 1 : 0], i == 0, T, x, y, z, v, gr);
#pragma unroll
      for (int s = 0; s < 2; ++s)
        if (s < nspin)
          zt[s * TILE + i * PT] =
              fma(k[s][3], gr[2], fma(k[s][2], gr[1], fma(k[s][1], gr[0], k[s][0] * v)));
    }
  } else {
    double v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = phi[i * PT];
#pragma unroll
    for (int s = 0; s < 2; ++s)
      if (s < nspin) {
#pragma unroll
        for (int i = 0; i < 16; ++i) zt[s * TILE + i * PT] = k[s][0] * v[i];
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
  // pairs of list blocks of the fullest batch (of the whole basis: 512 blocks of
  // which three are live, 131 k batches, 65 ms for 44)
  const int nmg = std::max(1, (pl.max_live + 1) / 2);
  const int64_t step = max_workgroups(256) / (8 * nmg * nspin) * 8 * g;  // batches of a launch
  for (int64_t b = b0; b < b1; b += step) {
    const int64_t be = std::min(b + step, b1), ng = ((be - b + g - 1) / g + 7) / 8 * 8;
    hipLaunchKernelGGL(gga ? density_fused_f64<true> : density_fused_f64<false>,
                       dim3((unsigned)(ng * nmg * nspin)), dim3(256), 0, s, pl.tab(), pl.P_total,
                       nspin, g, Pt, pl.b_off.p, pl.b_fbl.p, s0, b, be, nmg, narr, pl.funcs.p,
                       pl.terms.p, pl.px.p, pl.py.p, pl.pz.p, tiles, pstride, part);
    NKX_HIP_CHECK(hipGetLastError());
  }
}

void vk_z_slots(hipStream_t s, int64_t s0, int64_t s1, const Plan &pl, int narr, int nspin,
                int gga, double ascale, const double *coef, double *tiles) {
  if (s1 <= s0) return;
  hipLaunchKernelGGL(gga ? z_slots_f64<true> : z_slots_f64<false>, dim3((unsigned)(s1 - s0)),
                     dim3(256), 0, s, s0, pl.slot_b.p, pl.b_fbl.p, pl.funcs.p, pl.terms.p,
                     pl.px.p, pl.py.p, pl.pz.p, narr, nspin, coef, (int64_t)4 * pl.npts_pad,
                     ascale, tiles);
  NKX_HIP_CHECK(hipGetLastError());
}

}  // namespace nkx
