// Batched V_xc build on MI355X (gfx950), FP64 form.
//
// Data layout in HBM (one chunk of point batches at a time):
//   tile store   [slot][array][64 functions][PT points], array = Phi, dPhi/dx,
//                dPhi/dy, dPhi/dz, Z (GGA) or Phi, Z (LDA); spin-polarised
//                builds carry Z_alpha, Z_beta in place of Z.  A slot is one
//                (function block, point batch) pair that survived screening.
//   Pd           transpose of the permuted, zero-padded density matrix.
//   vpart        split-K partial V tiles [split][pair][64][64].
//
// Kernels per chunk:
//   colloc_tiles     Phi and grad Phi for every live slot (HBM-write bound).
//   density_x        X = P Phi on MFMA over the batch's live function blocks and
//                    the column sums of Phi X and grad Phi X
//                    (kernels_density.hip); density_f: the functional per
//                    batch; z_slots: Z = w (v_rho/2 Phi + 2 v_sigma grad rho .
//                    grad Phi) written back to the tile store.
//   vgemm            one workgroup per (function-block pair I <= J, split):
//                    acc += Phi_I Z_J^T + Z_I Phi_J^T over the batches where
//                    both blocks are live (MFMA-bound).
// and once per build: finish (split sum + un-permute + mirror, and the FP64
// energy / electron-count sums).
#include <algorithm>

#include "nkx_internal.hpp"
#include "sto_eval.hpp"
#include "vxc_kernels.hpp"

namespace nkx {

typedef double v4d __attribute__((ext_vector_type(4)));

// v_mfma_f64_16x16x4f64 lane layout (checked by tests/gpu_probe): lane l
// supplies A[l%16][l/16] and B[l/16][l%16]; result register r of lane l
// holds D[4r + l/16][l%16].

constexpr int FB = 64;   // functions per block
constexpr int PT = 64;   // points per batch
constexpr int TILE = FB * PT;

// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) colloc_tiles_f64(
    int64_t s0, const int *__restrict__ slot_b, const int *__restrict__ b_fbl,
    const FuncRec *__restrict__ F, const HarmTerm *__restrict__ T,
    const double *__restrict__ px, const double *__restrict__ py,
    const double *__restrict__ pz, int narr, int gga, double *__restrict__ tiles) {
  const int64_t s = s0 + blockIdx.x;
  const int b = slot_b[s];
  const int fb = b_fbl[s];
  __shared__ FuncRec fr[FB];
  if (threadIdx.x < FB) fr[threadIdx.x] = F[fb * FB + threadIdx.x];
  __syncthreads();
  const int g = threadIdx.x & (PT - 1);
  const int row = threadIdx.x / PT;
  const int64_t gp = (int64_t)b * PT + g;
  const double x = px[gp], y = py[gp], z = pz[gp];
  double *base = tiles + (int64_t)blockIdx.x * narr * TILE;
#pragma unroll 1
  for (int f = row; f < FB; f += 256 / PT) {
    const FuncRec rec = fr[f];
    const int e = f * PT + g;
    if (gga) {
      double v, a, bb, c;
      sto_value_grad<double>(rec, T, x, y, z, v, a, bb, c);
      base[e] = v;
      base[TILE + e] = a;
      base[2 * TILE + e] = bb;
      base[3 * TILE + e] = c;
    } else {
      base[e] = sto_value<double>(rec, T, x, y, z);
    }
  }
}

// ---------------------------------------------------------------------------
// acc(I, J) += Phi_I Z_J^T + Z_I Phi_J^T over batches where I and J are live.
constexpr int HP = 32;      // points per LDS stage
constexpr int LDP = HP + 1; // padded row

// blockIdx.x = (zs * nsplit + split) * npairs + pair; Z is tile array
// zbase + zs, and the partials go to vpart + zs * nsplit * npairs * FB * FB:
// written by the first chunk of a build, added to by the later ones.
__global__ void __launch_bounds__(256) vgemm_f64(
    int npairs, int nsplit, const int *__restrict__ pair_I, const int *__restrict__ pair_J,
    const int *__restrict__ tile_slot, MolTab mt, int64_t b0, int64_t b1, int64_t s0,
    int narr, int zbase, int first, const double *__restrict__ tiles,
    double *__restrict__ vpart) {
  const int p = blockIdx.x % npairs;
  const int split = (blockIdx.x / npairs) % nsplit;
  const int zs = blockIdx.x / (npairs * nsplit);
  const int zarr = zbase + zs;
  vpart += (int64_t)zs * nsplit * npairs * (FB * FB);
  const int I = pair_I[p], J = pair_J[p];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int l16 = lane & 15, q = lane >> 4;
  __shared__ double A0[FB][LDP], A1[FB][LDP], B0[FB][LDP], B1[FB][LDP];
  v4d acc[4];
  for (int j = 0; j < 4; ++j) acc[j] = v4d{0.0, 0.0, 0.0, 0.0};
  // batches of the pair's molecule inside [b0, b1)
  const int mol = mt.blk_mol[I];
  const int64_t mb0 = mt.b0[mol], mnb = mt.nb[mol];
  const int *tsI = tile_slot + mt.ts_off[mol] + (int64_t)mt.blk_local[I] * mnb - mb0;
  const int *tsJ = tile_slot + mt.ts_off[mol] + (int64_t)mt.blk_local[J] * mnb - mb0;
  const int64_t lo = b0 > mb0 ? b0 : mb0, hi = b1 < mb0 + mnb ? b1 : mb0 + mnb;
  for (int64_t b = lo + split; b < hi; b += nsplit) {
    const int sI = tsI[b], sJ = tsJ[b];
    if (sI < 0 || sJ < 0) continue;
    const double *tI = tiles + (sI - s0) * narr * TILE;
    const double *tJ = tiles + (sJ - s0) * narr * TILE;
    for (int h = 0; h < PT; h += HP) {
      {
        const double *zI = tI + zarr * TILE, *zJ = tJ + zarr * TILE;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int e = 2 * (u * 256 + (int)threadIdx.x);
          const int r = e / HP, c = e % HP;
          const int off = r * PT + h + c;
          const double2 a0 = *reinterpret_cast<const double2 *>(tI + off);
          const double2 a1 = *reinterpret_cast<const double2 *>(zI + off);
          const double2 b0v = *reinterpret_cast<const double2 *>(tJ + off);
          const double2 b1v = *reinterpret_cast<const double2 *>(zJ + off);
          A0[r][c] = a0.x;  A0[r][c + 1] = a0.y;
          A1[r][c] = a1.x;  A1[r][c + 1] = a1.y;
          B0[r][c] = b0v.x; B0[r][c + 1] = b0v.y;
          B1[r][c] = b1v.x; B1[r][c + 1] = b1v.y;
        }
      }
      __syncthreads();
#pragma unroll 2
      for (int k0 = 0; k0 < HP; k0 += 4) {
        const double aphi = A0[16 * wv + l16][k0 + q];
        const double az = A1[16 * wv + l16][k0 + q];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const double bz = B1[16 * j + l16][k0 + q];
          const double bphi = B0[16 * j + l16][k0 + q];
          acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(aphi, bz, acc[j], 0, 0, 0);
          acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(az, bphi, acc[j], 0, 0, 0);
        }
      }
      __syncthreads();
    }
  }
  double *out = vpart + ((int64_t)split * npairs + p) * (FB * FB);
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int mu = 16 * wv + 4 * r + q, nu = 16 * j + l16;
      out[mu * FB + nu] = first ? acc[j][r] : out[mu * FB + nu] + acc[j][r];
    }
}

// ---------------------------------------------------------------------------
// End of a build, one launch: the V tiles (sum of the split partials,
// un-permutation, mirror image) and the per-molecule E and N sums.
//
// Bound by reading the partials once.  Workgroup (pair p, row mu) of the first
// 64 npairs nz ones: wave k sums splits [k ns / 4, (k + 1) ns / 4) of the row's
// 64 elements with 16 loads in flight, and the four sums are added in wave
// order.  One workgroup per whole pair, a serial sum per thread, left the chip
// empty and took 1302 us on benzene (3 pairs, 335 splits, 33 MB) and 1835 us
// on 32 waters (91 pairs, 293 splits, 0.87 GB); now 11.5 us and 179 us (4.9
// TB/s).  The last nmol workgroups sum the per-batch (E, N_alpha, N_beta)
// triples of a molecule in a fixed order, eight loads ahead (60 us on 32
// waters as a launch of its own, 22 us on benzene).
constexpr int RSEG = 4;  // split segments (waves) per row

// sum over batches b0 + thread, + 256, ..., then a fixed tree
__device__ __forceinline__ void en_reduce(MolTab mt, int mol, const double *__restrict__ en,
                                          double *__restrict__ out, double (*sv)[256]) {
  const int64_t b0 = mt.b0[mol], b1 = b0 + mt.nb[mol];
  double v[3] = {0.0, 0.0, 0.0};
  int64_t b = b0 + threadIdx.x;
  for (; b + 7 * 256 < b1; b += 8 * 256) {
    double t[8][3];
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int c = 0; c < 3; ++c) t[u][c] = en[3 * (b + 256 * u) + c];
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c] += t[u][c];
  }
  for (; b < b1; b += 256)
    for (int c = 0; c < 3; ++c) v[c] += en[3 * b + c];
  for (int c = 0; c < 3; ++c) sv[c][threadIdx.x] = v[c];
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s)
      for (int c = 0; c < 3; ++c) sv[c][threadIdx.x] += sv[c][threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int c = 0; c < 3; ++c) out[3 * mol + c] = sv[c][0];
}

__global__ void __launch_bounds__(256) finish_kernel(
    int npairs, int nsplit, int nz, const int *__restrict__ pair_I,
    const int *__restrict__ pair_J, const int *__restrict__ fperm, MolTab mt, int nmol,
    const int *__restrict__ mol_nbf, const double *__restrict__ vpart,
    double *const *__restrict__ Vmol, const double *__restrict__ en, double *__restrict__ enout) {
  __shared__ double sv[3][256];
  const int64_t nv = (int64_t)npairs * nz * FB;
  if ((int64_t)blockIdx.x >= nv) {
    en_reduce(mt, (int)(blockIdx.x - nv), en, enout, sv);
    return;
  }
  const int mu = blockIdx.x & (FB - 1);
  const int p = (int)(blockIdx.x / FB) % npairs, zs = (int)(blockIdx.x / FB) / npairs;
  const int I = pair_I[p], J = pair_J[p];
  const int mol = mt.blk_mol[I];
  const int nbf = mol_nbf[mol];
  const int i = mt.blk_local[I] * FB + mu;
  if (i >= nbf) return;  // uniform: a padding row
  const int nu = threadIdx.x & (FB - 1), seg = threadIdx.x / FB;
  const int64_t st = (int64_t)npairs * (FB * FB);
  const double *src = vpart + ((int64_t)zs * nsplit * npairs + p) * (FB * FB) + mu * FB + nu;
  int s = (int)((int64_t)seg * nsplit / RSEG);
  const int s1 = (int)((int64_t)(seg + 1) * nsplit / RSEG);
  double v = 0.0;
  for (; s + 16 <= s1; s += 16) {
    double t[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) t[u] = src[(s + u) * st];
#pragma unroll
    for (int u = 0; u < 16; ++u) v += t[u];
  }
  for (; s < s1; ++s) v += src[s * st];
  sv[0][threadIdx.x] = v;
  __syncthreads();
  const int j = mt.blk_local[J] * FB + nu;
  if (seg || j >= nbf || (I == J && mu > nu)) return;
  v = ((sv[0][nu] + sv[0][FB + nu]) + sv[0][2 * FB + nu]) + sv[0][3 * FB + nu];
  const int oi = fperm[I * FB + mu], oj = fperm[J * FB + nu];
  double *V = Vmol[(int64_t)zs * nmol + mol];
  V[(int64_t)oi * nbf + oj] = v;
  V[(int64_t)oj * nbf + oi] = v;
}

// Zero fill (stream-ordered kernel, also valid inside a captured graph).
__global__ void __launch_bounds__(256) fill0_kernel(int64_t n, double *__restrict__ x) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    x[i] = 0.0;
}

// Pd = P permuted and zero-padded, or its transpose
__global__ void __launch_bounds__(256) gather_p_f64(int nbf, int nbf_pad,
                                                    const int *__restrict__ fperm, int tr,
                                                    const double *__restrict__ P,
                                                    double *__restrict__ Pd) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)nbf_pad * nbf_pad) return;
  const int i = (int)(e / nbf_pad), j = (int)(e % nbf_pad);
  double v = 0.0;
  if (i < nbf && j < nbf)
    v = tr ? P[(int64_t)fperm[j] * nbf + fperm[i]] : P[(int64_t)fperm[i] * nbf + fperm[j]];
  Pd[e] = v;
}

// Z = (w/2) Phi for the overlap build (S = Phi W Phi^T through vgemm).
__global__ void __launch_bounds__(256) zoverlap_f64(int64_t s0, const int *__restrict__ slot_b,
                                                    const double *__restrict__ pw, int narr,
                                                    double *__restrict__ tiles) {
  const int64_t s = s0 + blockIdx.x;
  const int b = slot_b[s];
  double *tb = tiles + (int64_t)blockIdx.x * narr * TILE;
  for (int e = threadIdx.x; e < TILE; e += 256)
    tb[(narr - 1) * TILE + e] = 0.5 * pw[(int64_t)b * PT + e % PT] * tb[e];
}

// ---------------------------------------------------------------------------
void vk_gather_p(hipStream_t s, int nbf, int nbf_pad, const int *fperm, bool transpose,
                 const double *P, double *Pd) {
  const int64_t n = (int64_t)nbf_pad * nbf_pad;
  hipLaunchKernelGGL(gather_p_f64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, nbf,
                     nbf_pad, fperm, transpose ? 1 : 0, P, Pd);
  NKX_HIP_CHECK(hipGetLastError());
}

void vk_colloc(hipStream_t s, int64_t s0, int64_t s1, const Plan &pl, int narr, int gga,
               double *tiles) {
  if (s1 <= s0) return;
  hipLaunchKernelGGL(colloc_tiles_f64, dim3((unsigned)(s1 - s0)), dim3(256), 0, s, s0,
                     pl.slot_b.p, pl.b_fbl.p, pl.funcs.p, pl.terms.p, pl.px.p, pl.py.p, pl.pz.p,
                     narr, gga, tiles);
  NKX_HIP_CHECK(hipGetLastError());
}

void vk_zoverlap(hipStream_t s, int64_t s0, int64_t s1, const Plan &pl, int narr,
                 double *tiles) {
  if (s1 <= s0) return;
  hipLaunchKernelGGL(zoverlap_f64, dim3((unsigned)(s1 - s0)), dim3(256), 0, s, s0, pl.slot_b.p,
                     pl.pw.p, narr, tiles);
  NKX_HIP_CHECK(hipGetLastError());
}

void vk_vgemm(hipStream_t s, int64_t b0, int64_t b1, int64_t s0, const Plan &pl, int nsplit,
              int narr, int nz, bool first, const double *tiles, double *vpart) {
  if (b1 <= b0 || pl.npairs == 0) return;
  hipLaunchKernelGGL(vgemm_f64, dim3((unsigned)(pl.npairs * nsplit * nz)), dim3(256), 0, s,
                     pl.npairs, nsplit, pl.pair_I.p, pl.pair_J.p, pl.tile_slot.p, pl.tab(), b0, b1,
                     s0, narr, narr - nz, first ? 1 : 0, tiles, vpart);
  NKX_HIP_CHECK(hipGetLastError());
}

void vk_finish(hipStream_t s, const Plan &pl, int nsplit, int nz, const double *vpart,
               double *const *Vmol_dev, const double *en, double *enout) {
  const int64_t nv = (int64_t)pl.npairs * nz * FB;
  const int64_t nwg = nv + (en ? pl.nmol : 0);
  if (nwg == 0) return;
  NKX_REQUIRE(nwg < (int64_t)1 << 31, NKX_ERR_UNSUPPORTED, "reduction grid too large");
  hipLaunchKernelGGL(finish_kernel, dim3((unsigned)nwg), dim3(256), 0, s, pl.npairs, nsplit, nz,
                     pl.pair_I.p, pl.pair_J.p, pl.fperm_d.p, pl.tab(), pl.nmol, pl.mol_nbf.p,
                     vpart, Vmol_dev, en, enout);
  NKX_HIP_CHECK(hipGetLastError());
}

void vk_en_reduce(hipStream_t s, const Plan &pl, const double *en, double *out) {
  hipLaunchKernelGGL(finish_kernel, dim3(pl.nmol), dim3(256), 0, s, 0, 0, 0, nullptr, nullptr,
                     nullptr, pl.tab(), pl.nmol, nullptr, nullptr, nullptr, en, out);
  NKX_HIP_CHECK(hipGetLastError());
}

void vk_fill0(hipStream_t s, double *x, int64_t n) {
  if (n <= 0) return;
  const int64_t blocks = std::min<int64_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(fill0_kernel, dim3((unsigned)blocks), dim3(256), 0, s, n, x);
  NKX_HIP_CHECK(hipGetLastError());
}

}  // namespace nkx
