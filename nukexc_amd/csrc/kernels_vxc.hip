// Batched V_xc build on MI355X (gfx950), FP64 form.
//
// Data layout in HBM (one chunk of point batches at a time):
//   tile store   [slot][array][64 functions][64 points], array = Phi, then Z (of
//                each spin).  A slot is one (function block, point batch) pair
//                that survived screening.  No gradient is stored: it is formed
//                again where it is used.
//   Pd           transpose of the permuted, zero-padded density matrix.
//   vpart        split-K partial V tiles [split][pair][64][64].
//
// Kernels per chunk:
//   colloc_tiles_f64   Phi of every live slot.
//   density_fused_f64  X = P Phi on MFMA over the batch's live function blocks
//                      and the column sums of Phi X and grad Phi X, then density_f
//                      (density_fp), the functional per batch, and z_slots_f64, Z =
//                      w (v_rho / 2 Phi + 2 v_sigma grad rho . grad Phi) into the
//                      tile store (kernels_density.hip, kernels_vxc_i8.hip).
//   vgemm_f64          one workgroup per (2 x 2 super-pair of blocks, or pair;
//                      split): V += Phi_I Z_J^T + Z_I Phi_J^T over the batches
//                      where both blocks are live.
// and once per build finish_kernel: split sum, un-permutation and mirror image, and
// the energy and electron-count sums.
#include <algorithm>

#include "nkx_internal.hpp"
#include "sto_run.hpp"
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
// One workgroup per live slot: thread t takes the 16 consecutive functions
// 16 (t / 64) .. +15 of the block at point t % 64 (sto_run.hpp).
__global__ void __launch_bounds__(256) colloc_tiles_f64(
    int64_t s0, const int *__restrict__ slot_b, const int *__restrict__ b_fbl,
    const FuncRec *__restrict__ F, const HarmTerm *__restrict__ T,
    const double *__restrict__ px, const double *__restrict__ py,
    const double *__restrict__ pz, int narr, double *__restrict__ tiles) {
  const int64_t s = s0 + blockIdx.x;
  const int b = slot_b[s];
  const int f0 = 16 * __builtin_amdgcn_readfirstlane(threadIdx.x / PT);
  const FuncRec *fr = F + (int64_t)b_fbl[s] * FB + f0;
  const int g = threadIdx.x & (PT - 1);
  const int64_t gp = (int64_t)b * PT + g;
  const double x = px[gp], y = py[gp], z = pz[gp];
  double *base = tiles + (int64_t)blockIdx.x * narr * TILE + f0 * PT + g;
  StoRun run;
#pragma unroll 1
  for (int i = 0; i < 16; ++i) {
    double v, gr[3];
    run.eval<false, false>(fr[i], fr[i ? i - 1 : 0], i == 0, T, x, y, z, v, gr);
    base[i * PT] = v;
  }
}

// ---------------------------------------------------------------------------
// V contraction on 2 x 2 block super-tiles: V(I, J) = Phi_I Z_J^T + Z_I Phi_J^T
// over the batches where I and J are live, for the four tiles (I_a, J_b) of a
// super-pair (blocks I_0 < I_1, J_0 < J_1 of one molecule, -1: missing).  On
// the diagonal (I = J) only Vbar = Phi Z^T of the four tiles is formed and
// added to its transpose at the end, half the products.  blockIdx.x = (zs
// nsplit + split) nsp + super-pair; Z is tile array zbase + zs, and the
// partials go to vpart + zs nsplit npairs 64^2, written by the first chunk of a
// build, added to by the later ones.
//
// One workgroup of eight waves per (super-pair, split); its batches b = lo +
// split + nsplit i are taken in windows of 512 candidates, compacted in
// ascending order into an LDS list of the four slots.  A batch runs in four
// stages of 16 points: Phi and Z of the J blocks are copied straight into LDS
// one stage ahead (two buffers), each wave loads its own rows of Phi_I and Z_I
// into registers one stage ahead, one wait and one barrier per stage.  A wave
// owns 32 rows of I_a and the 64 columns of J_b; with one J block 16 rows
// each; with one block in all, the four row groups twice, each with half of a
// stage's products.  The contraction index (points) is dealt to lanes in runs
// of four, so that a lane reads 32 contiguous bytes of a row; the 16-byte
// pieces of an LDS row are exchanged by bits 1 .. 3 of the row, so that sixteen
// rows fall on sixteen different bank groups.
//
// Bound by the FP64 MFMA rate (busy 67 % of the cycles on 100 waters; the rest is
// the wait at a stage's start, one workgroup per CU): 16 waters take 7.9 ms, 52 TFLOP/s,
// a 12-atom molecule with two spins 341 us, water 24 us (8.5 ms, 361 us and 27 us
// with each stage's slots looked up in LDS between its barrier and its copies).  One workgroup per
// block pair, both products on the diagonal too, read four tiles for every two
// products of them (58 GB on 16 waters): 9.9 ms, 737 us and 245 us.
//
// Where screening leaves few super-pairs whole (long chains, centres far apart) a
// unit is a single pair (sp_blk NULL), two waves to 16 rows, each with half of a
// stage's products: the work of a super-pair, 2.65 pairs, is the same with one
// live tile as with four.  build_plan counts both.  A chain of 700 atoms (7000
// functions, 21 of 110 blocks live in a batch) takes 231 ms and by super-pairs
// 279, one of 240 atoms 71 and 85; 100 waters (34 of 40) 237 and 176.
constexpr int VS = 16;             // points of a stage
constexpr int VSEC = FB * VS;      // doubles of one block's stage

// four doubles 32-byte aligned
__device__ __forceinline__ v4d ld4(const double *p) { return *reinterpret_cast<const v4d *>(p); }

// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima)
__device__ __forceinline__ void wait_vm0() { __builtin_amdgcn_s_waitcnt(0x0F70); }

__global__ void __launch_bounds__(512) vgemm_f64(
    int nsp, int nsplit, int grouped, const int4 *__restrict__ sp_blk,
    const int4 *__restrict__ sp_pidx, const int *__restrict__ pair_I,
    const int *__restrict__ pair_J, int npairs, const int *__restrict__ tile_slot, MolTab mt, int64_t b0, int64_t b1, int64_t s0,
    int narr, int zbase, int first, const double *__restrict__ tiles,
    double *__restrict__ vpart) {
  // Z_J0, Z_J1, Phi_J0, Phi_J1 of a stage; two buffers, declared apart so that
  // a copy into one is known not to touch the other
  __shared__ __attribute__((aligned(16))) double bufA[4][VSEC];
  __shared__ __attribute__((aligned(16))) double bufB[4][VSEC];
  __shared__ int ls[4][512];  // slots of I_0, I_1, J_0, J_1 per listed batch
  __shared__ int wcnt[8];
  // grouped: workgroups are dealt to the eight XCDs in turn, and the super-pairs of
  // a split run on one XCD and share its L2 for the batches' tiles; else splits
  // one after the other
  const int xcd = grouped ? blockIdx.x & 7 : 0, rr = grouped ? blockIdx.x >> 3 : blockIdx.x;
  const int nsg = grouped ? nsplit / 8 : nsplit;
  const int sp = rr % nsp, split = (rr / nsp) % nsg * (grouped ? 8 : 1) + xcd,
            zs = rr / (nsp * nsg);
  const int64_t zoff = (int64_t)(zbase + zs) * TILE;
  vpart += (int64_t)zs * nsplit * npairs * (FB * FB);
  const int4 blk = sp_blk ? sp_blk[sp] : make_int4(pair_I[sp], -1, pair_J[sp], -1);
  const int4 pix = sp_blk ? sp_pidx[sp] : make_int4(sp, -1, -1, -1);
  const bool diag = blk.x == blk.z;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, q = lane >> 4;
  // this wave's tile (wa, wb), rows row0 .. of I_wa, one or two groups of 16;
  // half: the half of a stage's products it forms (-1: all)
  const bool two = blk.w >= 0;           // two J blocks (then two I blocks)
  const bool one = !two && blk.y < 0;    // one block each side
  const int wa = one ? 0 : wv >> 2, wb = two ? wv & 1 : 0;
  const int row0 = two ? 32 * ((wv >> 1) & 1) : 16 * (wv & 3);
  const int half = one ? wv >> 2 : -1;
  v4d acc[2][4];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[g][j] = v4d{0.0, 0.0, 0.0, 0.0};
  // batches of the super-pair's molecule inside [b0, b1)
  const int mol = mt.blk_mol[blk.x];
  const int64_t mb0 = mt.b0[mol], mnb = mt.nb[mol];
  const int *ts0 = tile_slot + mt.ts_off[mol] - mb0;
  const int bl[4] = {blk.x, blk.y, blk.z, blk.w};
  int64_t tso[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) tso[u] = bl[u] >= 0 ? (int64_t)mt.blk_local[bl[u]] * mnb : -1;
  const int64_t lo = b0 > mb0 ? b0 : mb0, hi = b1 < mb0 + mnb ? b1 : mb0 + mnb;
  if (!first && lo + split >= hi) return;  // nothing to add

  struct AFrag {
    v4d f[2], z[2];  // rows of Phi_I, Z_I per row group
  };
  // a listed batch's slots of this wave's I block and of the J blocks, read a
  // batch ahead (so that no LDS look-up sits between a barrier and the copies)
  struct Slots {
    int I, J[2];
  };
  auto slots = [&](int i) {
    return Slots{__builtin_amdgcn_readfirstlane(ls[wa][i]),
                 {__builtin_amdgcn_readfirstlane(ls[2][i]),
                  __builtin_amdgcn_readfirstlane(ls[3][i])}};
  };
  // operands of stage st (point group) of a batch: this wave's rows to
  // registers (those of slot s0 where its tile is idle: never used), the J
  // blocks to LDS
  auto issue = [&](const Slots &sl, int st, double (*dst)[VSEC], AFrag &a) {
    const double *pI = tiles + (int64_t)(sl.I >= 0 ? sl.I - s0 : 0) * narr * TILE +
                       (row0 + l16) * PT + VS * st + 4 * q;
    a.f[0] = ld4(pI);
    if (two) a.f[1] = ld4(pI + 16 * PT);
    if (!diag) {
      a.z[0] = ld4(pI + zoff);
      if (two) a.z[1] = ld4(pI + zoff + 16 * PT);
    }
    // 8 rows x 128 bytes per copy, the waves in turn
#pragma unroll
    for (int jb = 0; jb < 2; ++jb) {
      if (jb && !two) continue;
      if (sl.J[jb] < 0) continue;
      const int r = 8 * wv + (lane >> 3);
      const int c = (lane & 7) ^ ((r >> 1) & 7);
      const double *src =
          tiles + (int64_t)(sl.J[jb] - s0) * narr * TILE + r * PT + VS * st + 2 * c;
      __builtin_amdgcn_global_load_lds(src + zoff, &dst[jb][8 * wv * VS], 16, 0, 0);
      if (!diag) __builtin_amdgcn_global_load_lds(src, &dst[2 + jb][8 * wv * VS], 16, 0, 0);
    }
  };
  // A (rows of I) x the section's 64 columns, four steps of four points
  auto phase = [&](const double *sec, const v4d (&a)[2]) {
    v4d bv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = 16 * j + l16, x = (r >> 1) & 7;
      const double2 u = *reinterpret_cast<const double2 *>(sec + r * VS + 2 * ((2 * q) ^ x));
      const double2 v = *reinterpret_cast<const double2 *>(sec + r * VS + 2 * ((2 * q + 1) ^ x));
      bv[j] = v4d{u.x, u.y, v.x, v.y};
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (half >= 0 && (e >> 1) != half) continue;  // uniform
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[0][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[0][e], bv[j][e], acc[0][j], 0, 0, 0);
      if (two) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[1][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[1][e], bv[j][e], acc[1][j], 0, 0, 0);
      }
    }
  };
  AFrag a0, a1;
  auto ready = [&]() {  // the stage's operands are there, the other buffer is free
    wait_vm0();
    __syncthreads();
  };
  auto products = [&](double (*cur)[VSEC], const AFrag &a) {
    phase(&cur[wb][0], a.f);
    if (!diag) phase(&cur[2 + wb][0], a.z);
  };

  for (int64_t c0 = lo + split; c0 < hi; c0 += 512 * (int64_t)nsplit) {
    const int64_t b = c0 + (int64_t)nsplit * threadIdx.x;
    int sl[4] = {-1, -1, -1, -1};
    if (b < hi) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (tso[u] >= 0) sl[u] = ts0[tso[u] + b];
    }
    const bool act = (sl[0] >= 0 || sl[1] >= 0) && (sl[2] >= 0 || sl[3] >= 0);
    const unsigned long long m = __ballot(act);
    __syncthreads();  // the previous window is done with the list and buffers
    if (lane == 0) wcnt[wv] = __popcll(m);
    __syncthreads();
    int off = 0, n = 0;
    for (int w = 0; w < 8; ++w) {
      if (w < wv) off += wcnt[w];
      n += wcnt[w];
    }
    n = __builtin_amdgcn_readfirstlane(n);
    if (act) {
      const int i = off + __popcll(m & ((1ull << lane) - 1ull));
#pragma unroll
      for (int u = 0; u < 4; ++u) ls[u][i] = sl[u];
    }
    __syncthreads();
    if (n == 0) continue;
    Slots cur = slots(0);
    issue(cur, 0, bufA, a0);
    for (int i = 0; i < n; ++i) {
      const bool live = cur.I >= 0 && (wb ? cur.J[1] : cur.J[0]) >= 0;
      ready();
      issue(cur, 1, bufB, a1);
      if (live) products(bufA, a0);
      ready();
      issue(cur, 2, bufA, a0);
      const Slots nxt = slots(i + 1 < n ? i + 1 : i);
      if (live) products(bufB, a1);
      ready();
      issue(cur, 3, bufB, a1);
      if (live) products(bufA, a0);
      ready();
      if (i + 1 < n) issue(nxt, 0, bufA, a0);
      if (live) products(bufB, a1);
      cur = nxt;
    }
  }

  double(*t)[FB + 1] = reinterpret_cast<double(*)[FB + 1]>(&bufA[0][0]);
  static_assert(sizeof(bufA) >= 32 * (FB + 1) * sizeof(double), "half a tile in a buffer");
  if (one) {  // the second halves' sums through LDS, 32 rows at a time
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      __syncthreads();
      if (half == 1 && (row0 >> 5) == h) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) t[(row0 & 31) + 4 * r + q][16 * j + l16] = acc[0][j][r];
      }
      __syncthreads();
      if (half == 0 && (row0 >> 5) == h) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[0][j][r] += t[(row0 & 31) + 4 * r + q][16 * j + l16];
      }
    }
  }
  if (diag) {
    // through LDS, tile by tile:
    // V(a, b) = Vbar(a, b) + Vbar(b, a)^T for (0, 0), (0, 1), (1, 1)
    const int ng = two ? 2 : 1;
    const int ntile = two ? 3 : (one ? 1 : 2);
    for (int k = 0; k < ntile; ++k) {
      // target tile (ta, tb), from tile (tb, ta)
      const int ta = k == 2 ? 1 : 0, tb = k == 0 ? 0 : 1;
      v4d add[2][4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {  // rows 32 h .. of the source = columns of the target
        __syncthreads();
        if (wa == tb && wb == ta && half != 1) {
#pragma unroll
          for (int g = 0; g < 2; ++g)
            if (g < ng && ((row0 + 16 * g) >> 5) == h) {
#pragma unroll
              for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                  t[((row0 + 16 * g) & 31) + 4 * r + q][16 * j + l16] = acc[g][j][r];
            }
        }
        __syncthreads();
        if (wa == ta && wb == tb) {
#pragma unroll
          for (int g = 0; g < 2; ++g)
            if (g < ng) {
#pragma unroll
              for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                  add[g][2 * h + j][r] = t[16 * j + l16][row0 + 16 * g + 4 * r + q];
            }
        }
      }
      if (wa == ta && wb == tb) {
#pragma unroll
        for (int g = 0; g < 2; ++g)
          if (g < ng)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[g][j] += add[g][j];
      }
    }
  }
  const int pp = wa ? (wb ? pix.w : pix.z) : (wb ? pix.y : pix.x);
  if (pp < 0 || half == 1) return;
  double *out = vpart + ((int64_t)split * npairs + pp) * (FB * FB);
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    if (g && !two) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int mu = row0 + 16 * g + 4 * r + q, nu = 16 * j + l16;
        out[mu * FB + nu] = first ? acc[g][j][r] : out[mu * FB + nu] + acc[g][j][r];
      }
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

struct VArgs {
  double *p[kVArgs];
};
__global__ void __launch_bounds__(256) finish_kernel(
    int npairs, int nsplit, int nz, const int *__restrict__ pair_I,
    const int *__restrict__ pair_J, const int *__restrict__ fperm, MolTab mt, int nmol,
    const int *__restrict__ mol_nbf, const double *__restrict__ vpart,
    VArgs va, double *const *__restrict__ Vmol, const double *__restrict__ en,
    double *__restrict__ enout) {
  __shared__ double sv[3][256];
  const unsigned wg = blockIdx.y * gridDim.x + blockIdx.x, nv = (unsigned)npairs * nz * FB;
  if (wg >= nv) {
    if (en && (int)(wg - nv) < nmol) en_reduce(mt, (int)(wg - nv), en, enout, sv);
    return;
  }
  const int mu = wg & (FB - 1);
  const int p = (int)(wg / FB) % npairs, zs = (int)(wg / FB) / npairs;
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
  const int out = zs * nmol + __builtin_amdgcn_readfirstlane(mol);
  double *V = Vmol ? Vmol[out] : va.p[out];
  V[(int64_t)oi * nbf + oj] = v;
  V[(int64_t)oj * nbf + oi] = v;
}

// Zero fill (stream-ordered kernel, also valid inside a captured graph).
__global__ void __launch_bounds__(256) fill0_kernel(int64_t n, double *__restrict__ x) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    x[i] = 0.0;
}

// out = P permuted and zero-padded, or its transpose, one matrix per blockIdx.y
__global__ void __launch_bounds__(256) gather_p_f64(GatherArgs a, int tr) {
  const GatherP g = a.g[blockIdx.y];
  const int nbf = g.nbf, nbf_pad = g.nfb * FB;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < (int64_t)nbf_pad * nbf_pad;
       e += (int64_t)gridDim.x * 256) {
    const int i = (int)(e / nbf_pad), j = (int)(e % nbf_pad);
    double v = 0.0;
    if (i < nbf && j < nbf) {
      const int fi = g.fperm[i], fj = g.fperm[j];
      v = g.P[tr ? (int64_t)fj * nbf + fi : (int64_t)fi * nbf + fj];
    }
    static_cast<double *>(g.out)[e] = v;
  }
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
void vk_gather_p(hipStream_t s, const std::vector<GatherP> &g, bool transpose) {
  for (size_t k = 0; k < g.size(); k += kGatherMax) {
    GatherArgs a{};
    const size_t n = std::min<size_t>(kGatherMax, g.size() - k);
    int64_t e = 0;
    for (size_t i = 0; i < n; ++i) {
      a.g[i] = g[k + i];
      e = std::max(e, (int64_t)FB * a.g[i].nfb * FB * a.g[i].nfb);
    }
    // (1024 blocks need one workgroup more than a launch takes)
    const int64_t nwg = std::min((e + 255) / 256, max_workgroups(256));
    hipLaunchKernelGGL(gather_p_f64, dim3((unsigned)nwg, (unsigned)n), dim3(256), 0, s, a,
                       transpose ? 1 : 0);
    NKX_HIP_CHECK(hipGetLastError());
  }
}

void vk_colloc(hipStream_t s, int64_t s0, int64_t s1, const Plan &pl, int narr,
               double *tiles) {
  if (s1 <= s0) return;
  hipLaunchKernelGGL(colloc_tiles_f64, dim3((unsigned)(s1 - s0)), dim3(256), 0, s, s0,
                     pl.slot_b.p, pl.b_fbl.p, pl.funcs.p, pl.terms.p, pl.px.p, pl.py.p, pl.pz.p,
                     narr, tiles);
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
  if (b1 <= b0 || pl.nspairs == 0) return;
  // Where the super-pairs do not fill the CUs once, pairs that take fewer rounds for
  // their size (a super-pair 2.65 pairs, 1.5 on the diagonal, 1.7 beside a single
  // block): 40 atoms (10 super-pairs, 28 pairs) with 8 splits 2.8 ms by pairs and 7.2
  // by super-pairs, with 16 2.9 and 3.6, with 24 2.8 and 2.4; benzene (1 and 3) with
  // 64 464 us and 579, with 96 465 and 401.
  bool by_pair = pl.v_by_pair;
  const int64_t ks = (int64_t)pl.nspairs * nsplit * nz, kp = (int64_t)pl.npairs * nsplit * nz;
  if (!by_pair && pl.npairs > pl.nspairs && ks <= 256)
    by_pair = (kp + 255) / 256 < (pl.max_mol_nfb <= 2 ? 1.5 : pl.max_mol_nfb == 3 ? 1.7 : 2.65);
  const int nsp = by_pair ? pl.npairs : pl.nspairs;
  const int64_t nwg = (int64_t)nsp * nsplit * nz;
  NKX_REQUIRE(nwg <= max_workgroups(512), NKX_ERR_UNSUPPORTED, "V contraction grid too large");
  // other numbers of splits leave XCDs with fewer of them than others, or none
  const int grouped = nsplit % 8 == 0;
  hipLaunchKernelGGL(vgemm_f64, dim3((unsigned)nwg), dim3(512), 0, s, nsp, nsplit, grouped,
                     reinterpret_cast<const int4 *>(by_pair ? nullptr : pl.sp_blk.p),
                     reinterpret_cast<const int4 *>(pl.sp_pidx.p), pl.pair_I.p, pl.pair_J.p,
                     pl.npairs, pl.tile_slot.p, pl.tab(), b0, b1, s0, narr, narr - nz,
                     first ? 1 : 0, tiles, vpart);
  NKX_HIP_CHECK(hipGetLastError());
}

void vk_finish(hipStream_t s, const Plan &pl, int nsplit, int nz, const double *vpart,
               double *const *V, double *const *Vmol_dev, const double *en, double *enout) {
  const int64_t nv = (int64_t)pl.npairs * nz * FB;
  const int64_t nwg = nv + (en ? pl.nmol : 0);
  if (nwg == 0) return;
  NKX_REQUIRE(nwg < (int64_t)1 << 31, NKX_ERR_UNSUPPORTED, "reduction grid too large");
  VArgs va{};
  if (!Vmol_dev) std::copy(V, V + (size_t)nz * pl.nmol, va.p);
  hipLaunchKernelGGL(finish_kernel, grid_2d(nwg, 256), dim3(256), 0, s, pl.npairs, nsplit, nz,
                     pl.pair_I.p, pl.pair_J.p, pl.fperm_d.p, pl.tab(), pl.nmol, pl.mol_nbf.p,
                     vpart, va, Vmol_dev, en, enout);
  NKX_HIP_CHECK(hipGetLastError());
}

void vk_en_reduce(hipStream_t s, const Plan &pl, const double *en, double *out) {
  hipLaunchKernelGGL(finish_kernel, dim3(pl.nmol), dim3(256), 0, s, 0, 0, 0, nullptr, nullptr,
                     nullptr, pl.tab(), pl.nmol, nullptr, nullptr, VArgs{}, nullptr, en, out);
  NKX_HIP_CHECK(hipGetLastError());
}

void vk_fill0(hipStream_t s, double *x, int64_t n) {
  if (n <= 0) return;
  const int64_t blocks = std::min<int64_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(fill0_kernel, dim3((unsigned)blocks), dim3(256), 0, s, n, x);
  NKX_HIP_CHECK(hipGetLastError());
}

}  // namespace nkx
