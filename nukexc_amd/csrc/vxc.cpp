// Plan construction and orchestration of the batched V_xc build.
//
// Plan (once per geometry / basis / screening setting):
//   * points sorted along a Morton curve and cut into batches of 64, the last
//     one padded with zero-weight copies of its final point;
//   * functions sorted by (screening-radius class, Morton code of the centre)
//     and cut into blocks of 64, padded with zero functions, so that a block
//     holds functions of similar extent at nearby centres;
//   * a (block, batch) pair is live when some function of the block reaches
//     the batch's bounding box within its screening radius (the radius where
//     N r^{n-1} e^{-zeta r} drops to the screening tolerance, the
//     compute_cutoff rule of stobasis.hpp:90-173);
//   * live pairs are numbered batch-major (CSR), which is also their slot
//     number in the tile store.
// Build (once per SCF iteration): see kernels_vxc.hip.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>
#include <numeric>
#include <string>

#include "morton.hpp"
#include "nkx_internal.hpp"
#include "vxc_kernels.hpp"

namespace nkx {

namespace {

struct Box {
  double lo[3], hi[3];
};

constexpr int FB = 64;
constexpr int PT = 64;

}  // namespace

namespace {

// Host side of one molecule's plan in local numbering (functions from 0).
struct PlanPart {
  int nbf = 0, nfb = 0;
  int64_t npts = 0, nb = 0;
  std::vector<int> fperm;  // sorted -> original function
  std::vector<FuncRec> fr;
  std::vector<HarmTerm> terms;
  std::vector<double> fn;  // centre and screening radius per sorted function
};

// Functions of basis B in plan order, their records and screening radii.
PlanPart make_part(int64_t npts, const BasisHost &B, double tol) {
  PlanPart pt;
  pt.npts = npts;
  pt.nb = (npts + PT - 1) / PT;
  // ---- functions ---------------------------------------------------------
  const int nbf = B.nbf;
  const int nfb = (nbf + FB - 1) / FB;
  const int nbf_pad = nfb * FB;
  pt.nbf = nbf;
  pt.nfb = nfb;
  std::vector<double> rad(nbf);
  Box cb{{1e300, 1e300, 1e300}, {-1e300, -1e300, -1e300}};
  for (int i = 0; i < nbf; ++i) {
    double nrm, cut;
    sto_norm_cutoff(B.n[i], B.zeta[i], tol, &nrm, &cut);
    // Same radial bound with the stored normalisation (callers may scale it).
    if (B.norm[i] != nrm && B.norm[i] > 0) {
      double r = cut;
      for (int it = 0; it < 60; ++it) {
        const double v = std::log(B.norm[i]) + (B.n[i] - 1) * std::log(r) - B.zeta[i] * r -
                         std::log(tol);
        if (v <= 0) break;
        r *= 1.25;
      }
      cut = r;
    }
    rad[i] = cut;
    const double ctr[3] = {B.cx[i], B.cy[i], B.cz[i]};
    for (int d = 0; d < 3; ++d) {
      cb.lo[d] = std::min(cb.lo[d], ctr[d]);
      cb.hi[d] = std::max(cb.hi[d], ctr[d]);
    }
  }
  std::vector<std::tuple<int, uint64_t, int>> fkey(nbf);
  for (int i = 0; i < nbf; ++i) {
    const double ctr[3] = {B.cx[i], B.cy[i], B.cz[i]};
    const int cls = (int)std::floor(2.0 * std::log2(std::max(rad[i], 0.25)));
    fkey[i] = std::make_tuple(cls, morton_code<false>(ctr, cb.lo, cb.hi), i);
  }
  std::sort(fkey.begin(), fkey.end());
  pt.fperm.resize(nbf);
  for (int i = 0; i < nbf; ++i) pt.fperm[i] = std::get<2>(fkey[i]);

  pt.fr.resize(nbf_pad);
  for (int sp = 0; sp < nbf_pad; ++sp) {
    FuncRec r{};
    if (sp < nbf) {
      const int i = pt.fperm[sp];
      const auto &t = solid_harmonic_terms(B.l[i], B.m[i]);
      r.cx = B.cx[i];
      r.cy = B.cy[i];
      r.cz = B.cz[i];
      r.zeta = B.zeta[i];
      r.norm = B.norm[i];
      r.k = B.n[i] - B.l[i] - 1;
      r.term_off = (int)pt.terms.size();
      r.term_cnt = (int)t.size();
      r.type = func_type(B.l[i], B.m[i]);
      pt.terms.insert(pt.terms.end(), t.begin(), t.end());
    } else {
      r.zeta = 1.0;
      r.norm = 0.0;
      r.term_off = 0;
      r.term_cnt = 0;
      r.type = 0;
    }
    pt.fr[sp] = r;
  }

  pt.fn.resize(4 * (size_t)nbf);
  for (int sp = 0; sp < nbf; ++sp) {
    const int i = pt.fperm[sp];
    pt.fn[4 * sp] = B.cx[i];
    pt.fn[4 * sp + 1] = B.cy[i];
    pt.fn[4 * sp + 2] = B.cz[i];
    pt.fn[4 * sp + 3] = rad[i];
  }
  return pt;
}

// The plan of the molecules' points (device) and bases: points, boxes and
// screening on the device, two waits for the host's share (the slot offsets
// from the per-batch counts, the kept block pairs).  All molecules are numbered
// globally, molecule by molecule.  A plan takes 0.19 ms on 121 k points and 80
// functions with its buffers in place (host loops: 6.6 ms); a context's first,
// with their allocation, 1.3 ms on 687 k points and 3.4 ms on 2.07 M with 800
// functions (50 and 174 ms).
void build_plan(Ctx &c, Plan &pl, const std::vector<MolPoints> &mols,
                const std::vector<const BasisHost *> &bases, double tol) {
  hipStream_t s = c.stream;
  PlanScratch &sc = c.plan_ws;
  PlanScratch::Scope scope{sc};
  const int nmol = (int)mols.size();
  std::vector<PlanPart> parts;
  for (int m = 0; m < nmol; ++m) parts.push_back(make_part(mols[m].npts, *bases[m], tol));
  ++pl.builds;  // from here on what a captured build holds of the plan is gone
  pl.nmol = 0;  // until the plan is whole
  pl.mol_nbf_h.resize(nmol);
  pl.mol_ld_h.resize(nmol);
  pl.mol_nfb_h.resize(nmol);
  pl.mol_blk0_h.resize(nmol);
  pl.mol_b0_h.resize(nmol);
  pl.mol_nb_h.resize(nmol);
  pl.mol_npts_h.resize(nmol);
  pl.mol_P_off_h.resize(nmol);
  pl.mol_Ps_off_h.resize(nmol);
  std::vector<int64_t> ts_off(nmol), pair_off(nmol);
  int nfb = 0;
  int64_t nb = 0, ts = 0, poff = 0, psoff = 0, npts = 0, pairs = 0;
  for (int m = 0; m < nmol; ++m) {
    const PlanPart &pt = parts[m];
    pl.mol_nbf_h[m] = pt.nbf;
    pl.mol_ld_h[m] = pt.nfb * FB;
    pl.mol_nfb_h[m] = pt.nfb;
    pl.mol_blk0_h[m] = nfb;
    pl.mol_b0_h[m] = nb;
    pl.mol_nb_h[m] = pt.nb;
    pl.mol_npts_h[m] = pt.npts;
    pl.mol_P_off_h[m] = poff;
    pl.mol_Ps_off_h[m] = psoff;
    ts_off[m] = ts;
    pair_off[m] = pairs;
    nfb += pt.nfb;
    nb += pt.nb;
    ts += (int64_t)pt.nfb * pt.nb;
    pairs += (int64_t)pt.nfb * pt.nfb;
    poff += (int64_t)pt.nfb * FB * pt.nfb * FB;
    psoff += mixed_p_bytes(pt.nfb);
    npts += pt.npts;
  }
  const int64_t npad = nb * PT;

  // ---- points, boxes and live pairs --------------------------------------
  pl.px.reserve(npad);
  pl.py.reserve(npad);
  pl.pz.reserve(npad);
  pl.pw.reserve(npad);
  pl.pidx.reserve(npad);
  sc.boxes.reserve(6 * nb);
  sc.live.reserve(ts);
  sc.count.reserve(2 * nb);
  sc.pairs.reserve(pairs);
  for (int m = 0; m < nmol; ++m)
    NKX_REQUIRE(parts[m].nfb <= 0xffff, NKX_ERR_UNSUPPORTED, "more than 65535 function blocks");
  std::vector<double *> fn(nmol);
  TablePack fpack;
  for (int m = 0; m < nmol; ++m) fpack.add(fn[m], parts[m].fn.data(), parts[m].fn.size());
  fpack.upload(sc.pin_fn, sc.fn, s);
  for (int m = 0; m < nmol; ++m) {
    const PlanPart &pt = parts[m];
    const int64_t b0 = pl.mol_b0_h[m], p0 = b0 * PT;
    vk_plan_points(s, sc, pt.npts, mols[m].pts, mols[m].w, pl.px.p + p0, pl.py.p + p0,
                   pl.pz.p + p0, pl.pw.p + p0, pl.pidx.p + p0, sc.boxes.p + 6 * b0);
    vk_plan_screen(s, pt.nb, pt.nbf, pt.nfb, sc.boxes.p + 6 * b0, fn[m], sc.live.p + ts_off[m],
                   sc.count.p + 2 * b0);
  }
  sc.pin_cnt.reserve(std::max<size_t>(2 * nb, pairs) * sizeof(int));
  int *host = reinterpret_cast<int *>(sc.pin_cnt.p);
  NKX_HIP_CHECK(hipMemcpyAsync(host, sc.count.p, 2 * nb * sizeof(int), hipMemcpyDeviceToHost, s));
  NKX_HIP_CHECK(hipStreamSynchronize(s));

  // ---- slots --------------------------------------------------------------
  pl.b_off_h.resize(nb + 1);
  int64_t nslots = 0;
  double nb2g = 0, nbg = 0;
  int64_t by_pair = 0, by_super = 0, max_live = 0;
  for (int m = 0; m < nmol; ++m)
    for (int64_t b = 0; b < parts[m].nb; ++b) {
      const int64_t gb = pl.mol_b0_h[m] + b;
      pl.b_off_h[gb] = (int)nslots;
      const unsigned cnt = (unsigned)host[2 * gb];
      const int64_t n = cnt & 0xffff, f = cnt >> 17, last = (cnt >> 16) & 1;
      nslots += n;
      max_live = std::max(max_live, n);
      // algorithmic work: true functions of the live blocks, true points
      const double nfun = host[2 * gb + 1];
      const double g = (double)std::min<int64_t>(PT, parts[m].npts - b * PT);
      nb2g += nfun * nfun * g;
      nbg += nfun * g;
      // the FP64 V contraction's work in 1/200 of a pair of blocks: by pairs (on
      // the diagonal 0.55), or by super-pairs (2.65, on the diagonal 1.5, beside an
      // odd last block 1.7), whole where one block of each side is live
      by_pair += n * (100 * (n - 1) + 110);
      by_super += f * (265 * (f - 1) + 300) + last * (340 * f + 110);
    }
  NKX_REQUIRE(nslots < (int64_t)INT32_MAX, NKX_ERR_UNSUPPORTED,
              "too many live (block, batch) pairs for 32-bit slot numbers");
  pl.b_off_h[nb] = (int)nslots;
  pl.b_off.upload(pl.b_off_h.data(), pl.b_off_h.size(), s);
  pl.b_fbl.reserve(std::max<int64_t>(nslots, 1));
  pl.slot_b.reserve(std::max<int64_t>(nslots, 1));
  pl.tile_slot.reserve(std::max<int64_t>(ts, 1));
  for (int m = 0; m < nmol; ++m)
    vk_plan_fill(s, parts[m].nb, parts[m].nfb, pl.mol_blk0_h[m], pl.mol_b0_h[m],
                 sc.live.p + ts_off[m], pl.b_off.p, pl.b_fbl.p, pl.slot_b.p,
                 pl.tile_slot.p + ts_off[m], sc.pairs.p + pair_off[m]);
  NKX_HIP_CHECK(
      hipMemcpyAsync(host, sc.pairs.p, pairs * sizeof(int), hipMemcpyDeviceToHost, s));
  // the function tables meanwhile
  const int nbf_pad = nfb * FB;
  std::vector<int> fperm(nbf_pad, 0), blk_mol(nfb), blk_local(nfb);
  std::vector<FuncRec> fr(nbf_pad);
  std::vector<HarmTerm> terms;
  int nbf_total = 0;
  for (int m = 0; m < nmol; ++m) {
    const PlanPart &pt = parts[m];
    const int blk0 = pl.mol_blk0_h[m];
    const int toff = (int)terms.size();
    for (int f = 0; f < pt.nfb; ++f) {
      blk_mol[blk0 + f] = m;
      blk_local[blk0 + f] = f;
    }
    for (int i = 0; i < pt.nbf; ++i) fperm[blk0 * FB + i] = pt.fperm[i];
    for (int i = 0; i < pt.nfb * FB; ++i) {
      FuncRec r = pt.fr[i];
      r.term_off += toff;
      fr[blk0 * FB + i] = r;
    }
    terms.insert(terms.end(), pt.terms.begin(), pt.terms.end());
    nbf_total += pt.nbf;
  }
  if (terms.empty()) terms.push_back(HarmTerm{0, 0, 0, 0, 0});
  NKX_HIP_CHECK(hipStreamSynchronize(s));

  // ---- kept pairs and super-pairs: blocks (2a, 2a + 1) x (2c, 2c + 1), a <= c,
  // per molecule, kept when one of the four tiles is a kept pair ------------
  pl.pair_I_h.clear();
  pl.pair_J_h.clear();
  std::vector<int> spb, spp;
  int64_t all_pairs = 0;
  for (int m = 0; m < nmol; ++m) {
    const int blk0 = pl.mol_blk0_h[m], nf = parts[m].nfb;
    const int *live = host + pair_off[m];
    std::vector<int> pid((size_t)nf * nf, -1);
    for (int I = 0; I < nf; ++I)
      for (int J = I; J < nf; ++J)
        if (live[(size_t)I * nf + J]) {
          pid[(size_t)I * nf + J] = (int)pl.pair_I_h.size();
          pl.pair_I_h.push_back(blk0 + I);
          pl.pair_J_h.push_back(blk0 + J);
        }
    all_pairs += (int64_t)nf * (nf + 1) / 2;
    auto at = [&](int I, int J) {
      return (I < 0 || J < 0 || I > J) ? -1 : pid[(size_t)I * nf + J];
    };
    const int ns = (nf + 1) / 2;
    for (int a = 0; a < ns; ++a)
      for (int cc = a; cc < ns; ++cc) {
        const int I0 = 2 * a, I1 = 2 * a + 1 < nf ? 2 * a + 1 : -1;
        const int J0 = 2 * cc, J1 = 2 * cc + 1 < nf ? 2 * cc + 1 : -1;
        const int px[4] = {at(I0, J0), at(I0, J1), a == cc ? -1 : at(I1, J0), at(I1, J1)};
        if (px[0] < 0 && px[1] < 0 && px[2] < 0 && px[3] < 0) continue;
        spb.insert(spb.end(), {blk0 + I0, I1 >= 0 ? blk0 + I1 : -1, blk0 + J0,
                               J1 >= 0 ? blk0 + J1 : -1});
        spp.insert(spp.end(), px, px + 4);
      }
  }

  pl.nbf = nmol == 1 ? parts[0].nbf : nbf_total;
  pl.nbf_pad = nbf_pad;
  pl.nfb = nfb;
  pl.fb = FB;
  pl.npts = npts;
  pl.npts_pad = npad;
  pl.nb = nb;
  pl.nslots = nslots;
  pl.pairs_kept = nslots;
  pl.npairs = (int)pl.pair_I_h.size();
  pl.pairs_full = pl.npairs == all_pairs;
  pl.nspairs = (int)(spb.size() / 4);
  pl.v_by_pair = by_pair < by_super;
  pl.max_live = (int)max_live;
  pl.max_mol_nfb = 0;
  for (int m = 0; m < nmol; ++m) pl.max_mol_nfb = std::max(pl.max_mol_nfb, parts[m].nfb);
  pl.work_nb2g = nb2g;
  pl.work_nbg = nbg;
  pl.P_total = poff;
  pl.fperm = fperm;
  TablePack pack;
  pack.add(pl.fperm_d.p, fperm.data(), fperm.size());
  pack.add(pl.funcs.p, fr.data(), fr.size());
  pack.add(pl.terms.p, terms.data(), terms.size());
  pack.add(pl.pair_I.p, pl.pair_I_h.data(), pl.npairs);
  pack.add(pl.pair_J.p, pl.pair_J_h.data(), pl.npairs);
  pack.add(pl.sp_blk.p, spb.data(), spb.size());
  pack.add(pl.sp_pidx.p, spp.data(), spp.size());
  pack.add(pl.blk_mol.p, blk_mol.data(), nfb);
  pack.add(pl.blk_local.p, blk_local.data(), nfb);
  pack.add(pl.mol_ld.p, pl.mol_ld_h.data(), nmol);
  pack.add(pl.mol_nbf.p, pl.mol_nbf_h.data(), nmol);
  pack.add(pl.mol_nfb.p, pl.mol_nfb_h.data(), nmol);
  pack.add(pl.mol_b0.p, pl.mol_b0_h.data(), nmol);
  pack.add(pl.mol_nb.p, pl.mol_nb_h.data(), nmol);
  pack.add(pl.mol_ts_off.p, ts_off.data(), nmol);
  pack.add(pl.mol_P_off.p, pl.mol_P_off_h.data(), nmol);
  pack.add(pl.mol_Ps_off.p, pl.mol_Ps_off_h.data(), nmol);
  pack.upload(sc.pin_tab, pl.tables, s);
  NKX_HIP_CHECK(hipStreamSynchronize(s));
  pl.pt = PT;
  pl.nmol = nmol;
}

}  // namespace

void ensure_plan(Ctx &c) {
  Plan &pl = c.plan;
  NKX_REQUIRE(c.grid.npts > 0, NKX_ERR_STATE, "no grid: call nkx_make_flat_grid or nkx_set_grid");
  NKX_REQUIRE(c.basis.nbf > 0, NKX_ERR_STATE, "no basis: call nkx_set_basis");
  if (pl.grid_version == c.grid.version && pl.basis_version == c.basis_version &&
      pl.screen_tol == c.opt.screen_tol && pl.pt == PT)
    return;
  pl.pt = 0;  // until the new plan is whole
  build_plan(c, pl, {MolPoints{c.grid.npts, c.grid.pts.p, c.grid.w.p}}, {&c.basis},
             c.opt.screen_tol);
  pl.grid_version = c.grid.version;
  pl.basis_version = c.basis_version;
  pl.screen_tol = c.opt.screen_tol;
}

// Plan of a molecule set: molecule m has points mols[m] and basis bases[m].
void build_molset_plan(Ctx &c, const std::vector<MolPoints> &mols,
                       const std::vector<BasisHost> &bases) {
  std::vector<const BasisHost *> b;
  for (const BasisHost &x : bases) b.push_back(&x);
  build_plan(c, c.mplan, mols, b, c.opt.screen_tol);
  c.mplan.screen_tol = c.opt.screen_tol;
}

namespace {

// Number of slots per chunk so that the chunk's tiles fit the budget.
// cap: the ctx's tile-store budget in bytes, 0 for min(48 GB, 40 % of free).
int64_t chunk_slot_budget(size_t slot_bytes, size_t cap) {
  size_t budget = cap;
  if (budget == 0) {
    size_t freeb = 0, total = 0;
    NKX_HIP_CHECK(hipMemGetInfo(&freeb, &total));
    budget = std::min<size_t>((size_t)48 << 30, freeb / 5 * 2);
  }
  budget = std::max<size_t>(budget, (size_t)64 << 20);
  return (int64_t)(budget / slot_bytes);
}

// Split count of the V contraction over batches, or the tuned value.  One
// workgroup of a unit (super-pair; bf16, and FP64 where few super-pairs are whole:
// pair) fits a CU at a time, so:
//   one unit:  256 splits, one equal workgroup per CU (mixed benzene, 99 x 578
//              points: 1536 us per build, 1617 with 320, 1608 with 335; FP64, V
//              alone: benzene 179 us, 310 with 128, 190 with 512, a 12-atom
//              molecule with two spins 155, 143 and 178)
//   a few:     512 splits each (16- and 24-atom molecules: within 1 % of the
//              best of 32 .. 1024)
//   many:      about 8192 workgroups (FP64: 4096), the tail of unequal units
//              levelled by their number; every split costs a tile of partials
//              per pair.  By pairs 65536, of which one takes a quarter of the
//              partials: V of a chain of 240 atoms 71.4 ms with 128 splits, 73.5 with
//              64, 86.5 with 8
// and never less than four batches per split (mixed water: 146 us with 4 to 5,
// 179 with 32), or in a molecule set 16 (FP64: 8) of an average molecule (8
// molecules, mixed: 2782 us, 2893 with 4; sets of 8, 64 and 20 molecules of 2 to 30
// atoms are within 1, 2 and 1 % of the best of 1 .. 64, mixed 1, 4 and 1 %).  FP64 with more workgroups than CUs: a
// multiple of eight, which vgemm_f64 deals to the XCDs evenly, where its partials
// stay below 1 GB (by pairs 2 GB; 100 waters, 210 super-pairs: 176 ms with 24
// splits, 179 with 20; a chain of 700 atoms by super-pairs 279 ms with 8, 320 with
// 3, by pairs 235 with 8, 227 with 16).
//
// In chunks (max_slots slots each), every split reads and writes its partials
// again in each: as many workgroups per chunk as CUs (by pairs, a quarter of the
// work and of the partials each, four times as many), or, where a chunk is long,
// that times the root of its share of work (units times batches over 1743, from
// 4.7 us per batch of a super-pair and 16 us for the partials of 256, and up to
// three times that where few chunks hold all; a set's chunk holds a share of its
// units).  V contraction, mixed, ms: 32 waters in chunks of 8 GB 16.8 with 96 to
// 192 splits, 19.4 with 512, in two of 48 GB 17.4 with 203, 16.6 with 293; 24
// waters in chunks of 64 MB 3.1 with 16, 49 with 512; 60 waters in chunks of 64 MB
// 26 with 2 to 4, 230 with 106, of 1 GB 16 with 8 to 32, 25 with 106.
int choose_nsplit(const Plan &pl, int precision, int64_t max_slots, int tuned = 0) {
  const bool f64 = precision == NKX_PREC_FP64;
  const bool by_pair = precision == NKX_PREC_MIXED_BF16 || (f64 && pl.v_by_pair);
  const int64_t units = by_pair ? pl.npairs : pl.nspairs;
  if (units == 0) return 1;
  int64_t ns = tuned;
  if (tuned <= 0) {
    const int64_t per = pl.nmol > 1 ? (f64 ? 8 : 16) * (int64_t)pl.nmol : 4;
    const int64_t target = !f64 ? 8192 : by_pair ? 65536 : 4096;
    ns = std::min<int64_t>(target / units + 1, units == 1 ? 256 : 512);
    ns = std::min<int64_t>(ns, pl.nb / per);
    if (max_slots < pl.nslots) {
      const double share = (double)max_slots / pl.nslots;
      const double u = pl.nmol > 1 ? std::max(1.0, units * share) : (double)units;
      const double waves =
          std::max(1.0, (1.0 + 2.0 * share) * std::sqrt(u * share * pl.nb / 1743.0));
      ns = std::min<int64_t>(ns, (int64_t)((by_pair ? 1024.0 : 256.0) * waves / u));
    }
    if (f64 && units * ns > 256) {
      const int64_t up = (ns + 7) / 8 * 8;
      if (max_slots >= pl.nslots &&
          up * pl.npairs * FB * FB * (int64_t)sizeof(double) <= (int64_t)(by_pair ? 2 : 1) << 30)
        ns = up;
      else if (ns > 8) ns = ns / 8 * 8;
    }
  }
  ns = std::max<int64_t>(1, std::min<int64_t>(ns, pl.nb));
  return (int)ns;
}

template <typename F>
void for_each_chunk(const Plan &pl, int64_t max_slots, F &&fn) {
  int64_t b0 = 0;
  while (b0 < pl.nb) {
    int64_t b1 = b0 + 1;
    // grow while the slot range fits (at least one batch per chunk, and a
    // workgroup of 256 per batch in one launch)
    int64_t lo = b0 + 1, hi = std::min(pl.nb, b0 + max_workgroups(256));
    while (lo < hi) {
      const int64_t mid = (lo + hi + 1) / 2;
      if (pl.b_off_h[mid] - pl.b_off_h[b0] <= max_slots) lo = mid;
      else hi = mid - 1;
    }
    b1 = lo;
    fn(b0, b1, (int64_t)pl.b_off_h[b0], (int64_t)pl.b_off_h[b1]);
    b0 = b1;
  }
}

}  // namespace

namespace {
// Device table of output pointers (kept alive in the workspace until the
// build synchronises); none for as many as vk_finish takes by value.
double *const *upload_ptrs(Ctx &c, double *const *V, size_t n) {
  if (n <= (size_t)kVArgs) return nullptr;
  c.ws.vptr_h.assign(V, V + n);
  c.ws.vptr.upload(c.ws.vptr_h.data(), n, c.stream);
  return c.ws.vptr.p;
}
}  // namespace

// Sizes and workspace of one build on plan pl (allocations happen here, so a
// captured build performs none).
BuildSetup prepare_build(Workspace &ws, const Plan &pl, int nspin, bool gga, int precision,
                         int tuned_split, int tuned_group, size_t mem_cap) {
  BuildSetup b;
  b.nspin = nspin;
  // density workgroup shape: tuned, else 2 batches per workgroup (FP64) /
  // the split form with 32 rows per wave and one batch (int8 form)
  b.group = tuned_group > 0 ? tuned_group : (precision == NKX_PREC_MIXED ? 65 : 2);
  b.gga = gga;
  const int nmol = pl.nmol;
  b.narr = 1 + nspin;  // Phi, Z per spin
  b.bf16 = precision == NKX_PREC_MIXED_BF16;
  b.mixed = precision == NKX_PREC_MIXED || b.bf16;
  NKX_REQUIRE(!b.bf16 || nspin == 1, NKX_ERR_UNSUPPORTED,
              "the spin-polarised build is available in the FP64 and int8 forms");
  NKX_REQUIRE(!b.bf16 || nmol == 1, NKX_ERR_UNSUPPORTED,
              "the split-bf16 form builds one molecule at a time");
  const size_t slot_bytes = b.bf16    ? (size_t)bf16_slot_bytes(gga ? 1 : 0)
                            : b.mixed ? (size_t)mixed_slot_bytes(gga ? 1 : 0)
                                      : (size_t)b.narr * FB * PT * sizeof(double);
  // per slot beyond the tile store: density partials per spin and (int8 form)
  // the second spin's Z section
  const size_t slot_extra =
      b.bf16 ? 0
             : (size_t)nspin * 4 * PT * sizeof(double) +
                   (b.mixed && nspin == 2 ? (size_t)mixed_zsection_bytes() : 0);
  int64_t max_slots = chunk_slot_budget(slot_bytes + slot_extra, mem_cap);
  // at least the largest single batch
  for (int64_t bb = 0; bb < pl.nb; ++bb)
    max_slots = std::max<int64_t>(max_slots, pl.b_off_h[bb + 1] - pl.b_off_h[bb]);
  b.slots_alloc = std::min<int64_t>(max_slots, std::max<int64_t>(pl.nslots, 1));
  b.nsplit = choose_nsplit(pl, precision, b.slots_alloc, tuned_split);
  if (b.mixed) {
    ws.mstore.reserve((size_t)b.slots_alloc * slot_bytes);
    if (!b.bf16 && nspin == 2)
      ws.zstore_b.reserve((size_t)b.slots_alloc * mixed_zsection_bytes());
    int64_t psb = 0;
    for (int m = 0; m < nmol; ++m) psb += mixed_p_bytes(pl.mol_nfb_h[m]);
    b.psb = psb;
    ws.Ps.reserve(b.bf16 ? (size_t)6 * pl.nbf_pad * pl.nbf_pad : (size_t)nspin * psb);
  } else {
    ws.tiles64.reserve((size_t)b.slots_alloc * b.narr * FB * PT);
    ws.Pd.reserve((size_t)nspin * pl.P_total);
  }
  if (!b.bf16) ws.dpart.reserve((size_t)nspin * b.slots_alloc * 4 * PT);
  ws.coef.reserve((size_t)4 * nspin * pl.npts_pad);
  ws.blockEN.reserve((size_t)3 * pl.nb);
  b.vsz = (size_t)b.nsplit * std::max(pl.npairs, 1) * FB * FB;
  ws.vpart.reserve(nspin * b.vsz);
  return b;
}

// The functional of the FP64 form from the density partials of one chunk.
static void fp64_functional(hipStream_t s, int nspin, int64_t b0, int64_t b1, int64_t s0,
                            const Plan &pl, int gga, const XcList &xl, Workspace &ws,
                            int64_t slots_alloc, double *epoint) {
  if (nspin == 2)
    vkm_density_finish_pol(s, b0, b1, s0, pl, gga, nullptr, nullptr, xl, ws.coef.p,
                           ws.coef.p + (size_t)4 * pl.npts_pad, ws.blockEN.p, ws.dpart.p,
                           ws.dpart.p + (size_t)slots_alloc * 4 * PT, epoint);
  else
    vkm_density_functional(s, b0, b1, s0, pl, gga, xl, ws.coef.p, ws.blockEN.p, ws.dpart.p,
                           epoint);
}

// Every launch of one build, stream-ordered; the last one writes the (E, N_alpha,
// N_beta) triples of all molecules into en_dst (page-locked).  No
// allocation, no memset, no synchronisation: the sequence can be captured.
void enqueue_build(Ctx &c, Workspace &ws, const Plan &pl, const BuildSetup &b,
                   const double *const *P, const XcList &xl, double *const *V,
                   double *const *Vtab, double *en_dst) {
  hipStream_t s = c.stream;
  const int nmol = pl.nmol, nspin = b.nspin, narr = b.narr, nsplit = b.nsplit;
  const bool bf16 = b.bf16, mixed = b.mixed;
  const size_t vsz = b.vsz;
  Timing &tm = c.timing;
  const int t_build = tm.begin(kStageBuild, s);
  int t = tm.begin(kStageFinal, s);
  uint16_t *bstore = reinterpret_cast<uint16_t *>(ws.mstore.p);
  uint16_t *bPs = reinterpret_cast<uint16_t *>(ws.Ps.p);
  std::vector<GatherP> gp;
  for (int sp = 0; sp < nspin; ++sp)
    for (int m = 0; m < nmol; ++m) {
      const double *Pm = P[(size_t)sp * nmol + m];
      const int nbf = pl.mol_nbf_h[m];
      const int *fp = pl.fperm_d.p + (size_t)pl.mol_blk0_h[m] * FB;
      if (bf16)
        vkb_gather_p(s, nbf, pl.nfb, fp, Pm, bPs);
      else
        gp.push_back({Pm, fp,
                      mixed ? (void *)(ws.Ps.p + (size_t)sp * b.psb + pl.mol_Ps_off_h[m])
                            : (void *)(ws.Pd.p + (size_t)sp * pl.P_total + pl.mol_P_off_h[m]),
                      nbf, pl.mol_nfb_h[m]});
      // the elements of block pairs without a common batch are never written
      if (!pl.pairs_full) vk_fill0(s, V[(size_t)sp * nmol + m], (int64_t)nbf * nbf);
    }
  if (mixed && !bf16)
    vkm_gather_p(s, gp);
  else
    vk_gather_p(s, gp, true);
  tm.end(t, s);
  for_each_chunk(pl, b.slots_alloc, [&](int64_t b0, int64_t b1, int64_t s0, int64_t s1) {
    const int ig = b.gga ? 1 : 0;
    const bool first = b0 == 0;  // the V partials are written, then added to
    int tt = tm.begin(kStageColloc, s);
    if (bf16)
      vkb_colloc(s, s0, s1, pl, ig, bstore);
    else if (mixed) {
      vkm_colloc(s, s0, s1, pl, ig, ws.mstore.p);
      vkm_pm_group(s, b0, b1, s0, pl, ig, ws.mstore.p);
    } else
      vk_colloc(s, s0, s1, pl, narr, ws.tiles64.p);
    tm.end(tt, s);
    tt = tm.begin(kStageDensity, s);
    if (bf16)
      vkb_density(s, 6, b0, b1, s0, pl, bPs, ig, bstore, xl, ws.coef.p, ws.blockEN.p);
    else if (mixed)
      for (int sp = 0; sp < nspin; ++sp)  // one contraction per spin
        vkm_density(s, b.group, b0, b1, s0, pl, ws.Ps.p + (size_t)sp * b.psb, ig,
                    ws.mstore.p, xl, ws.coef.p, ws.blockEN.p,
                    ws.dpart.p + (size_t)sp * b.slots_alloc * 4 * PT);
    else
      vk_density(s, nspin, b.group, b0, b1, s0, pl, ws.Pd.p, narr, ig, ws.tiles64.p, ws.dpart.p,
                 b.slots_alloc * 4 * PT);
    tm.end(tt, s);
    if (!bf16) {
      tt = tm.begin(kStageZ, s);
      if (!mixed) {
        fp64_functional(s, nspin, b0, b1, s0, pl, ig, xl, ws, b.slots_alloc, nullptr);
        vk_z_slots(s, s0, s1, pl, narr, nspin, ig, 1.0, ws.coef.p, ws.tiles64.p);
      } else if (nspin == 2)
        vkm_density_finish_pol(s, b0, b1, s0, pl, ig, ws.mstore.p, ws.zstore_b.p, xl,
                               ws.coef.p, ws.coef.p + (size_t)4 * pl.npts_pad, ws.blockEN.p,
                               ws.dpart.p, ws.dpart.p + (size_t)b.slots_alloc * 4 * PT);
      else
        vkm_density_finish(s, b0, b1, s0, pl, ig, ws.mstore.p, xl, ws.coef.p,
                           ws.blockEN.p, ws.dpart.p);
      tm.end(tt, s);
    }
    tt = tm.begin(kStageVgemm, s);
    if (bf16)
      vkb_vgemm(s, 6, b0, b1, s0, pl, nsplit, ig, first, bstore, ws.vpart.p);
    else if (mixed) {
      vkm_vgemm(s, b0, b1, s0, pl, nsplit, ig, first, ws.mstore.p, ws.vpart.p);
      if (nspin == 2)
        vkm_vgemm(s, b0, b1, s0, pl, nsplit, ig, first, ws.mstore.p, ws.vpart.p + vsz,
                  ws.zstore_b.p);
    }
    else
      vk_vgemm(s, b0, b1, s0, pl, nsplit, narr, nspin, first, ws.tiles64.p, ws.vpart.p);
    tm.end(tt, s);
  });
  t = tm.begin(kStageFinal, s);
  vk_finish(s, pl, nsplit, nspin, ws.vpart.p, V, Vtab, ws.blockEN.p, en_dst);
  tm.end(t, s);
  tm.end(t_build, s);
}

// One V_xc build on plan pl.  Molecule m, spin sp: density matrix
// P[sp * nmol + m] and potential V[sp * nmol + m] (device, nbf_m x nbf_m,
// row-major); E[m] and N[m * nspin + sp] on return.  nspin = 2 is FP64 only.
void build_on_plan(Ctx &c, Plan &pl, int nspin, const double *const *P, const XcList &xl,
                   bool gga, int precision, double *E, double *N, double *const *V) {
  const int nmol = pl.nmol;
  const BuildSetup b =
      prepare_build(c.ws, pl, nspin, gga, precision, c.opt.vgemm_split, c.opt.density_group,
                    c.opt.mem_budget);
  double *const *Vtab = upload_ptrs(c, V, (size_t)nspin * nmol);
  double *en = c.out_doubles((size_t)3 * nmol);
  enqueue_build(c, c.ws, pl, b, P, xl, V, Vtab, en);
  NKX_HIP_CHECK(hipStreamSynchronize(c.stream));
  c.timing.collect();
  c.work.flops_density = 2.0 * nspin * pl.work_nb2g;
  c.work.flops_v = 2.0 * nspin * pl.work_nb2g;
  c.work.colloc_elems = pl.work_nbg;
  for (int m = 0; m < nmol; ++m) {
    E[m] = en[3 * m];
    for (int sp = 0; sp < nspin; ++sp) N[(size_t)m * nspin + sp] = en[3 * m + 1 + sp];
  }
}

// ---- autotuner ------------------------------------------------------------
// Times one build per candidate (after one untimed build): first the batches
// per density workgroup (1, 2, 4), then the split count of the V contraction
// (1/4 .. 4 x the automatic choice), and keeps the fastest in the ctx options.
namespace {
// Times each candidate on plan pl (build() runs one build with the ctx
// options): first the density shape, then the V split count; keeps the
// fastest pair in the ctx options and returns its build time.
double autotune_on(Ctx &c, const Plan &pl, int precision, bool gga,
                   const std::function<void()> &build,
                   int *best_split, int *best_group) {
  const int base = prepare_build(c.ws, pl, 1, gga, precision, 0, 0, c.opt.mem_budget).nsplit;
  std::vector<int> splits;
  for (int k : {base / 4, base / 2, base, 2 * base, 4 * base}) {
    const int v = std::max(1, std::min<int>(k, (int)std::max<int64_t>(pl.nb, 1)));
    if (std::find(splits.begin(), splits.end(), v) == splits.end()) splits.push_back(v);
  }
  const bool bf16 = precision == NKX_PREC_MIXED_BF16;  // one batch per workgroup
  hipEvent_t a, b;
  NKX_HIP_CHECK(hipEventCreate(&a));
  NKX_HIP_CHECK(hipEventCreate(&b));
  const int saved_split = c.opt.vgemm_split, saved_group = c.opt.density_group;
  const bool timing = c.timing.on;
  c.timing.on = false;
  // the faster of two builds per candidate (one build alone is noisy at the
  // few-percent level that separates neighbouring split counts)
  auto timed = [&]() {
    double best_ms = 1e300;
    for (int rep = 0; rep < 2; ++rep) {
      NKX_HIP_CHECK(hipEventRecord(a, c.stream));
      build();
      NKX_HIP_CHECK(hipEventRecord(b, c.stream));
      NKX_HIP_CHECK(hipEventSynchronize(b));
      float ms = 0.f;
      NKX_HIP_CHECK(hipEventElapsedTime(&ms, a, b));
      best_ms = std::min(best_ms, (double)ms);
    }
    return best_ms;
  };
  double best = 1e300;
  try {
    c.opt.vgemm_split = base;
    build();  // warm caches and workspace
    int best_g = bf16 ? 1 : (precision == NKX_PREC_MIXED ? 65 : 2);
    // density shapes: point batches (64, 128 or 256 points) per workgroup
    // in the FP64 form; in the int8 form 65 (one batch) and 71 (one batch,
    // absolute block pairs in XCD tiles) -- 66 and 72 (two batches, 8 x 8
    // tiles) are never the fastest on large grids and are not timed
    const std::vector<int> shapes =
        precision == NKX_PREC_MIXED ? std::vector<int>{65, 71}
                                    : std::vector<int>{1, 2, 4};
    if (!bf16)
      for (int g : shapes) {
        c.opt.density_group = g;
        const double ms = timed();
        if (ms < best) {
          best = ms;
          best_g = g;
        }
      }
    c.opt.density_group = best_g;
    int best_k = base;
    best = 1e300;
    for (int k : splits) {
      c.opt.vgemm_split = k;
      const double ms = timed();
      if (ms < best) {
        best = ms;
        best_k = k;
      }
    }
    c.opt.vgemm_split = best_k;
    if (best_split) *best_split = best_k;
    if (best_group) *best_group = best_g;
  } catch (...) {
    c.opt.vgemm_split = saved_split;
    c.opt.density_group = saved_group;
    c.timing.on = timing;
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    throw;
  }
  c.timing.on = timing;
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  return best;
}
}  // namespace

double autotune(Ctx &c, const double *P, const XcList &xl, bool gga, int precision, double *V,
                int *best_split, int *best_group) {
  ensure_plan(c);
  double E, N;
  return autotune_on(
      c, c.plan, precision, gga, [&]() { vxc_build(c, P, xl, gga, precision, &E, &N, V); },
      best_split, best_group);
}

double molset_autotune(Ctx &c, const double *const *P, const XcList &xl, bool gga,
                       int precision, double *const *V, int *best_split, int *best_group) {
  NKX_REQUIRE(c.mplan.nmol > 0, NKX_ERR_STATE, "no molecule set: call nkx_molset_create");
  std::vector<double> E(c.mplan.nmol), N(c.mplan.nmol);
  return autotune_on(
      c, c.mplan, precision, gga,
      [&]() { build_on_plan(c, c.mplan, 1, P, xl, gga, precision, E.data(), N.data(), V); },
      best_split, best_group);
}

// ---- HIP graph of one build on the ctx grid and basis ----------------------
namespace {
// Capture one build on plan pl (nmol molecules: P[m], V[m]) into c.graph.
void capture_on_plan(Ctx &c, Plan &pl, int nspin, const double *const *P, const XcList &xl,
                     bool gga, int precision, double *const *V) {
  GraphState &gs = c.graph;
  gs.release();
  const int nmol = pl.nmol;
  const BuildSetup b =
      prepare_build(gs.ws, pl, nspin, gga, precision, c.opt.vgemm_split, c.opt.density_group,
                    c.opt.mem_budget);
  NKX_HIP_CHECK(hipHostMalloc(reinterpret_cast<void **>(&gs.en_pinned),
                              3 * (size_t)nmol * sizeof(double), hipHostMallocDefault));
  gs.nmol = nmol;
  gs.nspin = nspin;
  gs.vtab_h.assign(V, V + (size_t)nspin * nmol);
  gs.vtab.upload(gs.vtab_h.data(), (size_t)nspin * nmol, c.stream);
  NKX_HIP_CHECK(hipStreamSynchronize(c.stream));
  const bool timing = c.timing.on;
  c.timing.on = false;  // no event records inside the graph
  NKX_HIP_CHECK(hipStreamBeginCapture(c.stream, hipStreamCaptureModeThreadLocal));
  try {
    enqueue_build(c, gs.ws, pl, b, P, xl, V, gs.vtab.p, gs.en_pinned);
  } catch (...) {
    hipGraph_t broken = nullptr;
    (void)hipStreamEndCapture(c.stream, &broken);
    if (broken) (void)hipGraphDestroy(broken);
    c.timing.on = timing;
    throw;
  }
  c.timing.on = timing;
  NKX_HIP_CHECK(hipStreamEndCapture(c.stream, &gs.graph));
  NKX_HIP_CHECK(hipGraphInstantiate(&gs.exec, gs.graph, nullptr, nullptr, 0));
}
}  // namespace

void graph_capture(Ctx &c, int nspin, const double *const *P, const XcList &xl, bool gga,
                   int precision, double *const *V) {
  ensure_plan(c);
  capture_on_plan(c, c.plan, nspin, P, xl, gga, precision, V);
  GraphState &gs = c.graph;
  gs.molset = false;
  gs.plan_builds = c.plan.builds;
  gs.grid_version = c.grid.version;
  gs.basis_version = c.basis_version;
  gs.screen_tol = c.opt.screen_tol;
}

void molset_graph_capture(Ctx &c, const double *const *P, const XcList &xl, bool gga,
                          int precision, double *const *V) {
  NKX_REQUIRE(c.mplan.nmol > 0, NKX_ERR_STATE, "no molecule set: call nkx_molset_create");
  capture_on_plan(c, c.mplan, 1, P, xl, gga, precision, V);
  GraphState &gs = c.graph;
  gs.molset = true;
  gs.plan_builds = c.mplan.builds;
  gs.screen_tol = c.mplan.screen_tol;
}

// Replay the captured build; E[m], N[m] for each molecule of the capture
// (an open-shell capture: E[0], N[0] = N_alpha, N[1] = N_beta).
void graph_launch(Ctx &c, double *E, double *N) {
  GraphState &gs = c.graph;
  NKX_REQUIRE(gs.exec, NKX_ERR_STATE, "no captured build: call nkx_graph_capture");
  if (gs.molset)
    NKX_REQUIRE(gs.plan_builds == c.mplan.builds, NKX_ERR_STATE,
                "the molecule set changed since the capture");
  else
    // the count too: the settings may be those of the capture again and the plan
    // one of others made in between
    NKX_REQUIRE(gs.grid_version == c.grid.version && gs.basis_version == c.basis_version &&
                    gs.screen_tol == c.opt.screen_tol && gs.plan_builds == c.plan.builds,
                NKX_ERR_STATE, "grid, basis or screening changed since the capture");
  NKX_HIP_CHECK(hipGraphLaunch(gs.exec, c.stream));
  NKX_HIP_CHECK(hipStreamSynchronize(c.stream));
  if (gs.nspin == 2) {
    E[0] = gs.en_pinned[0];
    if (N) {
      N[0] = gs.en_pinned[1];
      N[1] = gs.en_pinned[2];
    }
    return;
  }
  for (int m = 0; m < gs.nmol; ++m) {
    E[m] = gs.en_pinned[3 * m];
    if (N) N[m] = gs.en_pinned[3 * m + 1];
  }
}

void GraphState::release() {
  if (exec) (void)hipGraphExecDestroy(exec);
  if (graph) (void)hipGraphDestroy(graph);
  if (en_pinned) (void)hipHostFree(en_pinned);
  exec = nullptr;
  graph = nullptr;
  en_pinned = nullptr;
}

// One V_xc build on the ctx grid and basis.  nspin = 1: P[0] is the total
// density matrix; nspin = 2: P[0], P[1] the spin density matrices.
void vxc_build_spin(Ctx &c, int nspin, const double *const *P, const XcList &xl, bool gga,
                    int precision, double *E, double *N, double *const *V) {
  ensure_plan(c);
  build_on_plan(c, c.plan, nspin, P, xl, gga, precision, E, N, V);
}

void vxc_build(Ctx &c, const double *P, const XcList &xl, bool gga, int precision, double *E,
               double *N, double *V) {
  vxc_build_spin(c, 1, &P, xl, gga, precision, E, N, &V);
}

// Nuclear gradient of E_xc at fixed P (kernels_grad.hip).  nspin = 1: P[0]
// is the total density matrix; nspin = 2: P[0], P[1] the spin density
// matrices.  Every basis function must sit on an atom of the grid; grad is
// host memory, 3 natoms.
void xc_grad(Ctx &c, int nspin, const double *const *P, const XcList &xl, bool gga,
             int partition, bool mixed, double *E, double *grad) {
  ensure_plan(c);
  Plan &pl = c.plan;
  Workspace &ws = c.ws;
  hipStream_t s = c.stream;
  const int natoms = c.grid.natoms;
  NKX_REQUIRE(natoms > 0 && natoms <= 2048, NKX_ERR_UNSUPPORTED,
              "the gradient supports 1 .. 2048 atoms");
  NKX_REQUIRE(partition >= 0 && partition <= 2, NKX_ERR_INVALID_ARGUMENT,
              "partition: 0 fixed weights, 1 capped Becke, 2 Becke");
  NKX_REQUIRE(nspin == 1 || nspin == 2, NKX_ERR_NSPIN, "nspin must be 1 or 2");
  // function (sorted order) -> atom
  std::vector<int> fatom(pl.nbf, -1);
  for (int sp = 0; sp < pl.nbf; ++sp) {
    const int i = pl.fperm[sp];
    const double ctr[3] = {c.basis.cx[i], c.basis.cy[i], c.basis.cz[i]};
    for (int a = 0; a < natoms && fatom[sp] < 0; ++a) {
      double d2 = 0.0;
      for (int k = 0; k < 3; ++k) d2 += std::pow(ctr[k] - c.grid.centers_host[3 * a + k], 2);
      if (d2 <= 1e-20) fatom[sp] = a;
    }
    NKX_REQUIRE(fatom[sp] >= 0, NKX_ERR_INVALID_ARGUMENT,
                "basis function " + std::to_string(i) + " is not centred on an atom of the grid");
  }
  NKX_REQUIRE(pl.nmol == 1, NKX_ERR_STATE, "the gradient runs on the ctx grid and basis");
  const int narr = 1 + nspin;  // Phi, Z per spin
  // FP64: the tile arrays; mixed: the int8 slot (sections and FP32 grad Phi),
  // the second spin's Y sections and the density partials; both plus the
  // per-slot gradient partials
  const size_t slot_bytes =
      mixed ? (size_t)mixed_slot_bytes(gga ? 1 : 0) + (size_t)nspin * 4 * PT * sizeof(double) +
                  (nspin == 2 ? (size_t)mixed_zsection_bytes() : 0)
            : ((size_t)narr * FB * PT + (size_t)nspin * 4 * PT) * sizeof(double);
  int64_t max_slots =
      chunk_slot_budget(slot_bytes + 3 * FB * sizeof(double), c.opt.mem_budget);
  for (int64_t b = 0; b < pl.nb; ++b)
    max_slots = std::max<int64_t>(max_slots, pl.b_off_h[b + 1] - pl.b_off_h[b]);
  const int64_t slots_alloc = std::min<int64_t>(max_slots, std::max<int64_t>(pl.nslots, 1));
  const int nseg = 32;
  // one-wave workgroups of the weight-derivative kernel: one wave of points
  // each up to 16384 workgroups, so that the dispatcher balances waves of
  // unequal cost (points near many atoms cost more); fewer for large
  // molecules, so that the per-workgroup partials stay within 2^25 doubles
  const int64_t nblk_cap =
      std::max<int64_t>(1024, ((int64_t)1 << 25) / std::max<int64_t>(3 * (int64_t)natoms, 1));
  const int nblk = (int)std::min<int64_t>(std::max<int64_t>(pl.npts_pad / 64, 1),
                                          std::min<int64_t>(16384, nblk_cap));
  const size_t psb = (size_t)mixed_p_bytes(pl.mol_nfb_h[0]);
  const size_t dsz = (size_t)slots_alloc * 4 * PT;
  if (mixed) {
    ws.mstore.reserve((size_t)slots_alloc * mixed_slot_bytes(gga ? 1 : 0));
    ws.Ps.reserve(nspin * psb);
    if (nspin == 2) ws.zstore_b.reserve((size_t)slots_alloc * mixed_zsection_bytes());
  } else {
    ws.tiles64.reserve((size_t)slots_alloc * narr * FB * PT);
    ws.Pd.reserve((size_t)nspin * pl.P_total);
  }
  ws.dpart.reserve(nspin * dsz);
  ws.coef.reserve((size_t)4 * nspin * pl.npts_pad);
  ws.blockEN.reserve((size_t)3 * pl.nb);
  // gradient buffers: ptab, epoint, tpt, cpart, gacc, wpart
  const size_t n_ep = pl.npts_pad, n_tp = 3 * pl.npts_pad, n_cp = (size_t)slots_alloc * 3 * FB;
  const size_t n_ga = (size_t)nseg * pl.nbf_pad * 3, n_gf = (size_t)pl.nbf_pad * 3;
  const size_t n_wp = (size_t)nblk * 3 * natoms, n_ws = (size_t)3 * natoms;
  // atom-pair table first, rounded to 256 bytes, so the others keep the
  // alignment of the allocation
  const size_t n_pt = ((size_t)2 * natoms * natoms + 31) & ~(size_t)31;
  ws.gbuf.reserve(n_pt + n_ep + n_tp + n_cp + n_ga + n_wp);
  double *ptab = ws.gbuf.p, *epoint = ptab + n_pt, *tpt = epoint + n_ep, *cpart = tpt + n_tp,
         *gacc = cpart + n_cp, *wpart = gacc + n_ga;
  // the results, page-locked: E, N; sums per atom; sums per function
  double *en = c.out_doubles(3 + n_ws + n_gf), *wsum = en + 3, *gfun = wsum + n_ws;
  ws.gint.reserve(pl.npts_pad);

  std::vector<GatherP> gp;
  for (int sp = 0; sp < nspin; ++sp)
    gp.push_back({P[sp], pl.fperm_d.p,
                  mixed ? (void *)(ws.Ps.p + sp * psb) : (void *)(ws.Pd.p + (size_t)sp * pl.P_total),
                  pl.nbf, pl.mol_nfb_h[0]});
  if (mixed)
    vkm_gather_p(s, gp);
  else
    vk_gather_p(s, gp, true);
  vk_fill0(s, gacc, (int64_t)n_ga);
  const int ig = gga ? 1 : 0;
  double *coef_b = ws.coef.p + (size_t)4 * pl.npts_pad;
  for_each_chunk(pl, slots_alloc, [&](int64_t b0, int64_t b1, int64_t s0, int64_t s1) {
    if (mixed) {
      // density by the split form (contraction per spin, then the functional
      // with w e per point), Y slices (the first spin's over the Z sections),
      // then the basis-centre term per spin
      vkm_colloc(s, s0, s1, pl, ig, ws.mstore.p);
      vkm_pm_group(s, b0, b1, s0, pl, ig, ws.mstore.p);
      for (int sp = 0; sp < nspin; ++sp)
        vkm_density(s, 65, b0, b1, s0, pl, ws.Ps.p + sp * psb, ig, ws.mstore.p, xl, ws.coef.p,
                    ws.blockEN.p, ws.dpart.p + sp * dsz);
      if (nspin == 1) {
        vkm_density_functional(s, b0, b1, s0, pl, ig, xl, ws.coef.p, ws.blockEN.p, ws.dpart.p,
                               epoint);
      } else {
        vkm_density_finish_pol(s, b0, b1, s0, pl, ig, nullptr, nullptr, xl, ws.coef.p, coef_b,
                               ws.blockEN.p, ws.dpart.p, ws.dpart.p + dsz, epoint);
        vkgm_y_slots(s, s0, s1, pl, ig, coef_b, ws.mstore.p, ws.zstore_b.p);
      }
      vkgm_y_slots(s, s0, s1, pl, ig, ws.coef.p, ws.mstore.p);
      vkgm_basis(s, b0, b1, s0, pl, ws.Ps.p, ig, ws.mstore.p, ws.coef.p, nullptr, false, cpart,
                 tpt);
      vkg_fold(s, b0, b1, s0, pl, nseg, cpart, gacc);
      if (nspin == 2) {
        vkgm_basis(s, b0, b1, s0, pl, ws.Ps.p + psb, ig, ws.mstore.p, coef_b, ws.zstore_b.p,
                   true, cpart, tpt);
        vkg_fold(s, b0, b1, s0, pl, nseg, cpart, gacc);
      }
    } else {
      vk_colloc(s, s0, s1, pl, narr, ws.tiles64.p);
      vk_density(s, nspin, 2, b0, b1, s0, pl, ws.Pd.p, narr, ig, ws.tiles64.p, ws.dpart.p,
                 (int64_t)dsz);
      fp64_functional(s, nspin, b0, b1, s0, pl, ig, xl, ws, slots_alloc, epoint);
      vk_z_slots(s, s0, s1, pl, narr, nspin, ig, 2.0, ws.coef.p, ws.tiles64.p);
      // (the density partials are done with: scratch of the point sums)
      for (int sp = 0; sp < nspin; ++sp) {
        vkg_basis(s, b0, b1, s0, pl, ws.Pd.p + (size_t)sp * pl.P_total, narr, narr - nspin + sp,
                  ig, ws.tiles64.p, ws.coef.p + (size_t)4 * sp * pl.npts_pad, sp > 0, cpart,
                  ws.dpart.p, tpt);
        vkg_fold(s, b0, b1, s0, pl, nseg, cpart, gacc);
      }
    }
  });
  vkg_colsum(s, nseg, pl.nbf_pad * 3, gacc, gfun);
  vk_en_reduce(s, pl, ws.blockEN.p, en);
  vkg_owners(s, pl, c.grid.owner.p, ws.gint.p);
  vkg_weights(s, pl, natoms, c.grid.centers.p, ws.gint.p, epoint, tpt, partition, nblk, ptab,
              wpart);
  vkg_colsum(s, nblk, 3 * natoms, wpart, wsum);
  NKX_HIP_CHECK(hipStreamSynchronize(s));
  for (int k = 0; k < 3 * natoms; ++k) grad[k] = wsum[k];
  for (int sp = 0; sp < pl.nbf; ++sp)
    for (int k = 0; k < 3; ++k) grad[3 * fatom[sp] + k] += gfun[3 * sp + k];
  *E = en[0];
}

// rho, grad rho and sigma of P at every grid point, in the grid's order: the
// FP64 batched density with an empty functional list, then a scatter through
// the point permutation.  Stream-ordered; outputs other than rho may be NULL.
void density_points(Ctx &c, const double *P, double *rho, double *gx, double *gy, double *gz,
                    double *sigma) {
  ensure_plan(c);
  Plan &pl = c.plan;
  NKX_REQUIRE(pl.nmol == 1, NKX_ERR_STATE, "the per-point density runs on the ctx grid and basis");
  Workspace &ws = c.ws;
  hipStream_t s = c.stream;
  const int narr = 1;  // Phi
  int64_t max_slots =
      chunk_slot_budget(((size_t)narr * FB * PT + 4 * PT) * sizeof(double), c.opt.mem_budget);
  for (int64_t b = 0; b < pl.nb; ++b)
    max_slots = std::max<int64_t>(max_slots, pl.b_off_h[b + 1] - pl.b_off_h[b]);
  const int64_t slots_alloc = std::min<int64_t>(max_slots, std::max<int64_t>(pl.nslots, 1));
  ws.tiles64.reserve((size_t)slots_alloc * narr * FB * PT);
  ws.dpart.reserve((size_t)slots_alloc * 4 * PT);
  ws.Pd.reserve((size_t)pl.P_total);
  ws.coef.reserve((size_t)4 * pl.npts_pad);
  ws.blockEN.reserve((size_t)3 * pl.nb);
  ws.gbuf.reserve((size_t)4 * pl.npts_pad);
  XcList none{};
  none.n = 0;
  vk_gather_p(s, {{P, pl.fperm_d.p, ws.Pd.p, pl.nbf, pl.mol_nfb_h[0]}}, true);
  for_each_chunk(pl, slots_alloc, [&](int64_t b0, int64_t b1, int64_t s0, int64_t s1) {
    vk_colloc(s, s0, s1, pl, narr, ws.tiles64.p);
    vk_density(s, 1, 2, b0, b1, s0, pl, ws.Pd.p, narr, 1, ws.tiles64.p, ws.dpart.p, 0);
    vkm_density_functional(s, b0, b1, s0, pl, 1, none, ws.coef.p, ws.blockEN.p, ws.dpart.p,
                           nullptr, ws.gbuf.p);
  });
  vk_scatter_density(s, pl, ws.gbuf.p, rho, gx, gy, gz, sigma);
}

int Timing::begin(int stage, hipStream_t s) {
  if (!on) return -1;
  const size_t k = pending_stage.size();
  if (k >= pool.size()) {
    hipEvent_t a, b;
    NKX_HIP_CHECK(hipEventCreate(&a));
    NKX_HIP_CHECK(hipEventCreate(&b));
    pool.emplace_back(a, b);
  }
  pending_stage.push_back(stage);
  NKX_HIP_CHECK(hipEventRecord(pool[k].first, s));
  return (int)k;
}

void Timing::end(int slot, hipStream_t s) {
  if (slot < 0) return;
  NKX_HIP_CHECK(hipEventRecord(pool[slot].second, s));
}

void Timing::collect() {
  for (size_t k = 0; k < pending_stage.size(); ++k) {
    float ms_k = 0.f;
    NKX_HIP_CHECK(hipEventElapsedTime(&ms_k, pool[k].first, pool[k].second));
    ms[pending_stage[k]] += ms_k;
    launches[pending_stage[k]] += 1;
  }
  pending_stage.clear();
}

void Timing::release() {
  for (auto &e : pool) {
    (void)hipEventDestroy(e.first);
    (void)hipEventDestroy(e.second);
  }
  pool.clear();
  pending_stage.clear();
}

void overlap_build(Ctx &c, double *S) {
  ensure_plan(c);
  Plan &pl = c.plan;
  Workspace &ws = c.ws;
  hipStream_t s = c.stream;
  const int narr = 2;
  int64_t max_slots =
      chunk_slot_budget((size_t)narr * FB * PT * sizeof(double), c.opt.mem_budget);
  for (int64_t b = 0; b < pl.nb; ++b)
    max_slots = std::max<int64_t>(max_slots, pl.b_off_h[b + 1] - pl.b_off_h[b]);
  const int64_t slots_alloc = std::min<int64_t>(max_slots, std::max<int64_t>(pl.nslots, 1));
  ws.tiles64.reserve((size_t)slots_alloc * narr * FB * PT);
  const int nsplit = choose_nsplit(pl, NKX_PREC_FP64, slots_alloc);
  const size_t vsz = (size_t)nsplit * std::max(pl.npairs, 1) * FB * FB;
  ws.vpart.reserve(vsz);
  vk_fill0(s, S, (int64_t)pl.nbf * pl.nbf);
  for_each_chunk(pl, slots_alloc, [&](int64_t b0, int64_t b1, int64_t s0, int64_t s1) {
    vk_colloc(s, s0, s1, pl, narr, ws.tiles64.p);
    vk_zoverlap(s, s0, s1, pl, narr, ws.tiles64.p);
    vk_vgemm(s, b0, b1, s0, pl, nsplit, narr, 1, b0 == 0, ws.tiles64.p, ws.vpart.p);
  });
  vk_finish(s, pl, nsplit, 1, ws.vpart.p, &S, nullptr, nullptr, nullptr);
  NKX_HIP_CHECK(hipStreamSynchronize(s));
}

}  // namespace nkx
