// Work-group level evaluation of one molecule's intermolecular energy at its
// current and (optionally) proposed position, in one pass over candidates.
//
// Preparation (wave 0): the neighbour source -- every molecule, the occupied
// slots of the cells spanning the old and proposed cell, or the Verlet list.
// Candidate scan (all lanes): each lane takes one candidate j a pass, tests the
// primary-site cutoff at the old and proposed position (SimulationStep.cpp:
// 317-330), and the hits of a round of passes are compacted into LDS in
// candidate order (ballot + mbcnt, two barriers a round).
// Pair phase (pair_phase): every (hit, site b) of the hits is one item, 64
// items a block, one lane an item; the block's lanes sum their site b with
// the moving molecule's sites a one after another (BruteForceStep.cpp:48-79),
// and the (block, site a) steps are dealt to the waves in equal runs.  Sums
// are FP64; per-wave DPP sums and a fixed-order sum over waves end the
// evaluation, so results are deterministic for a given work-group size.
#pragma once

#include "device_common.h"
#include "scan_items.h"
#include "wave.h"

namespace mcgpu {

// A real site of the moving molecule as the pair phase reads it (the same
// address in every lane: LDS broadcasts): old and proposed position and pair
// parameters.
struct alignas(16) MoveSite {
  double xo, yo, zo, xn, yn, zn;
  double s, e, q;
  float s32, e32;  // FP32 forms; sigma 0 without an LJ term (see mixed_item)
};

// A hit: an in-range molecule of the current evaluation.  x: first site; y:
// site count (6 bits), in range of the old (1 << 6) and of the proposed
// (1 << 7) position, the periodic image of its pairs per axis (3 bits from
// bit 8, 11 and 14: 0 none, 1 minus L, 5 plus L; the same for both
// positions), first site-parameter entry (from bit 20).
constexpr int kHitOld = 1 << 6;
constexpr int kHitNew = 1 << 7;
constexpr int kHitImage = 8;
constexpr int kHitParam = 20;
static_assert(kParamCap <= 2048 && kMaxSites < 64, "a hit packs both");

// A proposed move, ready to be evaluated and committed: what the phases of an
// evaluation read of the moving molecule, and its candidates.
struct MoveRecord {
  // the real sites, those with an LJ term (epsilon != 0) first
  MoveSite site[kMaxSites];
  // the first primary, old and proposed, and per axis how far a candidate's
  // wrapped displacement from the old one may be for its site pairs to share
  // one image (stage_move)
  double po[3], pn[3], lim[3];
  // the sites by index, proposed and old
  double nx[kMaxSites], ny[kMaxSites], nz[kMaxSites];
  double ox[kMaxSites], oy[kMaxSites], oz[kMaxSites];
  int2 cell[kScanEntries];  // cells of the range, or pieces: first slot, occupancy
  int32_t pofs[kMaxSites];  // primary offsets within the molecule
  int32_t mol, start, len, pstart, npri;
  int32_t n_real, n_lj;     // entries of site, and of which have an LJ term
  int32_t src;              // neighbour source
  int32_t nitems;           // candidate items it holds (with free cell slots)
  int32_t ncand;            // molecules it holds
  int32_t cell_w;           // items per entry of cell (cell source)
  int32_t co[3], cn[3];     // cell of the first primary, old and proposed
  int32_t fault;            // MCGPU_FAULT_* (0 = none)
  int32_t param, pf;        // first site-parameter entry, first primary's offset
};

// What every wave needs of a record first, loaded together: one LDS round trip
// instead of one per field and branch.
struct MoveHead {
  int mol, src, nitems, cell_w, fault;
};

__device__ __forceinline__ MoveHead load_head(const MoveRecord& m) {
  MoveHead h{m.mol, m.src, m.nitems, m.cell_w, m.fault};
  h.mol = __builtin_amdgcn_readfirstlane(h.mol);
  h.src = __builtin_amdgcn_readfirstlane(h.src);
  h.nitems = __builtin_amdgcn_readfirstlane(h.nitems);
  h.cell_w = __builtin_amdgcn_readfirstlane(h.cell_w);
  h.fault = __builtin_amdgcn_readfirstlane(h.fault);
  return h;
}

// LDS of an evaluation by NW waves.  PC: molecules whose primaries a launch
// may keep (0: none); NREC: move records; CAP: hits held before their pairs
// are summed.
template <int NW_, int PC, int NREC, int CAP>
struct EvalShared {
  static constexpr int kNW = NW_;
  static constexpr int kNT = NW_ * 64;
  static constexpr int kCap = CAP;
  static constexpr int kRound = kNW > 8 ? 1 : 2;  // scan passes a round
  static_assert(kRound * kNT <= kCap, "a round's hits fit");
  static constexpr int kPrim = PC;
  static constexpr int kCellLds = 1024;  // cells whose counts a launch keeps in LDS
  // What the pair loop reads comes first, within the 64 KiB that LDS
  // instructions reach with an immediate offset from one base.
  MoveRecord rec[NREC];
  SiteParam64 prm64[kParamCap];  // the box's site-parameter table
  // hits, compacted: from the front those whose pairs share one periodic
  // image, from the back those whose site pairs may wrap differently
  int2 hit[kCap];
  // copy of the box's cell occupancies, kept by launches that hold the box
  // for many moves (the batch kernel)
  int32_t ccount[PC ? kCellLds : 1];
  // per wave, the row sums of wave_row_sums: old energy in [0, 2 kNW), new in
  // [2 kNW, 4 kNW)
  double red[4 * kNW];
  unsigned redc[kNW];  // sites of the hits, per wave (boxes not uniform)
  unsigned cnt[kNW];   // hits of a round per wave: same image | other << 16
  // primaries of a single-primary box kept by a launch
  double px[PC ? PC : 1], py[PC ? PC : 1], pz[PC ? PC : 1];
};

// Copies the box's site-parameter table into LDS (threads [0, nt); the caller
// places a barrier before it is read).  Tables are at most kParamCap entries
// (checked when a box is created).
template <class SH>
__device__ __forceinline__ void load_params(const BoxView& bv, SH& sh, int nt) {
  for (int k = threadIdx.x; k < bv.n_param; k += nt) sh.prm64[k] = bv.p64[k];
}

// One wave stages up to two moves, lanes [0, 32) into one record and lanes
// [32, 64) into another (m: the calling lane's).  Lane k of a half holds site k
// at its old and proposed position.
//
// stage_sites: which sites go where, and their parameters, from table entry
// `param` on: the real sites become MoveSite records, those with an LJ term
// first, so that the pair phase runs the LJ arithmetic for those alone.
// Returns the record entry of the lane's site (-1: none).  In a uniform box it
// is the same for every molecule, so a launch does it once.  sh.prm64 must be
// loaded.
template <class SH>
__device__ __forceinline__ int stage_sites(const SH& sh, MoveRecord* m, int len, int param) {
  const int k = wlane() & 31;
  SiteParam64 p{0.0, 0.0, 0.0, 0.0};
  if (k < len) p = sh.prm64[param + k];
  const bool lj = p.real != 0.0 && p.e != 0.0;
  const bool rest = p.real != 0.0 && !lj;
  const unsigned long long blj = __ballot(lj), brest = __ballot(rest);
  const bool up = wlane() >= 32;
  const unsigned hlj = up ? (unsigned)(blj >> 32) : (unsigned)blj;
  const unsigned hrest = up ? (unsigned)(brest >> 32) : (unsigned)brest;
  const unsigned below = (1u << k) - 1u;
  const int nlj = __popc(hlj);
  const int at = lj ? __popc(hlj & below) : (rest ? nlj + __popc(hrest & below) : -1);
  if (at >= 0) {
    MoveSite& s = m->site[at];
    s.s = p.s;
    s.e = p.e;
    s.q = p.q;
    s.e32 = (float)p.e;
    s.s32 = s.e32 != 0.0f ? (float)p.s : 0.0f;
  }
  if (k == 0) {
    m->len = len;
    m->n_lj = nlj;
    m->n_real = nlj + __popc(hrest);
  }
  return at;
}

// stage_move: the coordinates, by the entry stage_sites gave and (proposed) by
// site for the commit; the old ones by site are the caller's (boxes with
// several primaries per molecule read them).  pf: the first primary's offset.
//
// lim: let w be a candidate's displacement from the old first primary, wrapped
// by k L with k in {-1, 0, 1}.  A site pair's raw displacement lies within
// reach2 of the two first primaries', and the proposed primary's within |move|
// of the old one's, so |w| <= L/2 - reach2 - |move| puts every site pair, at
// both positions, on the same side of +-L/2: the reference's wrap then adds
// k L to each of them.  A primary carried across the boundary has |move|
// close to L: its candidates then all take the wrap per site pair.
__device__ __forceinline__ void stage_move(const HotBox& hb, MoveRecord* m, int at, int len,
                                           int pf, double xo, double yo, double zo, double xn,
                                           double yn, double zn) {
  const int k = wlane() & 31;
  if (at >= 0) {
    MoveSite& s = m->site[at];
    s.xo = xo;
    s.yo = yo;
    s.zo = zo;
    s.xn = xn;
    s.yn = yn;
    s.zn = zn;
  }
  if (k < len) {
    m->nx[k] = xn;
    m->ny[k] = yn;
    m->nz[k] = zn;
  }
  if (k == pf) {
    m->po[0] = xo;
    m->po[1] = yo;
    m->po[2] = zo;
    m->pn[0] = xn;
    m->pn[1] = yn;
    m->pn[2] = zn;
    m->lim[0] = 0.5 * hb.L0 - hb.reach2 - fabs(xn - xo);
    m->lim[1] = 0.5 * hb.L1 - hb.reach2 - fabs(yn - yo);
    m->lim[2] = 0.5 * hb.L2 - hb.reach2 - fabs(zn - zo);
  }
}

// A molecule at its current position and, when given, at the proposed one
// (nxyz: x block, y block, z block): one wave, lane k holding site k.
struct Molecule {
  int start, len, param, pf, ps, pc, fault;
  int po;  // lane k: offset of primary k
  double xo, yo, zo, xn, yn, zn;
};

// Its loads, which need nothing staged, so that they run beside the parameter
// table's: a launch of one move is a chain of memory latencies (as a step
// after the table's barrier, through four index arrays, it was 2,800 of a
// launch's 13,200 cycles).
__device__ __forceinline__ Molecule load_molecule(const BoxView& bv, const HotBox& hb, int mol,
                                                  const double* nxyz) {
  const int k = wlane();
  Molecule q;
  q.start = mol * hb.uni_len;
  q.len = hb.uni_len;
  q.param = hb.uni_param;
  q.pf = hb.uni_p0;
  q.ps = mol;
  q.pc = 1;
  if (hb.uni_len == 0) {
    const MolMeta mm = hb.meta[mol];
    q.start = mm.start;
    q.len = mm.len;
    q.param = mm.param;
    q.pf = mm.p0;
    q.ps = mm.pstart;
    if (!hb.single_primary) q.pc = bv.mol_pidx_count[mol];
  }
  q.fault = q.len < 1 || q.len > kMaxSites ? MCGPU_FAULT_MOLLEN : 0;
  q.len = q.len < 1 ? 1 : (q.len > kMaxSites ? kMaxSites : q.len);
  q.pc = q.pc < 1 ? 1 : (q.pc > kMaxSites ? kMaxSites : q.pc);
  q.xo = q.yo = q.zo = q.xn = q.yn = q.zn = 0.0;
  if (k < q.len) {
    q.xo = hb.x[q.start + k];
    q.yo = hb.y[q.start + k];
    q.zo = hb.z[q.start + k];
    q.xn = nxyz ? nxyz[k] : q.xo;
    q.yn = nxyz ? nxyz[q.len + k] : q.yo;
    q.zn = nxyz ? nxyz[2 * q.len + k] : q.zo;
  }
  q.po = q.pf;
  if (!hb.single_primary && k < q.pc) q.po = bv.pidx[q.ps + k] - q.start;
  return q;
}

// And into record m, by the same wave, after the parameter table is staged.
template <class SH>
__device__ __forceinline__ void stage_molecule(const HotBox& hb, const Molecule& q, int mol,
                                               SH& sh, MoveRecord* m) {
  const int k = wlane();
  if (k < q.pc) m->pofs[k] = q.po;
  if (k == 0) {
    m->mol = mol;
    m->start = q.start;
    m->pstart = q.ps;
    m->npri = q.pc;
    m->fault = q.fault;
  }
  if (k < 32) {
    const int at = stage_sites(sh, m, q.len, q.param);
    if (k < q.len) {
      m->ox[k] = q.xo;
      m->oy[k] = q.yo;
      m->oz[k] = q.zo;
    }
    stage_move(hb, m, at, q.len, q.pf, q.xo, q.yo, q.zo, q.xn, q.yn, q.zn);
  }
}

// Any primary pair of (moving molecule at X/Y/Z, molecule with primaries
// ps .. ps+pc-1 in the mirror) within the cutoff (SimulationStep.cpp:317-330).
__device__ __forceinline__ bool primary_in_range(const BoxView& bv, int ps, int pc,
                                                 const double* X,
                                                 const double* Y,
                                                 const double* Z,
                                                 const int32_t* pofs,
                                                 int npri) {
  bool in = false;
  for (int q = 0; q < pc; q++) {
    const double qx = bv.px[ps + q], qy = bv.py[ps + q], qz = bv.pz[ps + q];
    for (int p = 0; p < npri; p++) {
      const int o = pofs[p];
      const double dx = wrap1(qx - X[o], bv.L[0]);
      const double dy = wrap1(qy - Y[o], bv.L[1]);
      const double dz = wrap1(qz - Z[o], bv.L[2]);
      in |= (dx * dx + dy * dy + dz * dz) <= bv.cutoff2;
    }
  }
  return in;
}

// wrap1, and k (0, 1.0 or -1.0, as the high word of a double) of d - k L.
__device__ __forceinline__ double wrap_k(double d, double L, int& k) {
  k = fabs(d) > 0.5 * L ? (__double2hiint(d) & (int)0x80000000) | 0x3ff00000 : 0;
  return fma(-__hiloint2double(k, 0), L, d);
}

// u / m for u < 2^20, with rm = 1 / m (v_rcp_f32): (u + 0.5) / m
// lies at least 0.5 / m from an integer, beyond the product's error of about
// 2^-22 u / m.
__device__ __forceinline__ int div_small(int u, float rm) {
  return (int)(((float)u + 0.5f) * rm);
}

// v - k L for the image code (0, 1, 5: k = 0, 1, -1) of a hit's y at bit `at`.
__device__ __forceinline__ double image_shifted(int y, int at, double v, double L) {
  const unsigned c = (unsigned)y >> at;
  return fma(-__hiloint2double((int)((c & 1) * 0x3ff00000u | (c & 4) << 29), 0), L, v);
}

// One item of the pair phase: a site b of a hit, held by one lane.
struct PairItem {
  double x, y, z;     // shifted by the periodic image of its hit
  double s, e, q;     // pair parameters (MIXED: half the charge)
  float s32, e32;
  int flags;          // kHitOld, kHitNew: the positions its hit is in range of
};

// Its MIXED parameters.  Sites without an LJ term get sigma 0 too, so that
// they never look like near contact.
__device__ __forceinline__ void mixed_item(PairItem& b, const SiteParam64& p) {
  b.q = 0.5 * p.q;
  b.e32 = (float)p.e;
  b.s32 = b.e32 != 0.0f ? (float)p.s : 0.0f;
}

// Sum over the moving molecule's sites [a0, a1) of their pairs with item b,
// at the old and (NEW) the proposed position: LJ = 4 eps_ab (s2^6 - s2^3), s2
// = sigma_ab^2 / r^2, and Coulomb = 332.06 q_a q_b / r (SimulationStep.cpp:
// 344-367; BruteForceStep.cpp:64-73).  LJ: the sites have an LJ term.
// WRAP: the reference's wrap per site pair.  GUARD:
// r^2 == 0 contributes nothing; without it such a pair makes the sum
// non-finite and the caller repeats the sum with GUARD.
// M holds the sites (NEW: with proposed positions).
template <bool MIXED, bool NEW, bool WRAP, bool LJ, bool GUARD, class M>
__device__ __forceinline__ void pair_sites(const M& m, const PairItem& b,
                                           const double L[3], int a0, int a1, double& eo,
                                           double& en) {
  auto dist2 = [&](double x, double y, double z) {
    double dx = b.x - x, dy = b.y - y, dz = b.z - z;
    if (WRAP) {
      int k;
      dx = wrap_k(dx, L[0], k);
      dy = wrap_k(dy, L[1], k);
      dz = wrap_k(dz, L[2], k);
    }
    return fma(dz, dz, fma(dy, dy, dx * dx));
  };
#pragma unroll 1
  for (int a = a0; a < a1; a++) {
    const auto A = m.site[a];
    const double qab = A.q * b.q;
    const double r2o = dist2(A.xo, A.yo, A.zo);
    double r2n = 0.0;
    if constexpr (NEW) r2n = dist2(A.xn, A.yn, A.zn);
    double e_o, e_n = 0.0;
    if (MIXED) {
      // both positions side by side, and one test of either for near contact
      const float ro = __builtin_amdgcn_rsqf((float)r2o);
      const float rn = NEW ? __builtin_amdgcn_rsqf((float)r2n) : 0.0f;
      double lo = 0.0, ln = 0.0;
      if (LJ) {
        const float sab = A.s32 * b.s32, eab = A.e32 * b.e32;
        const float so = pair_s6(ro, sab), sn = NEW ? pair_s6(rn, sab) : 0.0f;
        lo = (double)(eab * fmaf(so, so, -so));
        if (NEW) ln = (double)(eab * fmaf(sn, sn, -sn));
        if (fmaxf(so, sn) > kNearContactS6) {
          const double sab64 = A.s * b.s, eab64 = A.e * b.e;
          if (so > kNearContactS6) lo = pair_lj_near(r2o, sab64, eab64);
          if (sn > kNearContactS6) ln = pair_lj_near(r2n, sab64, eab64);
        }
      }
      e_o = fma(qab, refine_rinv32(r2o, ro), lo);
      if (NEW) e_n = fma(qab, refine_rinv32(r2n, rn), ln);
    } else {
      const double sab = A.s * b.s, eab = A.e * b.e;
      auto term = [&](double r2, double e) {  // e + the pair's energy
        const double rinv = rsqrt64(r2);
        e = fma(qab, rinv, e);
        if (LJ) {
          const double s2 = sab * (rinv * rinv);
          const double s6 = s2 * s2 * s2;
          e = fma(eab, fma(s6, s6, -s6), e);
        }
        return e;
      };
      if (!GUARD) {
        eo = term(r2o, eo);
        if (NEW) en = term(r2n, en);
        continue;
      }
      e_o = term(r2o, 0.0);
      if (NEW) e_n = term(r2n, 0.0);
    }
    eo += GUARD && r2o == 0.0 ? 0.0 : e_o;
    if (NEW) en += GUARD && r2n == 0.0 ? 0.0 : e_n;
  }
}

template <bool MIXED, bool NEW, bool WRAP>
__device__ __forceinline__ void pair_sites_all(const MoveRecord& m, const PairItem& b,
                                               const double L[3], int nlj, int a0, int a1,
                                               double& eo, double& en) {
  const int alj = a1 < nlj ? a1 : nlj;
  if (a0 < alj) pair_sites<MIXED, NEW, WRAP, true, false>(m, b, L, a0, alj, eo, en);
  const int ar = a0 > nlj ? a0 : nlj;
  if (ar < a1) pair_sites<MIXED, NEW, WRAP, false, false>(m, b, L, ar, a1, eo, en);
}

// Sums the pair energies of the compacted hits into e_old / e_new.  Items
// (hit, site b) are numbered hit by hit, max_len to a hit, and taken 64 to a
// block; a lane loads its item's site straight from the box (no staging
// through LDS, so no barrier and no LDS round trip between the load and its
// use) and keeps it while the block's sums run over the moving molecule's
// sites, whose records are LDS broadcasts.  The (block, site a) steps are
// dealt to the waves in runs of equal length, so a wave meets at most a few
// blocks and the waves finish together; a block's sites load while the
// previous block is summed.  Per step the FP64 arithmetic is 2 x 22
// instructions and the reciprocal square roots against the 66 of a layout
// with one lane per site a, which re-read b's position and parameters for
// each pair and tested the in-range flags there; here the flags choose once
// per block.  The caller places a barrier before the hits or the sites
// change.
template <bool MIXED, bool NEW, class SH>
__device__ __forceinline__ void pair_phase(const HotBox& hb, const SH& sh, const MoveRecord& m,
                                           int nsame, int nwrap, double& e_old,
                                           double& e_new) {
  constexpr int NW = SH::kNW;
  const int M = hb.max_len;
  const float rM = __builtin_amdgcn_rcpf((float)M);
  const int na = __builtin_amdgcn_readfirstlane(m.n_real);
  const int nlj = __builtin_amdgcn_readfirstlane(m.n_lj);
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  const double L[3] = {hb.L0, hb.L1, hb.L2};
  // blocks of the hits that wrap per site pair come first
  const int wblk = (nwrap * M + 63) >> 6;
  const int nblk = wblk + ((nsame * M + 63) >> 6);
  const int steps = nblk * na;
  int u = steps * w / NW;
  const int u_end = steps * (w + 1) / NW;
  if (u >= u_end) return;
  int blk = __builtin_amdgcn_readfirstlane(div_small(u, __builtin_amdgcn_rcpf((float)na)));
  int a0 = u - blk * na;
  auto load = [&](int k) {
    PairItem b;
    const bool wrap = k < wblk;  // wave-uniform
    const int tot = (wrap ? nwrap : nsame) * M;
    const int item = (wrap ? k : k - wblk) * 64 + wlane();
    // lanes past the items repeat the last one, lanes past a shorter
    // molecule its first site: valid addresses, and no flags
    const int it = item < tot ? item : tot - 1;
    const int h = div_small(it, rM);
    int o = it - h * M;
    const int2 r = sh.hit[wrap ? SH::kCap - 1 - h : h];
    const bool in = item < tot && o < (r.y & 63);
    o = in ? o : 0;
    const unsigned site = (unsigned)(r.x + o);
    b.x = hb.x[site];
    b.y = hb.y[site];
    b.z = hb.z[site];
    const int pk = (int)((unsigned)r.y >> kHitParam) + o;
    const SiteParam64 p = sh.prm64[pk];
    b.s = p.s;
    b.e = p.e;
    b.q = p.q;
    if (MIXED) mixed_item(b, p);
    // a dummy site: no pairs, whatever its distance
    b.flags = in && p.real != 0.0 ? r.y & (kHitOld | kHitNew) : 0;
    if (!wrap) {
      b.x = image_shifted(r.y, kHitImage, b.x, L[0]);
      b.y = image_shifted(r.y, kHitImage + 3, b.y, L[1]);
      b.z = image_shifted(r.y, kHitImage + 6, b.z, L[2]);
    }
    return b;
  };
  PairItem b = load(blk);
  for (;;) {
    const int a1 = na < a0 + (u_end - u) ? na : a0 + (u_end - u);
    u += a1 - a0;
    PairItem next = b;
    if (u < u_end) next = load(blk + 1);
    double eo = 0.0, en = 0.0;
    if (blk < wblk)
      pair_sites_all<MIXED, NEW, true>(m, b, L, nlj, a0, a1, eo, en);
    else
      pair_sites_all<MIXED, NEW, false>(m, b, L, nlj, a0, a1, eo, en);
    // sites at zero distance (or no longer finite): again with the guard (a
    // shifted site's displacement is within L/2, so the wrap leaves it)
    if (__ballot(b.flags != 0 && !(fabs(eo) + fabs(en) < __builtin_huge_val()))) {
      eo = en = 0.0;
      pair_sites<MIXED, NEW, true, true, true>(m, b, L, a0, a1, eo, en);
    }
    e_old += b.flags & kHitOld ? eo : 0.0;
    e_new += b.flags & kHitNew ? en : 0.0;
    if (u >= u_end) break;
    b = next;
    blk++;
    a0 = 0;
  }
}

// Neighbour source actually usable for this evaluation (block-uniform).
__device__ __forceinline__ int pick_source(const BoxView& bv, const MoveRecord& m,
                                           bool has_new) {
  const int mol = m.mol;
  if (bv.mode == MCGPU_NB_CELL && bv.cells.overflow[0] == 0) return MCGPU_NB_CELL;
  if (bv.mode == MCGPU_NB_VERLET && bv.verlet.stale[0] == 0 &&
      bv.verlet.count[mol] <= bv.verlet.cap) {
    const double* r = bv.verlet.ref + 3 * mol;
    if (has_new) {
      const double dx = wrap1(m.pn[0] - r[0], bv.L[0]);
      const double dy = wrap1(m.pn[1] - r[1], bv.L[1]);
      const double dz = wrap1(m.pn[2] - r[2], bv.L[2]);
      if (dx * dx + dy * dy + dz * dz > bv.verlet.skin_half2) return MCGPU_NB_BRUTE;
    }
    return MCGPU_NB_VERLET;
  }
  return MCGPU_NB_BRUTE;
}

// Piece q of a cell of n molecules from slot `first` on.
__device__ __forceinline__ int2 piece_of(int first, int n, int q, int width) {
  const int at = q * width;
  return make_int2(first + at, n - at < width ? n - at : width);
}

// One wave completes two records, each half of the wave its own (m; both halves
// may name the same): the neighbour source src (cells, or every molecule from
// jlo on, or the Verlet list).
//
// Cells: the cells of the record's old first primary and, when has_new, of its
// proposed one into m->co / m->cn, lane d < 3 of the half taking axis d, then the
// cells around them with their occupancies (from sh.ccount when lds_counts)
// into m->cell, the range along an axis as in make_range.  Candidate items are
// numbered cell_w to an entry (scan_width), so a lane finds its entry by one
// division instead of a prefix and an item -> cell map (which cost a barrier).
// A range of more than 64 cells, or of more items than div_small divides, scans
// every molecule.
template <class SH>
__device__ __forceinline__ void prepare_source(const BoxView& bv, const SH& sh, MoveRecord* m,
                                               int src, int jlo, bool has_new,
                                               bool lds_counts) {
  const int lane = wlane(), half = lane & 32, k = lane & 31;
  int nitems = bv.n_mol - jlo, ncand = nitems, cell_w = 1;
  if (src == MCGPU_NB_VERLET) nitems = ncand = bv.verlet.count[m->mol];
  if (src == MCGPU_NB_CELL) {
    const CellGrid& g = bv.cells;
    const int cap = g.cap;
    CellRange range;
    {
      const int d = k < 2 ? k : 2;
      const int n0 = g.n[0], n1 = g.n[1], n2 = g.n[2];
      const double w0 = g.inv_w[0], w1 = g.inv_w[1], w2 = g.inv_w[2];
      const int n = d == 0 ? n0 : (d == 1 ? n1 : n2);
      const double iw = d == 0 ? w0 : (d == 1 ? w1 : w2);
      const int co = cell_coord(m->po[d], iw, n);
      const int cn = has_new ? cell_coord(m->pn[d], iw, n) : co;
      if (k < 3) {
        m->co[k] = co;
        m->cn[k] = cn;
      }
      int delta = cn - co;
      if (2 * delta > n) delta -= n;
      if (2 * delta < -n) delta += n;
      int lo = co + (delta < 0 ? delta : 0) - 1;
      int cnt = (delta < 0 ? -delta : delta) + 3;
      lo = cnt >= n ? 0 : lo;
      cnt = cnt >= n ? n : cnt;
#pragma unroll
      for (int d2 = 0; d2 < 3; d2++) {
        range.lo[d2] = shuffle_i32(lo, half + d2);
        range.cnt[d2] = shuffle_i32(cnt, half + d2);
      }
    }
    const int total = range.total();
    bool cells = total <= kScanEntries;
    int na = 0, nb = 0;  // occupancies of cells k and k + 32 of the range
    int fa = 0, fb = 0;  // and their first slots
    if (cells && k < total) {
      const int c = range.cell(g, k);
      na = lds_counts ? sh.ccount[c] : g.count[c];
      na = na < cap ? na : cap;
      fa = c * cap;
      m->cell[k] = make_int2(fa, na);
    }
    if (__ballot(cells && total > 32)) {
      if (cells && k + 32 < total) {
        const int c = range.cell(g, k + 32);
        nb = lds_counts ? sh.ccount[c] : g.count[c];
        nb = nb < cap ? nb : cap;
        fb = c * cap;
        m->cell[k + 32] = make_int2(fb, nb);
      }
    }
    int w, sum, wb, sb;
    half_max_sum_i32(na, w, sum);
    if (__ballot(cells && total > 32)) {
      half_max_sum_i32(nb, wb, sb);
      w = w > wb ? w : wb;
      sum += sb;
    }
    int entries = total;
    const int width = cells ? scan_width(total, w, sum, SH::kNT) : w;
    if (__ballot(width < w)) {
      // pieces, in the cells' order
      const float rw = __builtin_amdgcn_rcpf((float)(width > 0 ? width : 1));
      const int ea = na > 0 ? div_small(na + width - 1, rw) : 0;
      const int eb = nb > 0 ? div_small(nb + width - 1, rw) : 0;
      const int pa = half_incl_scan_i32(ea);
      const int ta = shuffle_i32(pa, half + 31);
      const int pb = ta + half_incl_scan_i32(eb);
      const int tb = shuffle_i32(pb, half + 31);
      if (width < w) {
        for (int q = 0; q < ea; q++)
          m->cell[pa - ea + q] = piece_of(fa, na, q, width);
        for (int q = 0; q < eb; q++)
          m->cell[pb - eb + q] = piece_of(fb, nb, q, width);
        entries = tb;
        w = width;
      }
    }
    cells = cells && w <= kMaxScanItems / kScanEntries;
    src = cells ? MCGPU_NB_CELL : MCGPU_NB_BRUTE;
    nitems = cells ? w * entries : nitems;
    ncand = cells ? sum : ncand;
    cell_w = cells ? w : 1;
  }
  // A neighbour source never holds more candidates than molecules; if it
  // claims so its lists are corrupt: record it and evaluate nothing.
  const bool bad = ncand < 0 || ncand > bv.n_mol;
  if (k == 0) {
    m->src = src;
    m->nitems = bad ? 0 : nitems;
    m->ncand = ncand;
    m->cell_w = cell_w;
    if (bad) m->fault = MCGPU_FAULT_CANDIDATES;
  }
}

// A round of the scan: up to kRound passes of kNT candidate items from `base`
// on, one item a lane and pass.
template <class SH>
struct ScanRound {
  static constexpr int R = SH::kRound;
  int2 rec[R];                        // the lane's candidates as hits
  unsigned long long same[R], wrap[R];  // the wave's hits, by kind (ballots)
  unsigned count;                     // their numbers: same | wrap << 16
  unsigned sites;                     // sites of this lane's hits
};

// Items of the next round of `left`: one pass where that is enough, without the
// other's guards and registers (mixture of 3,000 with cells, 4 waves, 10.65 ->
// 10.25 us a move), else kRound passes, which saves two barriers a pass.  With
// more than 8 waves a round is one pass: two were 0.3 us better where one does
// not do (mixture of 3,000, 15 waves, 6.39 and 6.06) and as much worse where it
// does (16-site bicyclic of 4,000, 7.44 and 7.71).
template <class SH>
__device__ __forceinline__ int round_items(int left) {
  return left > SH::kNT ? SH::kRound * SH::kNT : SH::kNT;
}

// SRC: the neighbour source; PRIM: primaries from sh.px/py/pz; UNI: a uniform
// box.  Boxes with one primary per molecule.  The loads of the passes are
// issued together, first the candidates, then their primaries; a candidate
// then takes about 45 instructions.  Each combination has its own code: the
// choices inside it cost a chain of scalar branches and loads per pass
// (2,300 against 1,500 cycles for one pass of 256 molecules).
template <int R, int SRC, bool PRIM, bool UNI, bool NEW, class SH>
__device__ __forceinline__ void scan_round(const BoxView& bv, const HotBox& hb, const SH& sh,
                                           const MoveRecord& m, const MoveHead& h, int base,
                                           int jlo, ScanRound<SH>& r) {
  constexpr int NT = SH::kNT;
  const int t = threadIdx.x;
  const int nitems = h.nitems, cell_w = h.cell_w, mol = h.mol;
  const double pox = m.po[0], poy = m.po[1], poz = m.po[2];
  const double pnx = m.pn[0], pny = m.pn[1], pnz = m.pn[2];
  const double limx = m.lim[0], limy = m.lim[1], limz = m.lim[2];
  const double L0 = hb.L0, L1 = hb.L1, L2 = hb.L2, rc2 = hb.cutoff2;
  const float rw = __builtin_amdgcn_rcpf((float)cell_w);
  int j[R];  // candidate (-1: none)
  double qx[R], qy[R], qz[R];
#pragma unroll
  for (int p = 0; p < R; p++) {
    if (p > 0 && base + p * NT >= nitems) continue;  // block-uniform
    const int item = base + p * NT + t;
    const int it = item < nitems ? item : nitems - 1;
    if (SRC == MCGPU_NB_CELL) {
      const int k = div_small(it, rw);
      const int s = it - k * cell_w;
      const int2 c = m.cell[k];
      const bool in = item < nitems && s < c.y;
      const int v = hb.slots[(unsigned)(in ? c.x + s : 0)];
      j[p] = in ? v : -1;
    } else if (SRC == MCGPU_NB_VERLET) {
      const int v = bv.verlet.list[mol * bv.verlet.cap + it];
      j[p] = item < nitems ? v : -1;
    } else {
      j[p] = item < nitems ? jlo + it : -1;
    }
  }
#pragma unroll
  for (int p = 0; p < R; p++) {
    if (p > 0 && base + p * NT >= nitems) continue;
    if (j[p] < jlo) j[p] = mol;
    const unsigned jj = (unsigned)j[p];  // every lane loads a valid entry
    if (UNI) {  // the record follows from the index
      r.rec[p] = make_int2((int)jj * hb.uni_len, hb.uni_len | hb.uni_param << kHitParam);
    } else {
      const MolMeta mj = hb.meta[jj];
      r.rec[p] = make_int2(mj.start, mj.len | mj.param << kHitParam);
    }
    if (PRIM) {
      qx[p] = sh.px[jj];
      qy[p] = sh.py[jj];
      qz[p] = sh.pz[jj];
    } else {
      qx[p] = hb.px[jj];
      qy[p] = hb.py[jj];
      qz[p] = hb.pz[jj];
    }
  }
#pragma unroll
  for (int p = 0; p < R; p++) {
    if (p > 0 && base + p * NT >= nitems) continue;
    int kx, ky, kz;
    const double dx = wrap_k(qx[p] - pox, L0, kx);
    const double dy = wrap_k(qy[p] - poy, L1, ky);
    const double dz = wrap_k(qz[p] - poz, L2, kz);
    int info = fma(dz, dz, fma(dy, dy, dx * dx)) <= rc2 ? kHitOld : 0;
    if (NEW) {
      int unused;
      const double ex = wrap_k(qx[p] - pnx, L0, unused);
      const double ey = wrap_k(qy[p] - pny, L1, unused);
      const double ez = wrap_k(qz[p] - pnz, L2, unused);
      info |= fma(ez, ez, fma(ey, ey, ex * ex)) <= rc2 ? kHitNew : 0;
    }
    const bool hit = j[p] != mol && info != 0;
    const bool wrap = fabs(dx) > limx || fabs(dy) > limy || fabs(dz) > limz;
    if (!UNI) r.sites += hit ? (unsigned)(r.rec[p].y & 63) : 0u;
    r.rec[p].y |= info | ((unsigned)kx >> 29 | ((unsigned)ky >> 29) << 3 |
                          ((unsigned)kz >> 29) << 6)
                             << kHitImage;
    r.same[p] = __ballot(hit && !wrap);
    r.wrap[p] = __ballot(hit && wrap);
    r.count += (unsigned)__popcll(r.same[p]) | (unsigned)__popcll(r.wrap[p]) << 16;
  }
}

// The same for boxes with several primaries per molecule (any source), one
// pass at a time.
template <bool NEW, class SH>
__device__ __forceinline__ void scan_round_multi(const BoxView& bv, const HotBox& hb,
                                                 const MoveRecord& m, const MoveHead& hd,
                                                 int base, int jlo, ScanRound<SH>& r) {
  const int nitems = hd.nitems, cell_w = hd.cell_w, src = hd.src, mol = hd.mol;
  const float rw = __builtin_amdgcn_rcpf((float)cell_w);
#pragma unroll
  for (int p = 0; p < SH::kRound; p++) {
    if (p > 0 && base + p * SH::kNT >= nitems) continue;  // block-uniform
    const int item = base + p * SH::kNT + (int)threadIdx.x;
    int j = -1;
    if (item < nitems) {
      if (src == MCGPU_NB_CELL) {
        const int k = div_small(item, rw);
        const int s = item - k * cell_w;
        const int2 c = m.cell[k];
        j = s < c.y ? hb.slots[(unsigned)(c.x + s)] : -1;
      } else if (src == MCGPU_NB_VERLET) {
        j = bv.verlet.list[mol * bv.verlet.cap + item];
      } else {
        j = jlo + item;
      }
    }
    bool hit = false, wrap = false;
    if (j >= jlo && j != mol) {
      const MolMeta mj = hb.meta[(unsigned)j];
      const int ps = bv.mol_pidx_start[j], pc = bv.mol_pidx_count[j];
      int info = primary_in_range(bv, ps, pc, m.ox, m.oy, m.oz, m.pofs, m.npri) ? kHitOld : 0;
      if (NEW)
        info |= primary_in_range(bv, ps, pc, m.nx, m.ny, m.nz, m.pofs, m.npri) ? kHitNew : 0;
      hit = info != 0;
      int kx, ky, kz;
      wrap = fabs(wrap_k(hb.px[ps] - m.po[0], hb.L0, kx)) > m.lim[0];
      wrap |= fabs(wrap_k(hb.py[ps] - m.po[1], hb.L1, ky)) > m.lim[1];
      wrap |= fabs(wrap_k(hb.pz[ps] - m.po[2], hb.L2, kz)) > m.lim[2];
      info |= ((unsigned)kx >> 29 | ((unsigned)ky >> 29) << 3 | ((unsigned)kz >> 29) << 6)
              << kHitImage;
      r.rec[p] = make_int2(mj.start, info | mj.len | mj.param << kHitParam);
      r.sites += hit ? (unsigned)mj.len : 0u;
    }
    r.same[p] = __ballot(hit && !wrap);
    r.wrap[p] = __ballot(hit && wrap);
    r.count += (unsigned)__popcll(r.same[p]) | (unsigned)__popcll(r.wrap[p]) << 16;
  }
}

// Candidate scan + pair phase of record m, whose source is prepared, at the
// old position and (NEW) the proposed one.  Called by the threads of SH::kNW
// waves after a barrier that follows the preparation (h: m's head); a further
// wave of the work-group keeps step with eval_barriers.  prim_lds: the box's
// primaries are in sh.px/py/pz.  Leaves per-wave partial sums in sh.red (and,
// in boxes that are not uniform, sh.redc) and ends with a barrier.  Returns
// the number of in-range molecules.
template <bool NEW, class SH>
__device__ __forceinline__ int eval_core(const BoxView& bv, const HotBox& hb, SH& sh,
                                         const MoveRecord& m, const MoveHead& h, int jlo,
                                         bool mixed, bool prim_lds) {
  constexpr int R = SH::kRound;
  constexpr int NW = SH::kNW;
  constexpr int NT = SH::kNT;
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  const int src = h.src, nitems = h.nitems;
  const bool uni = hb.uni_len > 0;
  double eo = 0.0, en = 0.0;
  unsigned nsites = 0;
  int nsame = 0, nwrap = 0, base = 0, hits = 0;
  for (;;) {
    // rounds of R passes while their hits fit
    while (base < nitems) {
      const int step = round_items<SH>(nitems - base);
      if (nsame + nwrap + step > SH::kCap) break;
      ScanRound<SH> r;
      r.count = r.sites = 0;
#pragma unroll
      for (int p = 0; p < R; p++) r.same[p] = r.wrap[p] = 0;
#define MCGPU_SCAN_R(PASSES, SRC, PRIM)                                             \
  do {                                                                              \
    if (uni)                                                                        \
      scan_round<PASSES, SRC, PRIM, true, NEW>(bv, hb, sh, m, h, base, jlo, r);     \
    else                                                                            \
      scan_round<PASSES, SRC, PRIM, false, NEW>(bv, hb, sh, m, h, base, jlo, r);    \
  } while (0)
#define MCGPU_SCAN(SRC, PRIM)              \
  do {                                     \
    if (step > NT)                         \
      MCGPU_SCAN_R(R, SRC, PRIM);          \
    else                                   \
      MCGPU_SCAN_R(1, SRC, PRIM);          \
  } while (0)
      if (!hb.single_primary) {
        scan_round_multi<NEW>(bv, hb, m, h, base, jlo, r);
      } else if (SH::kPrim > 0) {
        if (prim_lds) {
          if (src == MCGPU_NB_CELL) MCGPU_SCAN(MCGPU_NB_CELL, true);
          else MCGPU_SCAN(MCGPU_NB_BRUTE, true);
        } else {
          if (src == MCGPU_NB_CELL) MCGPU_SCAN(MCGPU_NB_CELL, false);
          else MCGPU_SCAN(MCGPU_NB_BRUTE, false);
        }
      } else {
        if (src == MCGPU_NB_CELL) MCGPU_SCAN(MCGPU_NB_CELL, false);
        else if (src == MCGPU_NB_VERLET) MCGPU_SCAN(MCGPU_NB_VERLET, false);
        else MCGPU_SCAN(MCGPU_NB_BRUTE, false);
      }
#undef MCGPU_SCAN
#undef MCGPU_SCAN_R
      nsites += r.sites;
      if (wlane() == 0) sh.cnt[wave] = r.count;
      // the waves' counts, and this wave's place among them
      __syncthreads();
      const unsigned mine = wlane() < NW ? sh.cnt[wlane()] : 0u;
      const unsigned incl = (unsigned)wave_incl_row_i32((int)mine);
      const unsigned total = (unsigned)readlane_i32((int)incl, NW - 1);
      const unsigned pre = (unsigned)readlane_i32((int)(incl - mine), wave);
      int at0 = nsame + (int)(pre & 0xffff), at1 = nwrap + (int)(pre >> 16);
#pragma unroll
      for (int p = 0; p < R; p++) {
        if (p > 0 && step <= NT) continue;  // block-uniform
        const unsigned long long bit = 1ull << wlane();
        if (r.same[p] & bit) sh.hit[at0 + wave_rank(r.same[p])] = r.rec[p];
        if (r.wrap[p] & bit) sh.hit[SH::kCap - 1 - at1 - wave_rank(r.wrap[p])] = r.rec[p];
        at0 += __popcll(r.same[p]);
        at1 += __popcll(r.wrap[p]);
      }
      nsame += (int)(total & 0xffff);
      nwrap += (int)(total >> 16);
      base += step;
      __syncthreads();
    }
    hits += nsame + nwrap;
    if (mixed)
      pair_phase<true, NEW>(hb, sh, m, nsame, nwrap, eo, en);
    else
      pair_phase<false, NEW>(hb, sh, m, nsame, nwrap, eo, en);
    if (base >= nitems) break;
    __syncthreads();  // every lane is done with the hits before reuse
    nsame = nwrap = 0;
  }
  const double v = wave_row_sums(eo, en);
  if ((wlane() & 15) == 0) sh.red[(wlane() >> 4) * NW + wave] = v;
  if (!uni) {
    nsites = wave_sum_u32(nsites);
    if (wlane() == 0) sh.redc[wave] = nsites;
  }
  __syncthreads();
  return hits;
}

// The barriers of eval_core for a wave that does something else meanwhile:
// pair() while the others sum (what it does while they scan comes before the
// call).
template <class SH, class F>
__device__ __forceinline__ void eval_barriers(const SH& sh, const MoveHead& h, F pair) {
  constexpr int NW = SH::kNW;
  int n = 0, base = 0;
  for (bool first = true;; first = false) {
    while (base < h.nitems) {
      const int step = round_items<SH>(h.nitems - base);
      if (n + step > SH::kCap) break;
      __syncthreads();
      const unsigned c = wlane() < NW ? sh.cnt[wlane()] : 0u;
      const unsigned total =
          (unsigned)readlane_i32(wave_incl_row_i32((int)c), NW - 1);
      n += (int)(total & 0xffff) + (int)(total >> 16);
      base += step;
      __syncthreads();
    }
    if (first) pair();
    if (base >= h.nitems) break;
    __syncthreads();
    n = 0;
  }
  __syncthreads();
}


// Fixed-order totals of the per-wave partials left by eval_core, in every lane
// of the calling wave.
template <class SH>
__device__ __forceinline__ void eval_totals(const SH& sh, double& e_old, double& e_new) {
  constexpr int NW = SH::kNW;
  const int k = wlane() & 31;
  double v = k < 2 * NW ? sh.red[(wlane() >> 5) * 2 * NW + k] : 0.0;
  v += dpp_f64<0xb1>(v);
  v += dpp_f64<0x4e>(v);
  v += dpp_f64<0x124>(v);
  v += dpp_f64<0x128>(v);
  wave_half_totals(v, e_old, e_new);
}

// Moves molecule `mol` from cell cold to cell cnew in the cell lists (one
// lane): swap-remove from the old cell, append to the new one; a full cell
// marks the lists incomplete (scans then fall back to every molecule), and
// the call returns false.
__device__ __forceinline__ bool cell_move(const CellGrid& g, int mol, int cold,
                                          int cnew) {
  const int slot = g.mol_slot[mol];
  const int last = g.count[cold] - 1;
  const int lm = g.slots[cold * g.cap + last];
  g.slots[cold * g.cap + slot] = lm;
  g.mol_slot[lm] = slot;
  g.count[cold] = last;
  const int n = g.count[cnew];
  if (n < g.cap) {
    g.slots[cnew * g.cap + n] = mol;
    g.mol_slot[mol] = n;
    g.count[cnew] = n + 1;
    g.mol_cell[mol] = cnew;
    return true;
  }
  g.overflow[0] = 1;
  return false;
}

// The neighbour structures after molecule mol's first primary moved to (x, y,
// z) (one lane).
__device__ __forceinline__ void commit_lists(const BoxView& bv, int mol, double x, double y,
                                             double z) {
  if (bv.mode == MCGPU_NB_CELL && bv.cells.overflow[0] == 0) {
    const CellGrid& g = bv.cells;
    const int cnew = cell_index(g, cell_coord(x, g.inv_w[0], g.n[0]),
                                cell_coord(y, g.inv_w[1], g.n[1]),
                                cell_coord(z, g.inv_w[2], g.n[2]));
    const int cold = g.mol_cell[mol];
    if (cnew != cold) cell_move(g, mol, cold, cnew);
  }
  if (bv.mode == MCGPU_NB_VERLET) {
    const double* r = bv.verlet.ref + 3 * mol;
    const double dx = wrap1(x - r[0], bv.L[0]);
    const double dy = wrap1(y - r[1], bv.L[1]);
    const double dz = wrap1(z - r[2], bv.L[2]);
    if (dx * dx + dy * dy + dz * dz > bv.verlet.skin_half2) bv.verlet.stale[0] = 1;
  }
}

// Writes the proposed coordinates of record m into the box and keeps the
// primary mirror, cell lists and Verlet bookkeeping consistent.
__device__ __forceinline__ void commit_molecule(const BoxView& bv, const MoveRecord& m) {
  const int t = threadIdx.x;
  if (t < m.len) {
    bv.x[m.start + t] = m.nx[t];
    bv.y[m.start + t] = m.ny[t];
    bv.z[m.start + t] = m.nz[t];
  }
  if (t < m.npri) {
    const int o = m.pofs[t];
    bv.px[m.pstart + t] = m.nx[o];
    bv.py[m.pstart + t] = m.ny[o];
    bv.pz[m.pstart + t] = m.nz[o];
  }
  if (t == 0) commit_lists(bv, m.mol, m.pn[0], m.pn[1], m.pn[2]);
}

}  // namespace mcgpu
