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
#include "wave.h"

namespace mcgpu {

// A staged site of the full-energy kernel whose pairs take wrap1 per axis.
constexpr int kPairWrap = 1 << 20;

// A real site of the moving molecule as the pair phase reads it (the same
// address in every lane: LDS broadcasts): old and proposed position and pair
// parameters.
struct alignas(16) MoveSite {
  double xo, yo, zo, xn, yn, zn;
  double s, e, q;
  float s32, e32;
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

// PC: molecules whose primaries a launch may keep in LDS (0: none).
template <int NT, int PC = 0>
struct EvalShared {
  static constexpr int kCap = 1536;      // hits held before their pairs are summed
  static constexpr int kRound = NT >= 1024 ? 1 : (NT >= 512 ? 2 : 4);  // passes a round
  static_assert(kRound * NT <= kCap, "a round's hits fit");
  static constexpr int kPrim = PC;
  static constexpr int kCellLds = 1024;  // cells whose counts a launch keeps in LDS
  static constexpr int kNW = NT / 64;
  // What the pair loop reads comes first, within the 64 KiB that LDS
  // instructions reach with an immediate offset from one base.
  // the moving molecule's real sites, those with an LJ term (epsilon != 0)
  // first
  MoveSite site[kMaxSites];
  // the box's site-parameter table
  SiteParam64 prm64[kParamCap];
  SiteParam32 prm32[kParamCap];
  // hits, compacted: from the front those whose pairs share one periodic
  // image, from the back those whose site pairs may wrap differently
  int2 hit[kCap];
  // the moving molecule's first primary, old and proposed, and per axis how
  // far a candidate's wrapped displacement from the old one may be for its
  // site pairs to share one image (stage_move)
  double po[3], pn[3], lim[3];
  double ox[kMaxSites], oy[kMaxSites], oz[kMaxSites];
  double nx[kMaxSites], ny[kMaxSites], nz[kMaxSites];
  int32_t pofs[kMaxSites];   // primary offsets within the molecule
  int2 cell[64];             // cells of the current range: first slot, occupancy
  // copy of the box's cell occupancies, kept by launches that hold the box
  // for many moves (the batch kernel); prepare_cells_wave reads it when asked
  int32_t ccount[kCellLds];
  // per wave, the row sums of wave_row_sums: old energy in [0, 2 kNW), new in
  // [2 kNW, 4 kNW)
  double red[4 * kNW];
  unsigned redc[kNW];        // sites of the hits, per wave (boxes not uniform)
  unsigned cnt[kNW];         // hits of a round per wave: same image | other << 16
  int32_t npri;
  int32_t len;
  int32_t n_real;   // entries of site
  int32_t n_lj;     // of which the first n_lj have an LJ term
  int32_t flag;
  int32_t fault;    // MCGPU_FAULT_* raised by the last preparation (0 = none)
  int32_t src;      // neighbour source of the current evaluation
  int32_t nitems;   // candidate items it holds
  int32_t cell_w;   // items per cell (cell source)
  // primaries of a single-primary box kept by a launch (entries PC)
  double px[PC ? PC : 1], py[PC ? PC : 1], pz[PC ? PC : 1];
};

// Copies the box's site-parameter table into LDS (all threads; the caller
// places a barrier before it is read).  Tables are at most kParamCap entries
// (checked when a box is created).
template <int NT, int PC>
__device__ __forceinline__ void load_params(const BoxView& bv, EvalShared<NT, PC>& sh) {
  for (int k = threadIdx.x; k < bv.n_param; k += NT) {
    sh.prm64[k] = bv.p64[k];
    sh.prm32[k] = bv.p32[k];
  }
}

// Wave 0: the moving molecule's sites into LDS (lane k < len holds site k at
// its old and proposed position; its parameters start at table entry
// `param`): by site for the scan and the commit, and the real sites as
// MoveSite records, those with an LJ term first, so that the pair phase runs
// the LJ arithmetic for those alone.  pf: the first primary's offset.
// sh.prm64/prm32 must be loaded.
//
// lim: let w be a candidate's displacement from the old first primary, wrapped
// by k L with k in {-1, 0, 1}.  A site pair's raw displacement lies within
// reach2 of the two first primaries', and the proposed primary's within |move|
// of the old one's, so |w| <= L/2 - reach2 - |move| puts every site pair, at
// both positions, on the same side of +-L/2: the reference's wrap then adds
// k L to each of them.  A primary carried across the boundary has |move|
// close to L: its candidates then all take the wrap per site pair.
// The proposed sites stay by index too, for the commit (sh.nx .. sh.nz), and
// with by_site the old ones (boxes with several primaries per molecule).
template <int NT, int PC>
__device__ __forceinline__ void stage_move(const HotBox& hb, EvalShared<NT, PC>& sh, int len,
                                           int param, int pf, double xo, double yo, double zo,
                                           double xn, double yn, double zn, bool by_site) {
  const int lane = wlane();
  SiteParam64 p{0.0, 0.0, 0.0, 0.0};
  SiteParam32 p32{0.0f, 0.0f, 0.0f, 0.0f};
  if (lane < len) {
    p = sh.prm64[param + lane];
    p32 = sh.prm32[param + lane];
  }
  if (by_site && lane < len) {
    sh.ox[lane] = xo;
    sh.oy[lane] = yo;
    sh.oz[lane] = zo;
  }
  if (lane < len) {
    sh.nx[lane] = xn;
    sh.ny[lane] = yn;
    sh.nz[lane] = zn;
  }
  if (lane == pf) {
    sh.po[0] = xo;
    sh.po[1] = yo;
    sh.po[2] = zo;
    sh.pn[0] = xn;
    sh.pn[1] = yn;
    sh.pn[2] = zn;
    sh.lim[0] = 0.5 * hb.L0 - hb.reach2 - fabs(xn - xo);
    sh.lim[1] = 0.5 * hb.L1 - hb.reach2 - fabs(yn - yo);
    sh.lim[2] = 0.5 * hb.L2 - hb.reach2 - fabs(zn - zo);
  }
  const bool lj = p.real != 0.0 && p.e != 0.0;
  const bool rest = p.real != 0.0 && !lj;
  const unsigned long long blj = __ballot(lj), brest = __ballot(rest);
  const int nlj = __popcll(blj);
  if (lj || rest)
    sh.site[lj ? wave_rank(blj) : nlj + wave_rank(brest)] =
        MoveSite{xo, yo, zo, xn, yn, zn, p.s, p.e, p.q, p32.s, p32.e};
  if (lane == 0) {
    sh.len = len;
    sh.n_lj = nlj;
    sh.n_real = nlj + __popcll(brest);
  }
}

// Wave 0: molecule `mol` at its current position and, when given, at the
// proposed one (nxyz: x block, y block, z block) into LDS.  A barrier after
// load_params must precede it.
template <int NT, int PC>
__device__ __forceinline__ void load_molecule(const BoxView& bv, const HotBox& hb, int mol,
                                              const double* nxyz,
                                              EvalShared<NT, PC>& sh) {
  const int k = wlane();
  const int start = bv.mol_start[mol];
  int len = bv.mol_len[mol];
  const int fault = len < 1 || len > kMaxSites ? MCGPU_FAULT_MOLLEN : 0;
  len = len < 1 ? 1 : (len > kMaxSites ? kMaxSites : len);
  const int pbase = bv.mol_param[mol];
  double xo = 0.0, yo = 0.0, zo = 0.0, xn = 0.0, yn = 0.0, zn = 0.0;
  if (k < len) {
    xo = bv.x[start + k];
    yo = bv.y[start + k];
    zo = bv.z[start + k];
    xn = nxyz ? nxyz[k] : xo;
    yn = nxyz ? nxyz[len + k] : yo;
    zn = nxyz ? nxyz[2 * len + k] : zo;
  }
  const int ps = bv.mol_pidx_start[mol];
  int pc = bv.mol_pidx_count[mol];
  pc = pc < 1 ? 1 : (pc > kMaxSites ? kMaxSites : pc);
  if (k < pc) sh.pofs[k] = bv.pidx[ps + k] - start;
  if (k == 0) {
    sh.fault = fault;
    sh.npri = pc;
  }
  stage_move(hb, sh, len, pbase, bv.pidx[ps] - start, xo, yo, zo, xn, yn, zn, true);
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

// u / m for u < 2^20, with rm = 1 / m (v_rcp_f32): (u + 0.5) / m
// lies at least 0.5 / m from an integer, beyond the product's error of about
// 2^-22 u / m.
__device__ __forceinline__ int div_small(int u, float rm) {
  return (int)(((float)u + 0.5f) * rm);
}

// One item of the pair phase: a site b of a hit, held by one lane.
struct PairItem {
  double x, y, z;     // shifted by the periodic image of its hit
  double s, e, q;     // pair parameters
  float s32, e32;
  int flags;          // kHitOld, kHitNew: the positions its hit is in range of
};

// Sum over the moving molecule's sites [a0, a1) of their pairs with item b,
// at the old and (NEW) the proposed position.  LJ: the sites have an LJ term.
// WRAP: the reference's wrap per site pair.  GUARD:
// r^2 == 0 contributes nothing; without it such a pair makes the sum
// non-finite and the caller repeats the sum with GUARD.
template <bool MIXED, bool NEW, bool WRAP, bool LJ, bool GUARD, class SH>
__device__ __forceinline__ void pair_sites(const SH& sh, const PairItem& b,
                                           const double L[3], int a0, int a1, double& eo,
                                           double& en) {
  auto one = [&](const MoveSite& A, double x, double y, double z, double sab, double eab,
                 double qab, double& acc) {
    double dx = b.x - x, dy = b.y - y, dz = b.z - z;
    if (WRAP) {
      dx = wrap1(dx, L[0]);
      dy = wrap1(dy, L[1]);
      dz = wrap1(dz, L[2]);
    }
    const double r2 = fma(dz, dz, fma(dy, dy, dx * dx));
    double e;
    if (MIXED) {
      const float rinv = __builtin_amdgcn_rsqf((float)r2);
      const double rd = refine_rinv32(r2, rinv);
      e = LJ ? fma(qab, rd, pair_lj32(r2, rinv, A.s32, A.e32, b.s32, b.e32, A.s, A.e, b.s, b.e))
             : qab * rd;
    } else {
      const double rinv = rsqrt64(r2);
      e = qab * rinv;
      if (LJ) {
        const double s2 = sab * (rinv * rinv);
        const double s6 = s2 * s2 * s2;
        e = fma(eab, fma(s6, s6, -s6), e);
      }
    }
    acc += GUARD && r2 == 0.0 ? 0.0 : e;
  };
#pragma unroll 1
  for (int a = a0; a < a1; a++) {
    const MoveSite A = sh.site[a];
    const double sab = A.s * b.s, eab = A.e * b.e, qab = A.q * b.q;
    one(A, A.xo, A.yo, A.zo, sab, eab, qab, eo);
    if (NEW) one(A, A.xn, A.yn, A.zn, sab, eab, qab, en);
  }
}

template <bool MIXED, bool NEW, bool WRAP, class SH>
__device__ __forceinline__ void pair_sites_all(const SH& sh, const PairItem& b,
                                               const double L[3], int nlj, int a0, int a1,
                                               double& eo, double& en) {
  const int alj = a1 < nlj ? a1 : nlj;
  if (a0 < alj) pair_sites<MIXED, NEW, WRAP, true, false>(sh, b, L, a0, alj, eo, en);
  const int ar = a0 > nlj ? a0 : nlj;
  if (ar < a1) pair_sites<MIXED, NEW, WRAP, false, false>(sh, b, L, ar, a1, eo, en);
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
template <int NT, bool MIXED, bool NEW, int PC>
__device__ __forceinline__ void pair_phase(const HotBox& hb, const EvalShared<NT, PC>& sh,
                                           int nsame, int nwrap, double& e_old,
                                           double& e_new) {
  constexpr int NW = NT / 64;
  const int M = hb.max_len;
  const float rM = __builtin_amdgcn_rcpf((float)M);
  const int na = __builtin_amdgcn_readfirstlane(sh.n_real);
  const int nlj = __builtin_amdgcn_readfirstlane(sh.n_lj);
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
    const int2 r = sh.hit[wrap ? EvalShared<NT, PC>::kCap - 1 - h : h];
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
    if (MIXED) {
      b.s32 = sh.prm32[pk].s;
      b.e32 = sh.prm32[pk].e;
    }
    // a dummy site: no pairs, whatever its distance
    b.flags = in && p.real != 0.0 ? r.y & (kHitOld | kHitNew) : 0;
    if (!wrap) {
      // code 0, 1, 5 to k = 0, 1, -1; x - k L
      auto shift = [&](int at, double v, double Lx) {
        const unsigned c = (unsigned)r.y >> at;
        return fma(-__hiloint2double((int)((c & 1) * 0x3ff00000u | (c & 4) << 29), 0), Lx, v);
      };
      b.x = shift(kHitImage, b.x, L[0]);
      b.y = shift(kHitImage + 3, b.y, L[1]);
      b.z = shift(kHitImage + 6, b.z, L[2]);
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
      pair_sites_all<MIXED, NEW, true>(sh, b, L, nlj, a0, a1, eo, en);
    else
      pair_sites_all<MIXED, NEW, false>(sh, b, L, nlj, a0, a1, eo, en);
    // sites at zero distance (or no longer finite): again with the guard (a
    // shifted site's displacement is within L/2, so the wrap leaves it)
    if (__ballot(b.flags != 0 && !(fabs(eo) + fabs(en) < __builtin_huge_val()))) {
      eo = en = 0.0;
      pair_sites<MIXED, NEW, true, true, true>(sh, b, L, a0, a1, eo, en);
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
__device__ __forceinline__ int pick_source(const BoxView& bv, const double* nx,
                                           const double* ny, const double* nz,
                                           int p0, int mol, bool has_new) {
  if (bv.mode == MCGPU_NB_CELL && bv.cells.overflow[0] == 0) return MCGPU_NB_CELL;
  if (bv.mode == MCGPU_NB_VERLET && bv.verlet.stale[0] == 0 &&
      bv.verlet.count[mol] <= bv.verlet.cap) {
    const double* r = bv.verlet.ref + 3 * mol;
    if (has_new) {
      const double dx = wrap1(nx[p0] - r[0], bv.L[0]);
      const double dy = wrap1(ny[p0] - r[1], bv.L[1]);
      const double dz = wrap1(nz[p0] - r[2], bv.L[2]);
      if (dx * dx + dy * dy + dz * dz > bv.verlet.skin_half2) return MCGPU_NB_BRUTE;
    }
    return MCGPU_NB_VERLET;
  }
  return MCGPU_NB_BRUTE;
}

// Wave 0 (all 64 lanes): the cells of the old first primary sh.po and, when
// has_new, the proposed one sh.pn, lane d < 3 for axis d (other lanes repeat
// axis 2).
struct MoveCells {
  int co, cn;  // cell coordinates of this lane's axis
};

template <class SH>
__device__ __forceinline__ MoveCells move_cells(const BoxView& bv, const SH& sh, bool has_new) {
  const CellGrid& g = bv.cells;
  const int d = wlane() < 2 ? wlane() : 2;
  const int n = d == 0 ? g.n[0] : (d == 1 ? g.n[1] : g.n[2]);
  const double iw = d == 0 ? g.inv_w[0] : (d == 1 ? g.inv_w[1] : g.inv_w[2]);
  MoveCells c;
  c.co = cell_coord(sh.po[d], iw, n);
  c.cn = has_new ? cell_coord(sh.pn[d], iw, n) : c.co;
  return c;
}

// The cells around those of move_cells and their occupancies (from sh.ccount
// when lds_counts), as sh.cell; ncand the molecules in them.  The range along an axis follows make_range,
// one axis to a lane.  Candidate items are numbered cell_w to a cell, cell_w
// the largest occupancy, so a lane finds its cell by one division instead of
// a prefix and an item -> cell map (which cost a barrier); the lanes of free
// slots idle.  Returns false when the range exceeds 64 cells or an occupancy
// div_small's range (the caller then scans every molecule).
constexpr int kMaxCellItems = 1 << 20;

template <int NT, int PC>
__device__ __forceinline__ bool prepare_cells_wave(const BoxView& bv, EvalShared<NT, PC>& sh,
                                                   const MoveCells& mc, int* nitems,
                                                   int* ncand, int* cell_w,
                                                   bool lds_counts = false) {
  const CellGrid& g = bv.cells;
  const int lane = wlane();
  CellRange range;
  {
    const int d = lane < 2 ? lane : 2;
    const int n = d == 0 ? g.n[0] : (d == 1 ? g.n[1] : g.n[2]);
    int delta = mc.cn - mc.co;
    if (2 * delta > n) delta -= n;
    if (2 * delta < -n) delta += n;
    int lo = mc.co + (delta < 0 ? delta : 0) - 1;
    int cnt = (delta < 0 ? -delta : delta) + 3;
    lo = cnt >= n ? 0 : lo;
    cnt = cnt >= n ? n : cnt;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      range.lo[k] = readlane_i32(lo, k);
      range.cnt[k] = readlane_i32(cnt, k);
    }
  }
  const int total = range.total();
  if (total > 64) return false;
  int n = 0;
  if (lane < total) {
    const int c = range.cell(g, lane);
    n = lds_counts ? sh.ccount[c] : g.count[c];
    n = n < g.cap ? n : g.cap;
    sh.cell[lane] = make_int2(c * g.cap, n);
  }
  const int w = wave_max_i32(n);
  if (w > kMaxCellItems / 64) return false;
  *cell_w = w;
  *nitems = w * total;
  *ncand = (int)wave_sum_u32((unsigned)n);
  return true;
}

// wrap1, and k (0, 1.0 or -1.0, as the high word of a double) of d - k L.
__device__ __forceinline__ double wrap_k(double d, double L, int& k) {
  k = fabs(d) > 0.5 * L ? (__double2hiint(d) & (int)0x80000000) | 0x3ff00000 : 0;
  return fma(-__hiloint2double(k, 0), L, d);
}

// Candidate scan + pair phase over the prepared source (sh.src / nitems /
// cell_w and the cell table), for molecule `mol` at the LDS-held old position
// and (NEW) the proposed one.  Called by all NT threads after a barrier that
// follows the preparation.  prim_lds: the box's primaries are in sh.px/py/pz.
// Leaves per-wave partial sums in sh.red (and, in boxes that are not uniform,
// sh.redc) and ends with a barrier.  Returns the number of in-range molecules.
//
// Scan: one primary per molecule (bv.single_primary) takes about 45
// instructions a candidate, the next pass's candidates loading meanwhile; boxes with several primaries per
// molecule take the loops of primary_in_range.
template <int NT, bool MIXED, bool NEW, int PC>
__device__ __forceinline__ int eval_core(const BoxView& bv, const HotBox& hb,
                                         EvalShared<NT, PC>& sh, int mol, int jlo,
                                         bool prim_lds) {
  using SH = EvalShared<NT, PC>;
  constexpr int R = SH::kRound;
  constexpr int NW = NT / 64;
  const int t = threadIdx.x;
  const int src = __builtin_amdgcn_readfirstlane(sh.src);
  const int nitems = __builtin_amdgcn_readfirstlane(sh.nitems);
  const int cell_w = __builtin_amdgcn_readfirstlane(sh.cell_w);
  const float rw = __builtin_amdgcn_rcpf((float)cell_w);
  const int uni_len = hb.uni_len;
  const bool single = hb.single_primary;
  const double L0 = hb.L0, L1 = hb.L1, L2 = hb.L2, rc2 = hb.cutoff2;
  const double pox = sh.po[0], poy = sh.po[1], poz = sh.po[2];
  const double pnx = sh.pn[0], pny = sh.pn[1], pnz = sh.pn[2];
  const double limx = sh.lim[0], limy = sh.lim[1], limz = sh.lim[2];
  // molecule of a candidate item (-1: none)
  auto fetch = [&](int item) -> int {
    if (item >= nitems) return -1;
    if (src == MCGPU_NB_CELL) {
      const int k = div_small(item, rw);
      const int s = item - k * cell_w;
      const int2 c = sh.cell[k];
      return s < c.y ? bv.cells.slots[(unsigned)(c.x + s)] : -1;
    }
    if (src == MCGPU_NB_VERLET) return bv.verlet.list[mol * bv.verlet.cap + item];
    return jlo + item;
  };
  double eo = 0.0, en = 0.0;
  unsigned nsites = 0;  // sites of this lane's hits
  int nsame = 0, nwrap = 0, base = 0, hits = 0;
  for (;;) {
    // rounds of R passes while their hits fit
    while (base < nitems && nsame + nwrap + R * NT <= SH::kCap) {
      int2 rec[R];
      unsigned long long bsame[R], bwrap[R];
      unsigned c = 0;
      int jn = fetch(base + t);
#pragma unroll
      for (int p = 0; p < R; p++) {
        bsame[p] = bwrap[p] = 0;
        rec[p] = make_int2(0, 0);
        if (p > 0 && base + p * NT >= nitems) continue;  // block-uniform
        const int j = jn;
        if (p + 1 < R) jn = fetch(base + (p + 1) * NT + t);
        bool hit = false, wrap = false;
        if (j >= jlo && j != mol) {
          MolMeta mj;
          if (uni_len > 0) {  // uniform box: the record follows from the index
            mj.start = j * uni_len;
            mj.len = (int16_t)uni_len;
            mj.param = hb.uni_param;
          } else {
            mj = bv.meta[(unsigned)j];
          }
          int info;
          if (single) {
            double qx, qy, qz;
            if (PC > 0 && prim_lds) {
              qx = sh.px[j];
              qy = sh.py[j];
              qz = sh.pz[j];
            } else {
              qx = bv.px[(unsigned)j];
              qy = bv.py[(unsigned)j];
              qz = bv.pz[(unsigned)j];
            }
            int kx, ky, kz;
            const double dx = wrap_k(qx - pox, L0, kx);
            const double dy = wrap_k(qy - poy, L1, ky);
            const double dz = wrap_k(qz - poz, L2, kz);
            info = fma(dz, dz, fma(dy, dy, dx * dx)) <= rc2 ? kHitOld : 0;
            if (NEW) {
              const double ex = wrap1(qx - pnx, L0);
              const double ey = wrap1(qy - pny, L1);
              const double ez = wrap1(qz - pnz, L2);
              info |= fma(ez, ez, fma(ey, ey, ex * ex)) <= rc2 ? kHitNew : 0;
            }
            hit = info != 0;
            wrap = fabs(dx) > limx || fabs(dy) > limy || fabs(dz) > limz;
            info |= ((unsigned)kx >> 29 | ((unsigned)ky >> 29) << 3 | ((unsigned)kz >> 29) << 6)
                    << kHitImage;
          } else {
            const int ps = bv.mol_pidx_start[j], pc = bv.mol_pidx_count[j];
            const int npri = sh.npri;
            info = primary_in_range(bv, ps, pc, sh.ox, sh.oy, sh.oz, sh.pofs, npri) ? kHitOld : 0;
            if (NEW)
              info |=
                  primary_in_range(bv, ps, pc, sh.nx, sh.ny, sh.nz, sh.pofs, npri) ? kHitNew : 0;
            hit = info != 0;
            int kx, ky, kz;
            wrap = fabs(wrap_k(bv.px[ps] - pox, L0, kx)) > limx;
            wrap |= fabs(wrap_k(bv.py[ps] - poy, L1, ky)) > limy;
            wrap |= fabs(wrap_k(bv.pz[ps] - poz, L2, kz)) > limz;
            info |= ((unsigned)kx >> 29 | ((unsigned)ky >> 29) << 3 | ((unsigned)kz >> 29) << 6)
                    << kHitImage;
          }
          rec[p] = make_int2(mj.start, info | mj.len | mj.param << kHitParam);
          nsites += hit ? (unsigned)mj.len : 0u;
        }
        bsame[p] = __ballot(hit && !wrap);
        bwrap[p] = __ballot(hit && wrap);
        c += (unsigned)__popcll(bsame[p]) | (unsigned)__popcll(bwrap[p]) << 16;
      }
      // the waves' counts, and this wave's place among them
      if (wlane() == 0) sh.cnt[wave_id()] = c;
      __syncthreads();
      const unsigned mine = wlane() < NW ? sh.cnt[wlane()] : 0u;
      const unsigned incl = (unsigned)wave_incl_row_i32((int)mine);
      const unsigned total = (unsigned)readlane_i32((int)incl, NW - 1);
      const unsigned pre =
          (unsigned)readlane_i32((int)(incl - mine), __builtin_amdgcn_readfirstlane(wave_id()));
      int at0 = nsame + (int)(pre & 0xffff), at1 = nwrap + (int)(pre >> 16);
#pragma unroll
      for (int p = 0; p < R; p++) {
        const unsigned long long bit = 1ull << wlane();
        if (bsame[p] & bit) sh.hit[at0 + wave_rank(bsame[p])] = rec[p];
        if (bwrap[p] & bit) sh.hit[SH::kCap - 1 - at1 - wave_rank(bwrap[p])] = rec[p];
        at0 += __popcll(bsame[p]);
        at1 += __popcll(bwrap[p]);
      }
      nsame += (int)(total & 0xffff);
      nwrap += (int)(total >> 16);
      base += R * NT;
      __syncthreads();
    }
    hits += nsame + nwrap;
    pair_phase<NT, MIXED, NEW>(hb, sh, nsame, nwrap, eo, en);
    if (base >= nitems) break;
    __syncthreads();  // every lane is done with the hits before reuse
    nsame = nwrap = 0;
  }
  const double v = wave_row_sums(eo, en);
  if ((wlane() & 15) == 0) sh.red[(wlane() >> 4) * NW + wave_id()] = v;
  if (uni_len == 0) {
    nsites = wave_sum_u32(nsites);
    if (wlane() == 0) sh.redc[wave_id()] = nsites;
  }
  __syncthreads();
  return hits;
}

// Fixed-order totals of the per-wave partials left by eval_core, in every lane
// of the calling wave.
template <int NT, int PC>
__device__ __forceinline__ void eval_totals(const EvalShared<NT, PC>& sh, double& e_old,
                                            double& e_new) {
  constexpr int NW = NT / 64;
  const int k = wlane() & 31;
  double v = k < 2 * NW ? sh.red[(wlane() >> 5) * 2 * NW + k] : 0.0;
  v += dpp_f64<0xb1>(v);
  v += dpp_f64<0x4e>(v);
  v += dpp_f64<0x124>(v);
  v += dpp_f64<0x128>(v);
  wave_half_totals(v, e_old, e_new);
}

// Evaluates E_mol over candidates j >= jlo (j != mol) at the LDS-held old
// position, and (NEW) at the proposed position.  Must be called by all NT
// threads after load_molecule and a barrier.  Results are block-uniform.
template <int NT, bool MIXED, bool NEW, int PC>
__device__ __forceinline__ void eval_molecule(const BoxView& bv, const HotBox& hb, int mol, int jlo,
                                              EvalShared<NT, PC>& sh, double& e_old,
                                              double& e_new) {
  if (threadIdx.x < 64) {  // wave 0 prepares the neighbour source
    const int p0 = sh.pofs[0];
    int src = pick_source(bv, sh.nx, sh.ny, sh.nz, p0, mol, NEW);
    int nitems = 0, ncand = 0, cell_w = 1;
    if (src == MCGPU_NB_CELL &&
        !prepare_cells_wave(bv, sh, move_cells(bv, sh, NEW), &nitems, &ncand, &cell_w))
      src = MCGPU_NB_BRUTE;
    if (src == MCGPU_NB_VERLET) nitems = bv.verlet.count[mol];
    if (src == MCGPU_NB_BRUTE) nitems = bv.n_mol - jlo;
    if (src != MCGPU_NB_CELL) ncand = nitems;
    // A neighbour source never holds more candidates than molecules; if it
    // claims so its lists are corrupt: record it and evaluate nothing.
    int fault = 0;
    if (ncand < 0 || ncand > bv.n_mol) {
      fault = MCGPU_FAULT_CANDIDATES;
      nitems = 0;
    }
    if (threadIdx.x == 0) {
      sh.src = src;
      sh.nitems = nitems;
      sh.cell_w = cell_w;
      if (fault) sh.fault = fault;
    }
  }
  __syncthreads();
  eval_core<NT, MIXED, NEW>(bv, hb, sh, mol, jlo, false);
  eval_totals<NT>(sh, e_old, e_new);
  if (!NEW) e_new = 0.0;
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

// Writes the LDS-held proposed coordinates of `mol` into the box and keeps
// the primary mirror, cell lists and Verlet bookkeeping consistent.
template <int NT, int PC>
__device__ void commit_molecule(const BoxView& bv, int mol, const EvalShared<NT, PC>& sh) {
  const int t = threadIdx.x;
  const int start = bv.mol_start[mol];
  for (int k = t; k < sh.len; k += NT) {
    bv.x[start + k] = sh.nx[k];
    bv.y[start + k] = sh.ny[k];
    bv.z[start + k] = sh.nz[k];
  }
  if (t == 0) {
    const int ps = bv.mol_pidx_start[mol];
    for (int k = 0; k < sh.npri; k++) {
      bv.px[ps + k] = sh.nx[sh.pofs[k]];
      bv.py[ps + k] = sh.ny[sh.pofs[k]];
      bv.pz[ps + k] = sh.nz[sh.pofs[k]];
    }
    const int p0 = sh.pofs[0];
    if (bv.mode == MCGPU_NB_CELL && bv.cells.overflow[0] == 0) {
      const CellGrid& g = bv.cells;
      const int cnew = cell_index(g, cell_coord(sh.nx[p0], g.inv_w[0], g.n[0]),
                                  cell_coord(sh.ny[p0], g.inv_w[1], g.n[1]),
                                  cell_coord(sh.nz[p0], g.inv_w[2], g.n[2]));
      const int cold = g.mol_cell[mol];
      if (cnew != cold) cell_move(g, mol, cold, cnew);
    }
    if (bv.mode == MCGPU_NB_VERLET) {
      const double* r = bv.verlet.ref + 3 * mol;
      const double dx = wrap1(sh.nx[p0] - r[0], bv.L[0]);
      const double dy = wrap1(sh.ny[p0] - r[1], bv.L[1]);
      const double dz = wrap1(sh.nz[p0] - r[2], bv.L[2]);
      if (dx * dx + dy * dy + dz * dz > bv.verlet.skin_half2) bv.verlet.stale[0] = 1;
    }
  }
}

}  // namespace mcgpu
