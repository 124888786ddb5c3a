// Work-group level evaluation of one molecule's intermolecular energy at its
// current and (optionally) proposed position, in one pass over candidates.
//
// Preparation (wave 0): the neighbour source -- every molecule, the occupied
// slots of the cells spanning the old and proposed cell (their occupancies
// prefix-summed by a DPP wave scan, with an item -> cell map in LDS), or the
// Verlet list.
// Candidate scan (all lanes): each lane takes one candidate j, tests the
// primary-site cutoff at the old and proposed position (SimulationStep.cpp:
// 317-330), and the hits are compacted into LDS in candidate order (ballot +
// mbcnt, one barrier per pass).
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

template <int NT>
struct EvalShared {
  static constexpr int kCap = NT * 2 < 256 ? 256 : NT * 2;
  static constexpr int kItemCap = 2048;  // items with a cell entry in item_cell
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
  // in-range molecules of the current evaluation (hits), compacted:
  // site count | flags << 8 (bit0 old, bit1 new) | image code << 10 (see
  // image_code; the same for the old and the proposed position, else
  // kImageMixed)
  int32_t cand_lf[kCap];
  int32_t cand_start[kCap];  // first site
  int32_t cand_param[kCap];  // first site-parameter entry
  double ox[kMaxSites], oy[kMaxSites], oz[kMaxSites];
  double nx[kMaxSites], ny[kMaxSites], nz[kMaxSites];
  int32_t pofs[kMaxSites];   // primary offsets within the molecule
  int32_t cell_id[64];       // cells of the current range (at most 4x4x4)
  int32_t cell_pre[65];      // prefix of their occupancies
  uint8_t item_cell[kItemCap];  // range cell of each candidate item
  // copy of the box's cell occupancies, kept by launches that hold the box
  // for many moves (the batch kernel); prepare_cells_wave reads it when asked
  int32_t ccount[kCellLds];
  double red[kNW];
  double red2[kNW];
  unsigned long long redc[kNW];  // sites << 32 | candidates, per wave
  int32_t scan[2][kNW];          // hit counts per wave, double-buffered
  int32_t npri;
  int32_t len;
  int32_t n_real;   // entries of site
  int32_t n_lj;     // of which the first n_lj have an LJ term
  int32_t flag;
  int32_t fault;    // MCGPU_FAULT_* raised by the last preparation (0 = none)
  int32_t src;      // neighbour source of the current evaluation
  int32_t nitems;   // candidate items it holds
  int32_t ncells;   // cells of the range (cell source)
};

// Copies the box's site-parameter table into LDS (all threads; the caller
// places a barrier before it is read).  Tables are at most kParamCap entries
// (checked when a box is created).
template <int NT>
__device__ __forceinline__ void load_params(const BoxView& bv, EvalShared<NT>& sh) {
  for (int k = threadIdx.x; k < bv.n_param; k += NT) {
    sh.prm64[k] = bv.p64[k];
    sh.prm32[k] = bv.p32[k];
  }
}

// Wave 0: the moving molecule's sites into LDS (lane k < len holds site k at
// its old and proposed position; its parameters start at table entry
// `param`): by site for the scan and the commit, and the real sites as
// MoveSite records, those with an LJ term first, so that the pair phase runs
// the LJ arithmetic for those alone.  sh.prm64/prm32 must be loaded.
template <int NT>
__device__ __forceinline__ void stage_move(EvalShared<NT>& sh, int len, int param, double xo,
                                           double yo, double zo, double xn, double yn,
                                           double zn) {
  const int lane = wlane();
  SiteParam64 p{0.0, 0.0, 0.0, 0.0};
  SiteParam32 p32{0.0f, 0.0f, 0.0f, 0.0f};
  if (lane < len) {
    p = sh.prm64[param + lane];
    p32 = sh.prm32[param + lane];
    sh.ox[lane] = xo;
    sh.oy[lane] = yo;
    sh.oz[lane] = zo;
    sh.nx[lane] = xn;
    sh.ny[lane] = yn;
    sh.nz[lane] = zn;
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
template <int NT>
__device__ __forceinline__ void load_molecule(const BoxView& bv, int mol, const double* nxyz,
                                              EvalShared<NT>& sh) {
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
  stage_move(sh, len, pbase, xo, yo, zo, xn, yn, zn);
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

// floor(u / m) for u < 65536, 1 <= m <= 32, with magic = 2^32 / m + 1.
__device__ __forceinline__ int div_small(int u, unsigned long long magic) {
  return (int)(((unsigned long long)(unsigned)u * magic) >> 32);
}

// One item of the pair phase: a site b of a hit, held by one lane.
struct PairItem {
  double x, y, z;     // shifted by the periodic image of its hit
  double s, e, q;     // pair parameters
  float s32, e32;
  int flags;          // bit0: in range of the old position, bit1: of the new
  bool wrap;          // its pairs take wrap1 per axis (kImageMixed)
};

// Sum over the moving molecule's sites [a0, a1) of their pairs with item b,
// at the old and (NEW) the proposed position.  LJ: the sites have an LJ term.
// WRAP: items with b.wrap take the reference's wrap per site pair.  GUARD:
// r^2 == 0 contributes nothing; without it such a pair makes the sum
// non-finite and the caller repeats the sum with GUARD.
template <int NT, bool MIXED, bool NEW, bool WRAP, bool LJ, bool GUARD>
__device__ __forceinline__ void pair_sites(const EvalShared<NT>& sh, const PairItem& b,
                                           const double L[3], int a0, int a1, double& eo,
                                           double& en) {
  // a lane that needs no wrap adds k * 0
  const double L0 = WRAP && b.wrap ? L[0] : 0.0;
  const double L1 = WRAP && b.wrap ? L[1] : 0.0;
  const double L2 = WRAP && b.wrap ? L[2] : 0.0;
  const double h0 = 0.5 * L[0], h1 = 0.5 * L[1], h2 = 0.5 * L[2];
  auto wrap = [](double d, double h, double Lx) {
    const double k = d < -h ? 1.0 : (d > h ? -1.0 : 0.0);
    return fma(k, Lx, d);
  };
  auto one = [&](const MoveSite& A, double x, double y, double z, double sab, double eab,
                 double qab, double& acc) {
    double dx = b.x - x, dy = b.y - y, dz = b.z - z;
    if (WRAP) {
      dx = wrap(dx, h0, L0);
      dy = wrap(dy, h1, L1);
      dz = wrap(dz, h2, L2);
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

template <int NT, bool MIXED, bool NEW, bool WRAP>
__device__ __forceinline__ void pair_sites_all(const EvalShared<NT>& sh, const PairItem& b,
                                               const double L[3], int nlj, int a0, int a1,
                                               double& eo, double& en) {
  const int alj = a1 < nlj ? a1 : nlj;
  if (a0 < alj) pair_sites<NT, MIXED, NEW, WRAP, true, false>(sh, b, L, a0, alj, eo, en);
  const int ar = a0 > nlj ? a0 : nlj;
  if (ar < a1) pair_sites<NT, MIXED, NEW, WRAP, false, false>(sh, b, L, ar, a1, eo, en);
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
template <int NT, bool MIXED, bool NEW>
__device__ __forceinline__ void pair_phase(const BoxView& bv, const EvalShared<NT>& sh,
                                           int nhits, double& e_old, double& e_new) {
  constexpr int NW = NT / 64;
  const int M = bv.max_len;
  const unsigned long long magic = (1ull << 32) / (unsigned)M + 1ull;
  const int na = __builtin_amdgcn_readfirstlane(sh.n_real);
  const int nlj = __builtin_amdgcn_readfirstlane(sh.n_lj);
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  const double L[3] = {bv.L[0], bv.L[1], bv.L[2]};
  const int tot = nhits * M;
  const int nblk = (tot + 63) >> 6;
  const int steps = nblk * na;
  int u = steps * w / NW;
  const int u_end = steps * (w + 1) / NW;
  if (u >= u_end) return;
  // u / na for u < 2^15 (steps <= kCap * 32 / 64 * 32): (u + 0.5) / na lies
  // at least 0.5 / na from an integer, far beyond the reciprocal's error
  int blk = __builtin_amdgcn_readfirstlane(
      (int)(((float)u + 0.5f) * __builtin_amdgcn_rcpf((float)na)));
  int a0 = u - blk * na;
  auto load = [&](int k) {
    PairItem b{1e30, 1e30, 1e30, 0.0, 0.0, 0.0, 0.0f, 0.0f, 0, false};
    const int item = k * 64 + wlane();
    if (item < tot) {
      const int h = div_small(item, magic);
      const int o = item - h * M;
      const int lf = sh.cand_lf[h];
      if (o < (lf & 0xff)) {
        const int img = (lf >> 10) & 0x7f;
        b.wrap = img & kImageMixed;
        const int site = sh.cand_start[h] + o;
        b.x = bv.x[site] + (b.wrap ? 0.0 : image_shift(img & 3, L[0]));
        b.y = bv.y[site] + (b.wrap ? 0.0 : image_shift((img >> 2) & 3, L[1]));
        b.z = bv.z[site] + (b.wrap ? 0.0 : image_shift((img >> 4) & 3, L[2]));
        b.flags = (lf >> 8) & 3;
        const int pk = sh.cand_param[h] + o;
        const SiteParam64 p = sh.prm64[pk];
        b.s = p.s;
        b.e = p.e;
        b.q = p.q;
        if (MIXED) {
          b.s32 = sh.prm32[pk].s;
          b.e32 = sh.prm32[pk].e;
        }
        // a dummy site: no pairs, whatever its distance
        if (p.real == 0.0) b.flags = 0;
      }
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
    if (__ballot(b.wrap))
      pair_sites_all<NT, MIXED, NEW, true>(sh, b, L, nlj, a0, a1, eo, en);
    else
      pair_sites_all<NT, MIXED, NEW, false>(sh, b, L, nlj, a0, a1, eo, en);
    // sites at zero distance (or no longer finite): again with the guard
    if (__ballot(b.flags != 0 && !(fabs(eo) + fabs(en) < __builtin_huge_val()))) {
      eo = en = 0.0;
      pair_sites<NT, MIXED, NEW, true, true, true>(sh, b, L, a0, a1, eo, en);
    }
    e_old += b.flags & 1 ? eo : 0.0;
    e_new += b.flags & 2 ? en : 0.0;
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

// Wave 0 (all 64 lanes): the cells around old cell co and proposed cell cn,
// their occupancies (from sh.ccount when lds_counts), the prefix and, when
// fill, the item -> cell map (else the caller fills it with
// fill_item_cells).  Returns the cell count, or -1 when the range exceeds 64
// cells (the caller then scans every molecule); *nitems receives the
// candidate count.
template <int NT>
__device__ __forceinline__ int prepare_cells_wave(const BoxView& bv,
                                                  EvalShared<NT>& sh,
                                                  const int co[3], const int cn[3],
                                                  int* nitems, bool lds_counts = false,
                                                  bool fill = true) {
  const CellGrid& g = bv.cells;
  const CellRange range = make_range(g, co, cn);
  const int ncells = range.total();
  if (ncells > 64) return -1;
  const int lane = wlane();
  int n = 0, c = 0;
  if (lane < ncells) {
    c = range.cell(g, lane);
    n = lds_counts ? sh.ccount[c] : g.count[c];
    n = n < g.cap ? n : g.cap;
    sh.cell_id[lane] = c;
  }
  const int incl = wave_incl_scan_i32(n);
  sh.cell_pre[lane + 1] = incl;
  if (lane == 0) sh.cell_pre[0] = 0;
  if (fill) {
    const int end = incl < EvalShared<NT>::kItemCap ? incl : EvalShared<NT>::kItemCap;
    for (int k = incl - n; k < end; k++) sh.item_cell[k] = (uint8_t)lane;
  }
  *nitems = readlane_i32(incl, 63);
  return ncells;
}

// All NT threads: the item -> cell map of the ncells cells whose prefix
// prepare_cells_wave left in sh.cell_pre, NT / 64 threads per cell.  The
// caller places a barrier before and after it.
template <int NT>
__device__ __forceinline__ void fill_item_cells(EvalShared<NT>& sh, int ncells) {
  constexpr int kPer = NT / 64;
  const int c = threadIdx.x / kPer;
  if (c < ncells) {
    const int lim = EvalShared<NT>::kItemCap;
    int end = sh.cell_pre[c + 1];
    end = end < lim ? end : lim;
    for (int k = sh.cell_pre[c] + (int)threadIdx.x % kPer; k < end; k += kPer)
      sh.item_cell[k] = (uint8_t)c;
  }
}

// The range cell holding candidate `item` of the cell source.
template <int NT>
__device__ __forceinline__ int item_cell_of(const EvalShared<NT>& sh, int item,
                                            int ncells) {
  if (item < EvalShared<NT>::kItemCap) return sh.item_cell[item];
  int lo = 0, hi = ncells;  // last cell whose prefix <= item
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (sh.cell_pre[mid] <= item) lo = mid; else hi = mid;
  }
  return lo;
}

// Candidate scan + pair phase over the prepared source (sh.src / nitems /
// ncells and the cell tables), for molecule `mol` at the LDS-held old
// position and, when has_new, the proposed one.  Called by all NT threads
// after a barrier that follows the preparation.  Leaves per-wave partial
// sums in sh.red / red2 / redc and ends with a barrier.  The candidate and
// site counts are per-wave ballot counts.  NEW: evaluate the proposed
// position too.
template <int NT, bool MIXED, bool NEW>
__device__ __forceinline__ void eval_core(const BoxView& bv, EvalShared<NT>& sh,
                                          int mol, int jlo) {
  const int t = threadIdx.x;
  const int src = __builtin_amdgcn_readfirstlane(sh.src);
  const int nitems = __builtin_amdgcn_readfirstlane(sh.nitems);
  const int ncells = __builtin_amdgcn_readfirstlane(sh.ncells);
  const int npri = __builtin_amdgcn_readfirstlane(sh.npri);
  const int uni_len = bv.uni_len;
  double eo = 0.0, en = 0.0;
  unsigned ncand_w = 0, nsites_w = 0;  // this wave's candidates and hit sites
  int nhits = 0, par = 0;
  int base = 0;
  for (;;) {
  while (base < nitems) {
    const int item = base + t;
    int j = -1;
    if (item < nitems) {
      if (src == MCGPU_NB_CELL) {
        const int lo = item_cell_of(sh, item, ncells);
        j = bv.cells.slots[sh.cell_id[lo] * bv.cells.cap + (item - sh.cell_pre[lo])];
      } else if (src == MCGPU_NB_VERLET) {
        j = bv.verlet.list[mol * bv.verlet.cap + item];
      } else {
        j = jlo + item;
      }
    }
    int f = 0;
    MolMeta mj{0, 0, 0, 0, 0};
    const bool cand = j >= jlo && j != mol;
    const unsigned ncand = (unsigned)__popcll(__ballot(cand));
    if (cand) {
      if (uni_len > 0) {  // uniform box: the record follows from the index
        mj.start = j * uni_len;
        mj.len = (int16_t)uni_len;
        mj.param = bv.uni_param;
        mj.pstart = j;
      } else {
        mj = bv.meta[j];
      }
      int ps = j, pc = 1;  // one primary per molecule: no indirection
      if (!bv.single_primary) {
        ps = mj.pstart;
        pc = bv.mol_pidx_count[j];
      }
      f = primary_in_range(bv, ps, pc, sh.ox, sh.oy, sh.oz, sh.pofs, npri) ? 1 : 0;
      if (NEW)
        f |= primary_in_range(bv, ps, pc, sh.nx, sh.ny, sh.nz, sh.pofs, npri) ? 2 : 0;
      if (f) {
        // periodic image of the pair, from the first primaries
        const int o = sh.pofs[0];
        const double qx = bv.px[ps], qy = bv.py[ps], qz = bv.pz[ps];
        int img = image_code(qx - sh.ox[o], qy - sh.oy[o], qz - sh.oz[o], bv.L, bv.reach2);
        if (NEW &&
            image_code(qx - sh.nx[o], qy - sh.ny[o], qz - sh.nz[o], bv.L, bv.reach2) != img)
          img = kImageMixed;
        f |= img << 2;
      }
    }
    // compaction: rank within the wave, wave counts through LDS
    const unsigned long long bal = __ballot(f != 0);
    if (wlane() == 0) sh.scan[par][wave_id()] = __popcll(bal);
    __syncthreads();
    int pre = 0, total = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; w++) {
      const int c = sh.scan[par][w];
      pre += (w < wave_id()) ? c : 0;
      total += c;
    }
    par ^= 1;
    if (nhits + total > EvalShared<NT>::kCap) break;  // block-uniform: full, scan this pass again
    ncand_w += ncand;
    if (uni_len > 0)
      nsites_w += (unsigned)__popcll(bal) * (unsigned)uni_len;
    else
      nsites_w += wave_sum_u32(f ? (unsigned)mj.len : 0u);
    if (f) {
      const int pos = nhits + pre + wave_rank(bal);
      sh.cand_start[pos] = mj.start;
      sh.cand_param[pos] = mj.param;
      sh.cand_lf[pos] = mj.len | (f << 8);
    }
    nhits += total;
    base += NT;
  }
  __syncthreads();
  if (nhits > 0) pair_phase<NT, MIXED, NEW>(bv, sh, nhits, eo, en);
  if (base >= nitems) break;
  __syncthreads();  // every lane is done with the hits before reuse
  nhits = 0;
  }
  eo = wave_sum_f64(eo);
  if (NEW) en = wave_sum_f64(en);
  if (wlane() == 0) {
    sh.red[wave_id()] = eo;
    sh.red2[wave_id()] = en;
    sh.redc[wave_id()] = ((unsigned long long)nsites_w << 32) | ncand_w;
  }
  __syncthreads();
}

// Fixed-order totals of the per-wave partials left by eval_core.
template <int NT>
__device__ __forceinline__ void eval_totals(const EvalShared<NT>& sh, double& e_old,
                                            double& e_new, unsigned long long& counts) {
  double so = 0.0, sn = 0.0;
  unsigned long long c = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; w++) {
    so += sh.red[w];
    sn += sh.red2[w];
    c += sh.redc[w];
  }
  e_old = so;
  e_new = sn;
  counts = c;
}

// Evaluates E_mol over candidates j >= jlo (j != mol) at the LDS-held old
// position, and (NEW) at the proposed position.  Must be called by all NT
// threads after load_molecule and a barrier.  Results are block-uniform.
template <int NT, bool MIXED, bool NEW>
__device__ __forceinline__ void eval_molecule(const BoxView& bv, int mol, int jlo,
                                              EvalShared<NT>& sh, double& e_old,
                                              double& e_new) {
  if (threadIdx.x < 64) {  // wave 0 prepares the neighbour source
    const int p0 = sh.pofs[0];
    int src = pick_source(bv, sh.nx, sh.ny, sh.nz, p0, mol, NEW);
    int nitems = 0, ncells = 0;
    if (src == MCGPU_NB_CELL) {
      const CellGrid& g = bv.cells;
      int co[3], cn[3];
      co[0] = cell_coord(sh.ox[p0], g.inv_w[0], g.n[0]);
      co[1] = cell_coord(sh.oy[p0], g.inv_w[1], g.n[1]);
      co[2] = cell_coord(sh.oz[p0], g.inv_w[2], g.n[2]);
      if (NEW) {
        cn[0] = cell_coord(sh.nx[p0], g.inv_w[0], g.n[0]);
        cn[1] = cell_coord(sh.ny[p0], g.inv_w[1], g.n[1]);
        cn[2] = cell_coord(sh.nz[p0], g.inv_w[2], g.n[2]);
      } else {
        cn[0] = co[0];
        cn[1] = co[1];
        cn[2] = co[2];
      }
      ncells = prepare_cells_wave(bv, sh, co, cn, &nitems);
      if (ncells < 0) {
        src = MCGPU_NB_BRUTE;
        ncells = 0;
      }
    }
    if (src == MCGPU_NB_VERLET) nitems = bv.verlet.count[mol];
    if (src == MCGPU_NB_BRUTE) nitems = bv.n_mol - jlo;
    // A neighbour source never holds more candidates than molecules; if it
    // claims so its lists are corrupt: record it and evaluate nothing.
    int fault = 0;
    if (nitems < 0 || nitems > bv.n_mol) {
      fault = MCGPU_FAULT_CANDIDATES;
      nitems = 0;
    }
    if (threadIdx.x == 0) {
      sh.src = src;
      sh.nitems = nitems;
      sh.ncells = ncells;
      if (fault) sh.fault = fault;
    }
  }
  __syncthreads();
  eval_core<NT, MIXED, NEW>(bv, sh, mol, jlo);
  unsigned long long c;
  eval_totals<NT>(sh, e_old, e_new, c);
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
template <int NT>
__device__ void commit_molecule(const BoxView& bv, int mol,
                                const EvalShared<NT>& sh) {
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
