// Full-system energy on the device, a throughput kernel body shared by the
// single-box and batched paths.
#pragma once

#include "cells.h"
#include "device_common.h"
#include "eval.h"
#include "wave.h"

namespace mcgpu {

// Full-system energy (SimulationStep.cpp:40-71: every molecule pair within
// the primary cutoff of SimulationStep.cpp:317-330 once), one wave per
// molecule i, or several that share its candidates (full_split), and no
// barriers between waves:
//  * the lanes scan i's candidate partners -- with cell lists, i's own cell
//    (partners j > i) and the 13 neighbour cells on one side of it (any j),
//    so that every pair of cells is visited from one end only, or, with
//    fewer than 3 cells along an axis, every cell around i (j > i); without
//    cell lists, all j > i.  kFullWindows windows of 64 candidates are loaded
//    together (a window is a chain of two loads), and a candidate that is no
//    hit, six in seven, costs the distance test alone;
//  * the hits' ids are compacted into the wave's LDS list by ballot, and one
//    lane per hit turns them into the move kernels' records: from the front
//    those whose pairs share one periodic image, from the back those whose
//    site pairs may wrap differently;
//  * every site b of the hits is an item, 64 to a block; a lane loads its item
//    straight from the box while the previous block is summed, and takes it
//    against i's real sites, whose records are LDS broadcasts (pair_sites).
// Each block writes the sum of its waves; those are reduced in a fixed order
// elsewhere, so the total is deterministic.  Which molecule of a pair holds
// its terms differs from the reference's E_i(i) split (j > i); the set of
// pairs, and so the total up to summation order, is the same.
//
// Bound by the vector ALUs once the chip is full: they issue 61% of the time on
// a mixture of 20,000 molecules (22.8 million site pairs, 1,745 vector
// instructions a molecule).  us of the launch by its events, former kernel (hits'
// sites staged in LDS, two windows' bitmaps to map items) -> this one: mixture of
// 20,000 114.7 -> 94.9, bicyclic of 4,000 45.5 -> 42.5, of 1,733 35.1 -> 29.8 and
// of 512 (all pairs, MIXED) 39.4 -> 19.0, water of 4,096 MIXED 23.0 -> 20.6, of
// 700 17.2 -> 8.7.  Not kept (against 91 then): the block's four waves taking
// molecules of one cell and staging their candidates together (mixture of 20,000
// 110: the barriers cost more than the gathers saved), 3 or 4 windows (100, 114).
constexpr int kFullWindows = 2;  // windows of 64 candidates loaded together
constexpr int kFullHits = 64 * kFullWindows + 128;  // hits held before their pairs are summed
constexpr int kFullMap = 128;  // hits mapped to items at a time (boxes not uniform)
constexpr int kFullCells = 27;   // cells of one scan
// Boxes whose largest molecule has at least this many sites split the pairs
// by index parity over all 27 cells instead of the half shell: a molecule's
// share of the pair work then varies far less (per-SIMD maximum over mean
// 1.17 against 1.63 on a 4,000-molecule 16-site box), which pays for
// scanning twice the cells when each hit carries ~100+ site pairs.
constexpr int kParityLen = 8;

// A real site of molecule i as pair_sites reads it.
struct FullSite {
  double xo, yo, zo;
  double s, e, q;
  float s32, e32;
};

struct WaveEval {
  FullSite site[kMaxSites];
  int32_t id[kFullHits];  // the hits' molecules
  int2 hit[kFullHits];    // and records (kHitImage, kHitParam)
  // of a chunk's hits: first item, and a bitmap of the first items
  uint16_t first[kFullMap];
  unsigned long long marks[kFullMap * kMaxSites / 64];
  int2 cell[kScanEntries];  // cells of the scan, or pieces: first slot, occupancy; own first
};

// Pairs of hits [0, n) of one kind with i's sites (na, the first nlj of which
// have an LJ term); npairs counts the site pairs.
template <bool MIXED, bool WRAP>
__device__ __forceinline__ double full_pairs(const HotBox& hb, WaveEval& W,
                                             const SiteParam64* P, int na, int nlj, int n,
                                             unsigned& npairs) {
  const int lane = wlane();
  const double L[3] = {hb.L0, hb.L1, hb.L2};
  const int len = hb.uni_len;
  const float rlen = __builtin_amdgcn_rcpf((float)(len > 0 ? len : 1));
  const int step = len > 0 ? n : kFullMap;  // a uniform box maps by division
  double e = 0.0;
  for (int h0 = 0; h0 < n; h0 += step) {  // wave-uniform
    const int nh = n - h0 < step ? n - h0 : step;
    int items = nh * len;
    if (len == 0) {
      // first items of the chunk's hits, and their marks
      __builtin_amdgcn_wave_barrier();
      W.marks[lane] = 0ull;
      static_assert(kFullMap * kMaxSites / 64 == 64, "one word a lane");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int c = 0; c < kFullMap; c += 64) {
        const int h = c + lane;
        const int l = h < nh ? W.hit[WRAP ? kFullHits - 1 - (h0 + h) : h0 + h].y & 63 : 0;
        const int incl = wave_incl_scan_i32(l);
        const int f = items + incl - l;
        if (h < nh) {
          W.first[h] = (uint16_t)f;
          atomicOr(&W.marks[f >> 6], 1ull << (f & 63));
        }
        items += readlane_i32(incl, 63);
      }
      __builtin_amdgcn_wave_barrier();
    }
    const int nblk = (items + 63) >> 6;
    int before = -1;  // hits whose first item lies before the block, less one
    auto load = [&](int k) {
      PairItem b;
      const int item = k * 64 + lane;
      const int it = item < items ? item : items - 1;  // a valid address
      int h, o;
      if (len > 0) {
        h = div_small(it, rlen);
        o = it - h * len;
      } else {
        const unsigned long long word = W.marks[k];
        // marks at the block's positions 0..it (2 << 63 wraps to 0: all bits)
        h = before + __popcll(word & ((2ull << (it & 63)) - 1ull));
        before += __popcll(word);
        o = it - W.first[h];
      }
      const int2 r = W.hit[WRAP ? kFullHits - 1 - (h0 + h) : h0 + h];
      const unsigned site = (unsigned)(r.x + o);
      b.x = hb.x[site];
      b.y = hb.y[site];
      b.z = hb.z[site];
      const SiteParam64 p = P[((unsigned)r.y >> kHitParam) + o];
      b.s = p.s;
      b.e = p.e;
      b.q = p.q;
      if (MIXED) mixed_item(b, p);
      b.flags = item < items && p.real != 0.0 ? kHitOld : 0;  // dummy sites: no pairs
      if (!WRAP) {
        b.x = image_shifted(r.y, kHitImage, b.x, L[0]);
        b.y = image_shifted(r.y, kHitImage + 3, b.y, L[1]);
        b.z = image_shifted(r.y, kHitImage + 6, b.z, L[2]);
      }
      return b;
    };
    PairItem b = load(0);
    for (int k = 0; k < nblk; k++) {
      PairItem next = b;
      if (k + 1 < nblk) next = load(k + 1);
      double v = 0.0, unused = 0.0;
      if (nlj > 0) pair_sites<MIXED, false, WRAP, true, false>(W, b, L, 0, nlj, v, unused);
      if (nlj < na) pair_sites<MIXED, false, WRAP, false, false>(W, b, L, nlj, na, v, unused);
      // sites at zero distance (or no longer finite): again with the guard
      if (__ballot(b.flags != 0 && !(fabs(v) < __builtin_huge_val()))) {
        v = 0.0;
        pair_sites<MIXED, false, true, true, true>(W, b, L, 0, na, v, unused);
      }
      e += b.flags ? v : 0.0;
      npairs += (unsigned)(__popcll(__ballot(b.flags != 0)) * na);
      b = next;
    }
  }
  return e;
}

// Share `part` of `split` of molecule i's part of the full energy, lane by
// lane (windows of 64 candidates dealt in turn); pairs counts the real site
// pairs summed (wave-uniform).
template <bool MIXED>
__device__ __forceinline__ double wave_molecule_energy(const BoxView& bv, const HotBox& hb,
                                                       WaveEval& W, int i, int part, int split,
                                                       const SiteParam64* P, unsigned& pairs) {
  const int lane = wlane();
  int start, len, param, psi, pci;
  if (hb.uni_len > 0) {
    len = hb.uni_len;
    start = i * len;
    param = hb.uni_param;
    psi = i;
    pci = 1;
  } else {
    const MolMeta m = hb.meta[i];
    start = m.start;
    len = m.len;
    param = m.param;
    psi = hb.single_primary ? i : m.pstart;
    pci = hb.single_primary ? 1 : bv.mol_pidx_count[i];
  }
  // the primaries of i (at most kMaxSites) as lane values
  double pix = 0.0, piy = 0.0, piz = 0.0;
  if (lane < pci) {
    pix = hb.px[psi + lane];
    piy = hb.py[psi + lane];
    piz = hb.pz[psi + lane];
  }
  // i's real sites, those with an LJ term first
  int na, nlj;
  {
    SiteParam64 p{0.0, 0.0, 0.0, 0.0};
    double x = 0.0, y = 0.0, z = 0.0;
    if (lane < len) {
      x = hb.x[start + lane];
      y = hb.y[start + lane];
      z = hb.z[start + lane];
      p = P[param + lane];
    }
    const bool lj = p.real != 0.0 && p.e != 0.0;
    const bool rest = p.real != 0.0 && !lj;
    const unsigned long long blj = __ballot(lj), brest = __ballot(rest);
    nlj = __popcll(blj);
    na = nlj + __popcll(brest);
    const int at = lj ? wave_rank(blj) : nlj + wave_rank(brest);
    const float e32 = (float)p.e;
    if (lj || rest)
      W.site[at] = FullSite{x, y, z, p.s, p.e, p.q, e32 != 0.0f ? (float)p.s : 0.0f, e32};
  }
  const double p0x = readlane_f64(pix, 0), p0y = readlane_f64(piy, 0),
               p0z = readlane_f64(piz, 0);
  const double L0 = hb.L0, L1 = hb.L1, L2 = hb.L2, rc2 = hb.cutoff2;
  // how far a candidate's wrapped displacement may be for its site pairs to
  // share one image (see stage_move)
  const double limx = 0.5 * L0 - hb.reach2, limy = 0.5 * L1 - hb.reach2,
               limz = 0.5 * L2 - hb.reach2;
  // candidate items: without cells, j = i + 1 + item; with cells, cell_w to an
  // entry of the cell table (scan_width), so that a lane finds its entry by one
  // division
  const CellGrid& g = bv.cells;
  // (a scan of more items than div_small divides takes every molecule)
  const bool cells = hb.mode == MCGPU_NB_CELL && g.overflow[0] == 0 &&
                     g.cap <= kMaxScanItems / kFullCells;
  int nitems = hb.n_mol - (i + 1), cell_w = 1;
  int own = 0;  // items whose partners must exceed i
  bool parity = false;
  if (cells) {
    int co[3];
    co[0] = cell_coord(p0x, g.inv_w[0], g.n[0]);
    co[1] = cell_coord(p0y, g.inv_w[1], g.n[1]);
    co[2] = cell_coord(p0z, g.inv_w[2], g.n[2]);
    const bool shell = g.n[0] >= 3 && g.n[1] >= 3 && g.n[2] >= 3;
    // by parity: all 27 cells around i; i holds the pair with j when i + j is
    // even and j > i, or odd and j < i (every pair once, from either end)
    parity = shell && bv.max_len >= kParityLen;
    int ncell, c = 0;
    if (shell) {
      // own cell + the 13 offsets (dx, dy, dz) > (0, 0, 0) lexicographically,
      // or (parity) all, own in the middle
      ncell = parity ? 27 : 14;
      const int t = parity ? lane : lane + 13;
      if (lane < ncell) {
        int a = co[0] + t / 9 - 1, b = co[1] + (t / 3) % 3 - 1, d = co[2] + t % 3 - 1;
        a += a < 0 ? g.n[0] : 0;
        a -= a >= g.n[0] ? g.n[0] : 0;
        b += b < 0 ? g.n[1] : 0;
        b -= b >= g.n[1] ? g.n[1] : 0;
        d += d < 0 ? g.n[2] : 0;
        d -= d >= g.n[2] ? g.n[2] : 0;
        c = cell_index(g, a, b, d);
      }
    } else {
      // fewer than 3 cells along some axis: every cell around i, j > i
      const CellRange r = make_range(g, co, co);
      ncell = r.total();
      if (lane < ncell) c = r.cell(g, lane);
    }
    int cnt = 0;
    if (lane < ncell) {
      cnt = g.count[c];
      cnt = cnt < g.cap ? cnt : g.cap;
      W.cell[lane] = make_int2(c * g.cap, cnt);
    }
    const int largest = wave_max_i32(cnt);
    cell_w = largest;
    // (only beyond twice the box's mean is the sum worth its instructions)
    if (__builtin_expect((float)largest * (float)cells_total(g) > 2.0f * (float)hb.n_mol, 0))
      cell_w = scan_width(ncell, largest, (int)wave_sum_u32((unsigned)cnt), 64 * kFullWindows);
    int entries = ncell, own_entries = 1;
    if (__builtin_expect(cell_w < largest, 0)) {  // wave-uniform: pieces, in the cells' order
      const float rw = __builtin_amdgcn_rcpf((float)cell_w);
      const int n = cnt > 0 ? div_small(cnt + cell_w - 1, rw) : 0;
      const int incl = wave_incl_scan_i32(n);
      for (int q = 0; q < n; q++)
        W.cell[incl - n + q] = piece_of(c * g.cap, cnt, q, cell_w);
      entries = readlane_i32(incl, 63);
      own_entries = readlane_i32(n, 0);
    }
    nitems = entries * cell_w;
    own = parity ? 0 : (shell ? own_entries * cell_w : nitems);
  }
  const float rw = __builtin_amdgcn_rcpf((float)(cell_w > 0 ? cell_w : 1));
  __builtin_amdgcn_wave_barrier();
  double e = 0.0;
  unsigned np = 0;
  int nh = 0;
  const int stride = 64 * split;
  for (int base = 64 * part; base < nitems; base += kFullWindows * stride) {
    int j[kFullWindows];
    double qx[kFullWindows], qy[kFullWindows], qz[kFullWindows];
#pragma unroll
    for (int w = 0; w < kFullWindows; w++) {
      if (w > 0 && base + w * stride >= nitems) continue;  // wave-uniform
      const int item = base + w * stride + lane;
      const int it = item < nitems ? item : nitems - 1;
      if (cells) {
        const int k = div_small(it, rw);
        const int s = it - k * cell_w;
        const int2 c = W.cell[k];
        const bool in = item < nitems && s < c.y;
        const int v = hb.slots[(unsigned)(in ? c.x + s : c.x)];
        const bool ok = in && v != i &&
                        (parity ? (((i ^ v) & 1) == 0) == (v > i) : (item >= own || v > i));
        j[w] = ok ? v : -1;
      } else {
        j[w] = item < nitems ? i + 1 + it : -1;
      }
    }
#pragma unroll
    for (int w = 0; w < kFullWindows; w++) {
      if (w > 0 && base + w * stride >= nitems) continue;
      const unsigned jj = (unsigned)(j[w] >= 0 ? j[w] : i);  // every lane loads a valid entry
      const unsigned pj = hb.single_primary ? jj : (unsigned)bv.mol_pidx_start[jj];
      qx[w] = hb.px[pj];
      qy[w] = hb.py[pj];
      qz[w] = hb.pz[pj];
    }
#pragma unroll
    for (int w = 0; w < kFullWindows; w++) {
      if (w > 0 && base + w * stride >= nitems) continue;
      const double dx = wrap1(qx[w] - p0x, L0);
      const double dy = wrap1(qy[w] - p0y, L1);
      const double dz = wrap1(qz[w] - p0z, L2);
      bool hit = fma(dz, dz, fma(dy, dy, dx * dx)) <= rc2;
      if (!hb.single_primary && j[w] >= 0) {
        const int psj = bv.mol_pidx_start[j[w]];
        const int pcj = bv.mol_pidx_count[j[w]];
        for (int q = 0; q < pcj; q++) {
          const double ax = hb.px[psj + q], ay = hb.py[psj + q], az = hb.pz[psj + q];
          for (int p = 0; p < pci; p++) {
            const double ex = wrap1(ax - readlane_f64(pix, p), L0);
            const double ey = wrap1(ay - readlane_f64(piy, p), L1);
            const double ez = wrap1(az - readlane_f64(piz, p), L2);
            hit |= ex * ex + ey * ey + ez * ez <= rc2;
          }
        }
      }
      hit = hit && j[w] >= 0;
      const unsigned long long b = __ballot(hit);
      if (hit) W.id[nh + wave_rank(b)] = j[w];
      nh += __popcll(b);
    }
    // sum when the next windows' hits might not fit, and at the end
    if (nh <= kFullHits - 64 * kFullWindows && base + kFullWindows * stride < nitems) continue;
    __builtin_amdgcn_wave_barrier();
    int nsame = 0, nwrap = 0;
    for (int h0 = 0; h0 < nh; h0 += 64) {
      const bool in = h0 + lane < nh;
      const unsigned jj = (unsigned)(in ? W.id[h0 + lane] : i);
      const unsigned pj = hb.single_primary ? jj : (unsigned)bv.mol_pidx_start[jj];
      int2 rec = make_int2((int)jj * hb.uni_len, hb.uni_len | hb.uni_param << kHitParam);
      if (hb.uni_len == 0) {
        const MolMeta m = hb.meta[jj];
        rec = make_int2(m.start, m.len | m.param << kHitParam);
      }
      int kx, ky, kz;
      const double dx = wrap_k(hb.px[pj] - p0x, L0, kx);
      const double dy = wrap_k(hb.py[pj] - p0y, L1, ky);
      const double dz = wrap_k(hb.pz[pj] - p0z, L2, kz);
      const bool wr = fabs(dx) > limx || fabs(dy) > limy || fabs(dz) > limz;
      rec.y |= (int)(((unsigned)kx >> 29 | ((unsigned)ky >> 29) << 3 |
                      ((unsigned)kz >> 29) << 6)
                     << kHitImage);
      const unsigned long long same = __ballot(in && !wr), wrap = __ballot(in && wr);
      if (in) W.hit[wr ? kFullHits - 1 - nwrap - wave_rank(wrap) : nsame + wave_rank(same)] = rec;
      nsame += __popcll(same);
      nwrap += __popcll(wrap);
    }
    __builtin_amdgcn_wave_barrier();
    if (nwrap > 0) e += full_pairs<MIXED, true>(hb, W, P, na, nlj, nwrap, np);
    if (nsame > 0) e += full_pairs<MIXED, false>(hb, W, P, na, nlj, nsame, np);
    nh = 0;
    __builtin_amdgcn_wave_barrier();
  }
  pairs = np;
  return e;
}

// Waves that share one molecule's candidates: a box of few molecules would
// leave most of the chip without a wave, and its waves with long scans.  us
// with 1, 2 and 4: 512 bicyclic 28.0 19.0 17.1, 700 water 13.9 10.6 9.3, 1,500
// water 17.8 14.0 14.6, 1,733 bicyclic 35.1 30.8 35.0, 3,000 water 21.4 23.4
// 26.5.
inline int full_split(int n_mol) { return n_mol > 2048 ? 1 : (n_mol > 1024 ? 2 : 4); }

// Blocks of a full-energy pass over n_mol molecules, 4 waves each.
__host__ __device__ inline int full_blocks(int n_mol, int split) {
  return (n_mol * split + 3) / 4;
}

// A 256-lane work-group's share of a box's full energy, blockIdx.x below
// full_blocks: its sum into partial[blockIdx.x] and, when pairs is given, the
// real site pairs it summed into pairs[blockIdx.x].
struct FullShared {
  WaveEval ws[4];
  SiteParam64 p64[kParamCap];
  double sum[4], np[4];
};

template <bool MIXED>
__device__ __forceinline__ void full_energy_block(const BoxView& bv, int split, double* partial,
                                                  double* pairs, FullShared& sh) {
  if ((int)blockIdx.x >= full_blocks(bv.n_mol, split)) return;  // the whole block
  for (int k = threadIdx.x; k < bv.n_param; k += 256) sh.p64[k] = bv.p64[k];
  const HotBox hb = hot_box(bv);
  __syncthreads();
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int at = (int)blockIdx.x * 4 + w;
  const int i = split == 4 ? at >> 2 : (split == 2 ? at >> 1 : at);
  unsigned np = 0;
  double e = 0.0;
  if (i < hb.n_mol)
    e = wave_molecule_energy<MIXED>(bv, hb, sh.ws[w], i, at - i * split, split, sh.p64, np);
  e = wave_sum_f64(e);
  if (wlane() == 0) {
    sh.sum[w] = e;
    sh.np[w] = (double)np;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = (sh.sum[0] + sh.sum[1]) + (sh.sum[2] + sh.sum[3]);
    if (pairs) pairs[blockIdx.x] = (sh.np[0] + sh.np[1]) + (sh.np[2] + sh.np[3]);
  }
}

// The lane's share of a fixed-order sum of n partials by the NT lanes of a
// block: eight loads in flight.
template <int NT>
__device__ __forceinline__ double full_sum(const double* a, int n) {
  double s = 0.0;
  for (int b = threadIdx.x; b < n; b += 8 * NT) {
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = b + k * NT < n ? a[b + k * NT] : 0.0;
#pragma unroll
    for (int k = 0; k < 8; k++) s += v[k];
  }
  return s;
}

}  // namespace mcgpu
