// Cell-list construction on the device (the build's correct counterpart of
// NLCCalcs::createNLC / getCell, NLCStep.cpp:125-180,245-253).  Molecules
// are binned by their first primary site into fixed-capacity slots; the
// slots of every cell are then put in molecule order, so the candidate order
// (and the summation order) does not depend on atomic arrival order.
#pragma once

#include <climits>

#include "device_common.h"
#include "wave.h"

namespace mcgpu {

__device__ __forceinline__ int cells_total(const CellGrid& g) {
  return g.n[0] * g.n[1] * g.n[2];
}

// Molecule m into the cell of its first primary (mirror entry
// mol_pidx_start[m]); a full cell marks the lists incomplete.
__device__ __forceinline__ void cells_assign_one(const BoxView& bv, int m) {
  const CellGrid& g = bv.cells;
  const int p = bv.mol_pidx_start[m];
  const int c = cell_index(g, cell_coord(bv.px[p], g.inv_w[0], g.n[0]),
                           cell_coord(bv.py[p], g.inv_w[1], g.n[1]),
                           cell_coord(bv.pz[p], g.inv_w[2], g.n[2]));
  const int slot = atomicAdd(&g.count[c], 1);
  g.mol_cell[m] = c;
  if (slot < g.cap) {
    g.slots[c * g.cap + slot] = m;
  } else {
    atomicOr(g.overflow, 1);
  }
}

// One wave orders cell c's slots by molecule id: each lane takes one entry
// and its rank is the number of smaller ids in the cell (ids are distinct),
// counted against the entries read across lanes.  Cells of more than 64
// entries are ordered by one lane (insertion sort).
__device__ __forceinline__ void cells_sort_wave(const CellGrid& g, int c) {
  const int lane = wlane();
  int n = g.count[c];
  n = n < g.cap ? n : g.cap;
  int32_t* s = g.slots + (size_t)c * g.cap;
  if (n <= 64) {
    const int v = lane < n ? s[lane] : INT_MAX;
    int rank = 0;
    for (int k = 0; k < n; k++) rank += readlane_i32(v, k) < v ? 1 : 0;
    if (lane < n) {
      s[rank] = v;
      g.mol_slot[v] = rank;
    }
    return;
  }
  if (lane == 0) {
    for (int i = 1; i < n; i++) {
      const int v = s[i];
      int k = i - 1;
      while (k >= 0 && s[k] > v) {
        s[k + 1] = s[k];
        k--;
      }
      s[k + 1] = v;
    }
    for (int i = 0; i < n; i++) g.mol_slot[s[i]] = i;
  }
}

// The whole build by one work-group of 16 waves, for boxes it suits
// (cells_build_fits), without three launches, device-wide atomics and their
// wait: a stable counting sort by cell.  A wave takes consecutive molecules
// and numbers them within each cell, 64 at a time, over counters of its own; a
// prefix over the waves' counters then gives every molecule its slot.  The
// lists are those of assign and sort above.  Bound by memory latency (a
// dependent first access costs about a microsecond), so all positions load
// together.  refresh: the primary mirror entries [0, refresh) are read from the
// sites first.  flag (host-visible memory, optional) receives the overflow
// flag.
// us for a call that rebuilds the lists of a box, before (three kernels, and a
// copy of the flag to wait for in between) and after: 1,733 molecules 41.8 and
// 12.5, 4,096 46.1 and 15.7, 8,192 47.2 and 25.0 (8,300, three kernels, 29.2 now
// that the flag comes without a wait).  (The molecules of a batch linked per cell, and
// the links walked for the rank, took up to 11,000 cycles a batch: consecutive
// molecules lie in few cells.)
constexpr int kBuildWaves = 16;
constexpr int kBuildBatches = 8;  // batches of 64 a wave takes
constexpr int kBuildCells = 2048;
constexpr int kBuildMol = kBuildWaves * kBuildBatches * 64;

inline bool cells_build_fits(int n_mol, int ncell) {
  return n_mol <= kBuildMol && ncell <= kBuildCells;
}

struct CellBuild {
  uint16_t count[kBuildCells][kBuildWaves];
  int32_t over;
};

__device__ __forceinline__ void cells_build_block(const BoxView& bv, int refresh,
                                                  int32_t* flag, CellBuild& sh) {
  constexpr int NT = 64 * kBuildWaves;
  const CellGrid& g = bv.cells;
  const int ncell = cells_total(g), n = bv.n_mol, t = threadIdx.x, lane = wlane();
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  uint32_t* words = (uint32_t*)&sh.count[0][0];
  for (int k = t; k < ncell * kBuildWaves / 2; k += NT) words[k] = 0;
  if (t == 0) sh.over = 0;
  // with one primary per molecule, each lane refreshes its own molecules'
  const bool own = refresh > 0 && bv.single_primary;
  if (!own)
    for (int k = t; k < refresh; k += NT) {
      const int s = bv.pidx[k];
      bv.px[k] = bv.x[s];
      bv.py[k] = bv.y[s];
      bv.pz[k] = bv.z[s];
    }
  __syncthreads();
  // batches of each wave, and its first molecule
  const int nb = (n + NT - 1) / NT;
  const int m0 = w * nb * 64 + lane;
  int cell[kBuildBatches], at[kBuildBatches];
  double x[kBuildBatches], y[kBuildBatches], z[kBuildBatches];
#pragma unroll
  for (int b = 0; b < kBuildBatches; b++) {
    if (b >= nb) continue;  // block-uniform
    const int m = m0 + b * 64 < n ? m0 + b * 64 : n - 1;
    if (!own)
      at[b] = bv.single_primary ? m : bv.mol_pidx_start[m];
    else
      at[b] = bv.uni_len > 0 ? m * bv.uni_len + bv.uni_p0 : bv.pidx[m];
  }
#pragma unroll
  for (int b = 0; b < kBuildBatches; b++) {
    if (b >= nb) continue;
    x[b] = own ? bv.x[at[b]] : bv.px[at[b]];
    y[b] = own ? bv.y[at[b]] : bv.py[at[b]];
    z[b] = own ? bv.z[at[b]] : bv.pz[at[b]];
  }
#pragma unroll
  for (int b = 0; b < kBuildBatches; b++) {
    if (b >= nb) continue;
    const int m = m0 + b * 64;
    const int c = cell_index(g, cell_coord(x[b], g.inv_w[0], g.n[0]),
                             cell_coord(y[b], g.inv_w[1], g.n[1]),
                             cell_coord(z[b], g.inv_w[2], g.n[2]));
    if (own && m < n) {
      bv.px[m] = x[b];
      bv.py[m] = y[b];
      bv.pz[m] = z[b];
    }
    // the batch's members of one cell after another
    unsigned long long todo = __ballot(m < n);
    int rank = 0, members = 0;
    while (todo) {  // wave-uniform
      const int c0 = readlane_i32(c, __builtin_ctzll(todo));
      const unsigned long long same = __ballot(c == c0) & todo;
      if (c == c0) {
        rank = wave_rank(same);
        members = __popcll(same);
      }
      todo &= ~same;
    }
    cell[b] = c;
    at[b] = 0;
    if (m < n) {
      uint16_t* k = &sh.count[c][w];
      const int before = *k;
      at[b] = before + rank;
      __builtin_amdgcn_wave_barrier();  // every lane has read
      if (rank == 0) *k = (uint16_t)(before + members);
    }
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  for (int c = t; c < ncell; c += NT) {
    int sum = 0;
#pragma unroll
    for (int k = 0; k < kBuildWaves; k++) {
      const int v = sh.count[c][k];
      sh.count[c][k] = (uint16_t)sum;
      sum += v;
    }
    g.count[c] = sum;
    if (sum > g.cap) sh.over = 1;
  }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < kBuildBatches; b++) {
    const int m = m0 + b * 64;
    if (b >= nb || m >= n) continue;
    const int c = cell[b], slot = sh.count[c][w] + at[b];
    g.mol_cell[m] = c;
    if (slot < g.cap) {
      g.slots[c * g.cap + slot] = m;
      g.mol_slot[m] = slot;
    }
  }
  if (t == 0) {
    g.overflow[0] = sh.over;
    if (flag) *flag = sh.over;
  }
}

}  // namespace mcgpu
