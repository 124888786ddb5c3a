// Batched boxes: hundreds of independent boxes advanced by one persistent
// launch.  One work-group owns one box for the whole launch and runs the
// reference's step loop (Simulation.cpp:219-264) on the device: its own
// glibc-TYPE_3 RNG stream (MathLibrary.cpp:27-33), the rigid trial move
// (SimulationStep.cpp:520-566), old+new energy in one pass, the Metropolis
// test (SimulationStep.cpp:794-803), commit or nothing (rollback is free:
// proposals never touch the box).  No grid-wide synchronisation: boxes are
// independent, so a launch is as long as its slowest box.
//
// Box memory is carved from one HBM arena (admission by footprint).  NPT
// volume moves run on a stream of their own beside a launch, decided on the
// device by a short sequence of multi-box kernels around the full-energy
// pass (see queue_volume_moves).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstring>
#include <map>
#include <new>
#include <string>
#include <vector>

#include "box_internal.h"
#include "cells.h"
#include "eval.h"
#include "fastmath.h"
#include "fullenergy.h"
#include "mcgpu_host.h"
#include "wave.h"

namespace mcgpu {

// Per-box control/state, written by the kernel, mirrored to the host after
// every launch.
struct BoxCtl {
  int64_t steps_done;
  int64_t accepted;
  int64_t steps_target;
  int64_t next_stop;  // the kernel stops this box when steps_done reaches it
  int64_t work_cand;   // candidate molecules examined (sum over moves)
  int64_t work_sites;  // sites of in-range molecules loaded
  int64_t work_self;   // sites of the moving molecule (old + proposed)
  int64_t vol_moves;   // NPT volume moves tried / accepted
  int64_t vol_acc;
  int64_t fallbacks;   // moves of a cell-list box that scanned every molecule
  double energy;
  double start_energy;
  double L[3];         // current edges
  double lrc;          // current tail correction (scaled with 1/V)
  // the volume move in flight
  double v_old, v_new, u_accept;
  double L_old[3];
  int32_t status;  // kRunning / kDone / kVolumePending
  int32_t fault;   // MCGPU_FAULT_* that stopped the box (0 = none)
};
constexpr int32_t kRunning = 0, kDone = 1, kVolumePending = 2;

struct BatchBox {
  BoxView bv;
  Rng31* rng;
  int32_t* tr_mol;
  double* tr_de;
  int8_t* tr_acc;
  double* partial;  // the full-energy pass's sums, one per block
  double* bx;       // [n_site] x3: coordinates before an NPT rescale
  double* by;
  double* bz;
  mcgpu_volume_record* tr_vol;  // [tr_vol_cap] NPT volume moves (record_trace)
  double max_t;
  double max_r;
  int32_t precision;
  int32_t record;
  // NPT: pressure (kcal/mol/A^3), half-width of the volume step (A^3),
  // moves between volume moves; cell geometry inputs (cutoff, primary
  // spread, the cells the allocation holds; 0 = no cell lists)
  double pressure;
  double dv;
  double cutoff;
  double spread;
  int32_t vol_interval;
  int32_t ncell_cap;
  int64_t tr_vol_cap;
  // NPT cell boxes: the other set of cell-list arrays and its mode.  A
  // volume move builds the new geometry's lists in it and swaps it in; an
  // undone move swaps the untouched lists back.
  CellGrid cells_alt;
  int32_t mode_alt;
  int32_t pad_alt;
};

// One box of a batched full-energy / rescale / cell pass.
struct VolItem {
  int32_t slot;
  int32_t undo;  // rejected volume move: restore the coordinates
  double f;      // edge scale factor of the rescale
};

// ------------------------------------------------------------- kernel

// Work-group sizes: kGroupWaves waves evaluate, and one more, the side wave,
// draws and builds the next move meanwhile.  (The sizes are named by their
// evaluating lanes, 256, 512 and 1,024; the largest group has 15 waves and the
// side wave.)
constexpr int kGroups = 3;
constexpr int kGroupNT[kGroups] = {256, 512, 1024};
constexpr int kGroupWaves[kGroups] = {4, 8, 15};
constexpr int group_threads(int g) { return (kGroupWaves[g] + 1) * 64; }

// Work-groups of each size that a CU holds at once.  All use 120-128 registers
// a lane, four waves a SIMD, and a group of five waves puts two of them on one
// SIMD: two such groups fit, not the three that the occupancy query counts by
// their 15 waves (groups of 320 lanes that wait 0.5 ms: 512 end after 0.5 ms,
// 513-768 after 1.0, whatever their LDS).  The larger ones fill the LDS.
constexpr int kGroupResident[kGroups] = {2, 1, 1};
// XCDs take a launch's work-groups in turn, whether or not they have room.
constexpr int kXcdUnits = 32;

// Molecules whose primaries a work-group keeps in LDS, and hits it holds: what
// is left beside the other tables of the CU's 160 KiB for the larger ones.  The
// smallest stays below a third of it (beyond, the compiler takes the registers
// of three waves a SIMD, and one group fits).
constexpr int kGroupPrim[kGroups] = {864, 4864, 4864};
constexpr int kGroupHits[kGroups] = {1024, 1536, 1536};

// A stretch of the generator's stream, 64 positions as a ring: position i in
// entry i mod 64, what each of its uses would need.
struct DrawRing {
  double q[kRing];             // r / RAND_MAX (MathLibrary.cpp:31-33)
  double sn[kRing], cs[kRing]; // sin and cos of the rotation angle it stands for
  double limit[kRing];         // as the Metropolis uniform: accepted when dE <= limit
};

// LDS state of one work-group's box for a launch.  ev.rec[cur] is the move
// being evaluated; the other two records take the next move, for the case
// that the current one takes no uniform draw (record cur + 1 mod 3) and that
// it takes one (cur + 2 mod 3).
// What a launch counts (wave 2 keeps it: in LDS, as the scalar registers are
// short and spill).
struct Books {
  double energy;
  int64_t steps, cand, sites, self;
  int32_t acc, fallbacks;
};

template <int G>
struct BatchShared {
  EvalShared<kGroupWaves[G], kGroupPrim[G], 3, kGroupHits[G]> ev;
  DrawRing ring;
  int8_t site_at[kMaxSites];  // uniform boxes: record entry of each site (-1: none)
  int32_t stop;   // the launch's time is up before the next move
  int32_t go;     // the current move runs (else the box stops this launch)
  int32_t cur;
  int32_t used;   // the move before the current one took its uniform draw
  int32_t ovf;    // the cell lists are incomplete
  Books books;
};

// The side wave: the next 31 positions of the stream, from `head` on, into the
// ring; w is the window before them and becomes the one after.  Each position
// gets all its uses, whichever it will have: that costs one pass of sine,
// cosine and logarithm per 31 positions (about 3.6 moves), not per move.
// FMA contraction is off so the doubles match the reference's; the two
// divisions by constants are the correctly rounded quotients, from the
// rounded reciprocal and one residual step (Markstein).
//
// The Metropolis test exp(-dE / kT) >= u (SimulationStep.cpp:794-803) is kept
// as dE <= -kT ln u, which also holds for every dE < 0 (u <= 1); u = 0 accepts
// any dE.
__device__ __forceinline__ void draw_ahead(const BatchBox& B, DrawRing& ring, int& w, int head) {
#pragma clang fp contract(off)
  w = stream_next31(w);
  auto divide = [](double a, double b, double rb) {
    const double q = a * rb;
    return fma(fma(-q, b, a), rb, q);
  };
  const double q = divide((double)(int)((unsigned)w >> 1), 2147483647.0, 1.0 / 2147483647.0);
  const double a = -B.max_r, b = B.max_r;
  const double angle = (b - a) * q + a;
  double sn, cs;
  sincos_fp64(divide(angle * 3.14159265358979, 180.0, 1.0 / 180.0), sn, cs);
  const double limit = -B.bv.kT * log(q);
  const int at = (head + wlane()) & 63;
  if (wlane() < 31) {
    ring.q[at] = q;
    ring.sn[at] = sn;
    ring.cs[at] = cs;
    ring.limit[at] = limit;
  }
}

// The record of the calling lane's half for the next move.
template <class BS>
__device__ __forceinline__ MoveRecord* next_record(BS& S, int cur) {
  const int at = cur + 1 + (wlane() >> 5);
  return &S.ev.rec[at >= 3 ? at - 3 : at];
}

// One wave: the two candidates for the next move, lanes 32 v .. 32 v + 31
// building the move whose draws start at stream position pos + v into
// ev.rec[(cur + 1 + v) mod 3] (Simulation.cpp:219-264 draw order: molecule,
// vertex, dX, dY, dZ, rX, rY, rZ; SimulationStep.cpp:520-566).
//
// Lane k < len of a half holds site k; the pivot is loaded by every lane
// beside its own site.  Every site except the pivot is rotated about the pivot
// by the X, Y, Z Euler angles and all are translated (SimulationStep.cpp:
// 387-422, 545-565).  FMA contraction is off so the doubles match the
// reference's.
template <class BS>
__device__ __forceinline__ void build_moves(BS& S, const BatchBox& B, const BoxView& bv,
                                            const HotBox& hb, int cur, int pos) {
#pragma clang fp contract(off)
  const DrawRing& ring = S.ring;
  const int lane = wlane();
  const int k = lane & 31;
  const int d0 = pos + (lane >> 5);  // position of the first draw
  MoveRecord* m = next_record(S, cur);
  const int n = hb.n_mol;
  const double qm = ring.q[d0 & 63], qv = ring.q[(d0 + 1) & 63];
  int mol = (int)(((double)n - 0.0) * qm + 0.0);
  mol = mol >= n ? n - 1 : mol;  // rand() == RAND_MAX
  // the molecule's record
  int start, len, param, pf, pstart, npri;
  int fault = 0;
  if (hb.uni_len > 0) {
    len = hb.uni_len;
    start = mol * len;
    param = hb.uni_param;
    pf = hb.uni_p0;
    pstart = mol;
    npri = 1;
  } else {
    const MolMeta mm = hb.meta[(unsigned)mol];
    start = mm.start;
    len = mm.len;
    param = mm.param;
    pf = mm.p0;
    pstart = mm.pstart;
    npri = hb.single_primary ? 1 : bv.mol_pidx_count[mol];
    if (len < 1 || len > kMaxSites) {
      fault = MCGPU_FAULT_MOLLEN;
      len = len < 1 ? 1 : kMaxSites;
    }
    npri = npri < 1 ? 1 : (npri > kMaxSites ? kMaxSites : npri);
  }
  int vtx = (int)(((double)len - 0.0) * qv + 0.0);
  vtx = vtx >= len ? len - 1 : vtx;
  const unsigned site = (unsigned)(start + (k < len ? k : 0));
  const unsigned pivot = (unsigned)(start + vtx);
  const double xo = hb.x[site], yo = hb.y[site], zo = hb.z[site];
  const double pvx = hb.x[pivot], pvy = hb.y[pivot], pvz = hb.z[pivot];
  int pof = pf;
  if (npri > 1 && k < npri) pof = bv.pidx[pstart + k] - start;
  const double a = -B.max_t, b = B.max_t;
  const double tx = (b - a) * ring.q[(d0 + 2) & 63] + a;
  const double ty = (b - a) * ring.q[(d0 + 3) & 63] + a;
  const double tz = (b - a) * ring.q[(d0 + 4) & 63] + a;
  const double c0 = ring.cs[(d0 + 5) & 63], s0 = ring.sn[(d0 + 5) & 63];
  const double c1 = ring.cs[(d0 + 6) & 63], s1 = ring.sn[(d0 + 6) & 63];
  const double c2 = ring.cs[(d0 + 7) & 63], s2 = ring.sn[(d0 + 7) & 63];
  if (k < npri) m->pofs[k] = pof;
  if (k == 0) {
    m->mol = mol;
    m->start = start;
    m->len = len;
    m->pstart = pstart;
    m->npri = npri;
    m->param = param;
    m->pf = pf;
    m->fault = fault;
  }
  double X = xo, Y = yo, Z = zo;
  if (k != vtx) {
    X += -pvx;
    Y += -pvy;
    Z += -pvz;
    double u = Y, w = Z;  // rotateX
    Y = u * c0 + w * s0;
    Z = w * c0 - u * s0;
    u = Z;
    w = X;  // rotateY
    Z = u * c1 + w * s1;
    X = w * c1 - u * s1;
    u = X;
    w = Y;  // rotateZ
    X = u * c2 + w * s2;
    Y = w * c2 - u * s2;
    X += pvx;
    Y += pvy;
    Z += pvz;
  }
  if (k < len) {
    m->ox[k] = xo;
    m->oy[k] = yo;
    m->oz[k] = zo;
    m->nx[k] = X + tx;
    m->ny[k] = Y + ty;
    m->nz[k] = Z + tz;
  }
}

// The candidates completed: wrapped by their first primary (SimulationStep.cpp:
// 710-729), staged, and their neighbour sources prepared.
template <class BS>
__device__ __forceinline__ void finish_moves(BS& S, const BoxView& bv, const HotBox& hb,
                                             int cur, bool cc) {
  auto& sh = S.ev;
  const int k = wlane() & 31;
  MoveRecord* m = next_record(S, cur);
  const int len = hb.uni_len > 0 ? hb.uni_len : m->len;
  const int pf = hb.uni_len > 0 ? hb.uni_p0 : m->pf;
  const int kk = k < len ? k : 0;
  const double xo = m->ox[kk], yo = m->oy[kk], zo = m->oz[kk];
  double X = m->nx[kk], Y = m->ny[kk], Z = m->nz[kk];
  const double qx = m->nx[pf], qy = m->ny[pf], qz = m->nz[pf];
  const int at = hb.uni_len > 0 ? S.site_at[k] : stage_sites(sh, m, len, m->param);
  const double sx = qx < 0 ? hb.L0 : (qx > hb.L0 ? -hb.L0 : 0.0);
  const double sy = qy < 0 ? hb.L1 : (qy > hb.L1 ? -hb.L1 : 0.0);
  const double sz = qz < 0 ? hb.L2 : (qz > hb.L2 ? -hb.L2 : 0.0);
  // (only a shift by L changes a bit: x + 0.0 would turn -0.0 into 0.0)
  X = sx != 0.0 ? X + sx : X;
  Y = sy != 0.0 ? Y + sy : Y;
  Z = sz != 0.0 ? Z + sz : Z;
  stage_move(hb, m, at, len, pf, xo, yo, zo, X, Y, Z);
  const int src = hb.mode == MCGPU_NB_CELL && S.ovf == 0 ? MCGPU_NB_CELL : MCGPU_NB_BRUTE;
  prepare_source(bv, sh, m, src, 0, true, cc);
}

// One wave: the sites of move m committed, and its primaries in the mirror (and
// in LDS, when the launch keeps them there).
template <class BS>
__device__ __forceinline__ void commit_sites(BS& S, const HotBox& hb, const MoveRecord& m,
                                             bool prim) {
  const int lane = wlane();
  if (lane < m.len) {
    const unsigned s = (unsigned)(m.start + lane);
    hb.x[s] = m.nx[lane];
    hb.y[s] = m.ny[lane];
    hb.z[s] = m.nz[lane];
  }
  if (hb.single_primary) {
    if (lane == 0) {
      const int mol = m.mol;
      const double x = m.pn[0], y = m.pn[1], z = m.pn[2];
      hb.px[(unsigned)mol] = x;
      hb.py[(unsigned)mol] = y;
      hb.pz[(unsigned)mol] = z;
      if (prim) {
        S.ev.px[mol] = x;
        S.ev.py[mol] = y;
        S.ev.pz[mol] = z;
      }
    }
  } else if (lane < m.npri) {
    const int o = m.pofs[lane];
    const unsigned k = (unsigned)(m.pstart + lane);
    hb.px[k] = m.nx[o];
    hb.py[k] = m.ny[o];
    hb.pz[k] = m.nz[o];
  }
}

// One wave: the cell lists after move m.  Returns whether they changed.  The
// cell of the first primary changes for a few per cent of moves; the old cell
// is the one its current position maps to (cells are assigned from the same
// positions), checked against the list before it is used.
template <class BS>
__device__ __forceinline__ bool commit_cells(BS& S, const BoxView& bv, const HotBox& hb,
                                             const MoveRecord& m, bool cc) {
  const int lane = wlane();
  if (hb.mode != MCGPU_NB_CELL || S.ovf) return false;
  const bool cross = lane < 3 && m.co[lane] != m.cn[lane];
  if (!__ballot(cross)) return false;
  const CellGrid& g = bv.cells;
  if (lane == 0) {
    const int co = cell_index(g, m.co[0], m.co[1], m.co[2]);
    const int cn = cell_index(g, m.cn[0], m.cn[1], m.cn[2]);
    if (g.mol_cell[m.mol] == co) {
      const bool placed = cell_move(g, m.mol, co, cn);
      if (cc) {  // the LDS occupancies follow the lists
        S.ev.ccount[co] -= 1;
        if (placed) S.ev.ccount[cn] += 1;
      }
      if (!placed) S.ovf = 1;
    } else {
      g.overflow[0] = 1;  // lists disagree with positions: scan everything
      S.ovf = 1;
    }
  }
  return true;
}

// The side wave of the batch kernel: the generator's stream, and the next
// move's record, built while the other waves evaluate.  While they scan, it
// moves the next molecule (its stream positions are in the ring); while they
// sum, it completes the record, refills the ring when the move after it would
// run dry, and looks at the clock.  (The waves of a work-group run two loops
// with the same barriers, so that neither holds the other's registers.)
template <class BS>
__device__ __forceinline__ void side_loop(BS& S, const BatchBox& B, const BoxView& bv,
                                          const HotBox& hb, bool cc, long long budget,
                                          long long t_start) {
  const int lane = wlane();
  // it shares its SIMD with evaluating waves, which wait for it at the
  // barriers: its instructions go first
  __builtin_amdgcn_s_setprio(3);
  // the generator's stream, from position 0, and the first move
  Rng31* rs = B.rng;
  const int rng_f = __builtin_amdgcn_readfirstlane(rs->f);
  int w = lane < 31 ? rs->s[(rng_f + lane) % 31] : 0;
  StreamAt at;
  draw_ahead(B, S.ring, w, 0);
  at.head = 31;
  if (hb.uni_len > 0) {  // the same sites in every move's record
    for (int r = 0; r < 3; r++) {
      const int entry = stage_sites(S.ev, &S.ev.rec[r], hb.uni_len, hb.uni_param);
      if (lane < 32) S.site_at[lane] = (int8_t)entry;
    }
  }
  build_moves(S, B, bv, hb, 0, 0);
  finish_moves(S, bv, hb, 0, cc);
  __syncthreads();
  for (int s = 0;; s++) {
    __syncthreads();
    const int cur = __builtin_amdgcn_readfirstlane(S.cur);
    const int go = __builtin_amdgcn_readfirstlane(S.go);
    const int used = __builtin_amdgcn_readfirstlane(S.used);
    const MoveHead h = load_head(S.ev.rec[cur]);
    if (s > 0) stream_advance(at, 8 + used);
    if (!go || h.fault) break;
    build_moves(S, B, bv, hb, cur, at.pos + 8);
    eval_barriers(S.ev, h, [&]() {
      finish_moves(S, bv, hb, cur, cc);
      if (stream_low(at)) {
        draw_ahead(B, S.ring, w, at.head);
        at.head += 31;
      }
      if (budget > 0) {
        const bool up = (wall_clock64() - t_start) >= budget;
        if (lane == 0) S.stop = up;
      }
    });
  }
  // the words before the next draw, in the generator's order (the ring is at
  // most 57 positions ahead)
  for (int back = at.head - at.pos; back > 0; back -= 28)
    w = stream_back(w, back < 28 ? back : 28);
  const int f = stream_front(at, rng_f);
  if (lane < 31) rs->s[(f + lane) % 31] = w;
  if (lane == 0) {
    rs->f = f;
    rs->r = (f + 28) % 31;
  }
}

// The evaluating waves of the batch kernel, over up to `sweeps` moves of the
// box with control block c (written back by wave 2, which keeps the books).
template <class BS>
__device__ __forceinline__ void eval_loop(BS& S, const BatchBox& B, const BoxView& bv,
                                          const HotBox& hb, BoxCtl& c, bool prim, bool cc,
                                          int sweeps) {
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  const int lane = wlane();
  const bool mixed = B.precision == MCGPU_MIXED;
  // moves this launch may make, and those made before it
  const int64_t room = c.next_stop - c.steps_done;
  int n_move = (int)(room < sweeps ? (room < 0 ? 0 : room) : sweeps);
  pin_scalar(n_move);
  if (wave == 2 && lane == 0) S.books = Books{c.energy, c.steps_done, 0, 0, 0, 0, 0};
  int hits = 0, cur = 0;
  int pos = 0;  // ring entry of the current move's first draw
  int s = 0;
  __syncthreads();
  for (;; s++) {
    // Move s - 1 decided, three waves each for itself: wave 0 picks move s and
    // keeps the cell lists, wave 1 commits the sites, wave 2 keeps the books.
    if (wave < 3) {
      const MoveRecord& m = S.ev.rec[cur];
      double de = 0.0;
      bool acc = false;
      int used = 0;
      if (s > 0) {
        double eo, en;
        const double limit = S.ring.limit[(pos + 8) & (kRing - 1)];
        eval_totals(S.ev, eo, en);
        de = en - eo;
        acc = __builtin_amdgcn_readfirstlane(de <= limit ? 1 : 0);
        used = __builtin_amdgcn_readfirstlane(de < 0 ? 0 : 1);
      }
      if (wave == 0) {
        const int next = cur + 1 + used >= 3 ? cur + used - 2 : cur + 1 + used;
        const bool go = s < n_move && !S.stop;
        if (acc) {
          // built from the state before the commit?
          bool again = __builtin_amdgcn_readfirstlane(S.ev.rec[next].mol == m.mol ? 1 : 0);
          again |= commit_cells(S, bv, hb, m, cc);
          if (go && again) {
            commit_sites(S, hb, m, prim);  // (as wave 1 does)
            __threadfence_block();
            build_moves(S, B, bv, hb, cur, pos + 8);
            finish_moves(S, bv, hb, cur, cc);
          }
        }
        if (lane == 0) {
          S.cur = next;
          S.used = used;
          S.go = go;
        }
      } else if (wave == 1) {
        if (acc) commit_sites(S, hb, m, prim);
      } else if (s > 0) {
        const int sites = hb.uni_len > 0
                              ? hits * hb.uni_len
                              : (int)wave_sum_u32(lane < S.ev.kNW ? S.ev.redc[lane] : 0u);
        if (lane == 0) {
          Books k = S.books;
          if (B.record) {
            B.tr_mol[k.steps] = m.mol;
            B.tr_de[k.steps] = de;
            B.tr_acc[k.steps] = (int8_t)acc;
          }
          k.steps++;
          k.energy = acc ? k.energy + de : k.energy;
          k.acc += acc ? 1 : 0;
          // (every source of a batched move lists the moving molecule itself)
          k.cand += m.ncand - 1;
          k.self += 2 * m.len;
          k.sites += sites;
          // a cell-list box whose move scanned every molecule
          if (hb.mode == MCGPU_NB_CELL) k.fallbacks += m.src != MCGPU_NB_CELL ? 1 : 0;
          S.books = k;
        }
      }
    }
    __syncthreads();
    cur = __builtin_amdgcn_readfirstlane(S.cur);
    const int go = __builtin_amdgcn_readfirstlane(S.go);
    const int used = __builtin_amdgcn_readfirstlane(S.used);
    const MoveHead h = load_head(S.ev.rec[cur]);
    if (s > 0) pos = (pos + 8 + used) & (kRing - 1);
    if (!go || h.fault) break;
    hits = eval_core<true>(bv, hb, S.ev, S.ev.rec[cur], h, 0, mixed, prim);
  }
  if (wave == 2 && lane == 0) {
    const int fault = S.go ? S.ev.rec[cur].fault : 0;
    c.steps_done = S.books.steps;
    c.accepted += S.books.acc;
    c.work_cand += S.books.cand;
    c.work_sites += S.books.sites;
    c.work_self += S.books.self;
    c.fallbacks += S.books.fallbacks;
    c.energy = S.books.energy;
    if (fault) c.fault = fault;
    if (c.steps_done >= c.steps_target || c.fault)
      c.status = kDone;
    else if (c.steps_done >= c.next_stop)
      c.status = kVolumePending;
  }
}

// The persistent launch: work-group g owns box active[1 + g] and runs up to
// `sweeps` trial moves on it, stopping early at the box's step target, at a
// pending NPT volume move, or when `budget` wall-clock ticks have passed
// since the work-group started (0 = no time limit).  The LATE instance runs
// the boxes of a tick whose NPT volume move comes first (the volume pass
// queued just before it on its stream, beside the rest of the tick): their
// budget counts from *t0, the wall clock stamped on that stream as the tick
// began, so they stop with the rest of the tick.
//
// A move is a chain of latencies, not of throughput, so as little as possible
// stands between one evaluation and the next: adding up the waves' sums, the
// decision, the commit, and picking the next move's record.  That record is ready:
// while the others scanned and summed, the side wave built the next move (for
// both cases, the current one taking its uniform draw or not) from a ring of
// draws whose sines, cosines and Metropolis logarithms it takes 31 positions at
// a time, and listed its cells.  Wave 0 builds it again only when the committed
// move was of the same molecule or changed the cell lists.
//
// Small boxes stay bound by that chain (256 water: 7,800 cycles a move, four
// barriers, the scan's and the pair sums' loads); 16-site molecules by the
// vector ALUs of the box's one compute unit (23,000 pair evaluations a move at
// about 25 instructions each).  us a move, one box alone, best size, with wave
// 0 drawing, rotating, listing and deciding in turn and the hits' sites staged
// through LDS -> now: water of 256 7.1 -> 3.29 and of 4,096 with cells 9.2 ->
// 4.6, mixture of 3,000 with cells 14.5 -> 6.5, bicyclic of 4,000 with cells
// 14.1 -> 7.7 (MIXED 13.9 -> 7.5).
template <int G, bool LATE>
__global__ __launch_bounds__(group_threads(G), G == 1 ? 3 : 4) void k_batch(
    const BatchBox* __restrict__ table, BoxCtl* ctl, const int32_t* active, int sweeps,
    long long budget, const long long* t0) {
  constexpr int NT = group_threads(G);
  constexpr int NW = kGroupWaves[G];
  __shared__ BatchShared<G> S;
  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  // active = [count, slot 0, slot 1, ...]; the grid is rounded up
  if ((int)blockIdx.x >= __builtin_amdgcn_readfirstlane(active[0])) return;
  const int slot = __builtin_amdgcn_readfirstlane(active[1 + blockIdx.x]);
  long long t_start = LATE ? *t0 : wall_clock64();
  pin_scalar(t_start);
  // the descriptor is read in place (scalar loads from a table this launch
  // does not write)
  const BatchBox& B = table[slot];
  const BoxView& bv = B.bv;
  const HotBox hb = hot_box(bv);
  load_params(bv, S.ev, NT);
  // the cell occupancies into LDS, when the grid fits: only this launch's
  // commits change them until it ends
  const bool cell_box = bv.mode == MCGPU_NB_CELL;
  const int ncell = cell_box ? bv.cells.n[0] * bv.cells.n[1] * bv.cells.n[2] : 0;
  const bool cc = cell_box && ncell <= S.ev.kCellLds;
  if (cc)
    for (int c = t; c < ncell; c += NT) S.ev.ccount[c] = bv.cells.count[c];
  // and the primaries, when they fit
  const bool prim = bv.single_primary && bv.n_mol <= kGroupPrim[G];
  if (prim)
    for (int j = t; j < bv.n_mol; j += NT) {
      S.ev.px[j] = bv.px[j];
      S.ev.py[j] = bv.py[j];
      S.ev.pz[j] = bv.pz[j];
    }
  if (t == 0) {
    S.ovf = cell_box ? bv.cells.overflow[0] : 0;
    S.stop = 0;
    S.used = 0;
    S.cur = 0;
  }
  __syncthreads();
  if (wave == NW)
    side_loop(S, B, bv, hb, cc, budget, t_start);
  else
    eval_loop(S, B, bv, hb, ctl[slot], prim, cc, sweeps);
}

// What an admission sends to the device, packed in pinned host memory: the
// descriptor, the control block and the generator, each padded to 16 bytes,
// then the slot's arrays (or a piece of them) as they lie in the arena.  Copied by
// the blocks of one launch.  160 admissions of 128-4,096 molecules: 24 ms with 15
// pageable copies and three small ones each and a wait for them (and so for the
// former box's set-up), 8.6 ms this way.
struct AdmitHead {
  alignas(16) BatchBox box;
  alignas(16) BoxCtl ctl;
  alignas(16) Rng31 rng;
};

constexpr size_t kAdmitHead = (sizeof(AdmitHead) + 255) & ~size_t(255);

__global__ __launch_bounds__(256) void k_admit(const AdmitHead* from, BatchBox* box, BoxCtl* ctl,
                                               Rng31* rng, char* arrays, size_t bytes) {
  auto words = [](void* to, const void* src, int n) {  // n bytes, a multiple of 4
    for (int k = threadIdx.x; k < n / 4; k += 256) ((int32_t*)to)[k] = ((const int32_t*)src)[k];
  };
  if (blockIdx.x == 0) {
    words(box, &from->box, sizeof(BatchBox));
    words(ctl, &from->ctl, sizeof(BoxCtl));
    words(rng, &from->rng, sizeof(Rng31));
  }
  const char* src = (const char*)from + kAdmitHead;
  const size_t step = (size_t)gridDim.x * 256 * 16;
  for (size_t at = (blockIdx.x * 256 + threadIdx.x) * 16; at < bytes; at += step)
    *(double2*)(arrays + at) = *(const double2*)(src + at);
}
static_assert(sizeof(BatchBox) % 4 == 0 && sizeof(BoxCtl) % 4 == 0 && sizeof(Rng31) % 4 == 0,
              "copied in words");

// ---------------------------------------- batched NPT passes (many boxes)
//
// One launch covers every box of a list (blockIdx.y = list entry), so the
// volume moves of all boxes due in a tick cost a handful of launches.

// Cell geometry of a box for its current edges (the host's cell_geometry):
// cells of width >= rc + 2 spread, cell mode while the grid fits the
// allocation, else the all-molecule scan.
__device__ void set_geometry_dev(BatchBox& B) {
  BoxView& v = B.bv;
  if (B.ncell_cap == 0) {
    v.mode = MCGPU_NB_BRUTE;
    return;
  }
  const double w = B.cutoff + 2.0 * B.spread + 1e-9;
  int n[3];
  for (int d = 0; d < 3; d++) {
    n[d] = (int)floor(v.L[d] / w);
    n[d] = n[d] < 1 ? 1 : n[d];
  }
  if (n[0] * n[1] * n[2] > B.ncell_cap) {
    v.mode = MCGPU_NB_BRUTE;
    return;
  }
  for (int d = 0; d < 3; d++) {
    v.cells.n[d] = n[d];
    v.cells.inv_w[d] = n[d] / v.L[d];
  }
  v.mode = MCGPU_NB_CELL;
}

// The wall clock into *t0: the start of a tick for the boxes that move after
// their volume move.
__global__ void k_stamp_clock(long long* t0) { *t0 = wall_clock64(); }

// NPT volume move, first half, one thread per listed box (semantics: see
// queue_volume_moves): u1 and u2 drawn from the box's own generator, the
// new edges and cell geometry set, the scale factor handed to the rescale.
// V' is the product of the new edges, as acceptVolumeMove reads it
// (SimulationStep.cpp:476-481); a proposal <= 0 keeps the box (f = 1) and
// is rejected by the decision.
__global__ void k_vol_begin(BatchBox* table, BoxCtl* ctl, VolItem* items, int k) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= k) return;
  const int s = items[i].slot;
  BatchBox& B = table[s];
  BoxCtl& c = ctl[s];
  Rng31 g = *B.rng;
  const double u1 = random_real(rng31_next(g), 0.0, 1.0);
  c.u_accept = random_real(rng31_next(g), 0.0, 1.0);
  *B.rng = g;
  BoxView& v = B.bv;
  for (int d = 0; d < 3; d++) c.L_old[d] = v.L[d];
  c.v_old = v.L[0] * v.L[1] * v.L[2];
  const double v_prop = c.v_old + B.dv * (2.0 * u1 - 1.0);
  const double f = v_prop > 0.0 ? cbrt(v_prop / c.v_old) : 1.0;
  items[i].f = f;
  items[i].undo = 0;
  for (int d = 0; d < 3; d++) v.L[d] = c.L_old[d] * f;
  c.v_new = v_prop > 0.0 ? v.L[0] * v.L[1] * v.L[2] : v_prop;
  // the new geometry's cell lists go to the other set of arrays; the
  // current lists stay as they are for an undo
  const CellGrid cur = v.cells;
  v.cells = B.cells_alt;
  B.cells_alt = cur;
  B.mode_alt = v.mode;
  set_geometry_dev(B);
}

// Second half, after the full energy at the new volume (out[2 i + 1]):
// the acceptance test, the running energy and LRC on acceptance, the old
// edges and geometry (and the undo flag for the coordinates) on rejection,
// and the box's next volume stop.  e_pairs: the pair energy at the new
// volume.
__device__ void vol_decide(BatchBox& B, BoxCtl& c, VolItem& item, double e_pairs) {
#pragma clang fp contract(off)
  const bool valid = c.v_new > 0.0;
  const double lrc_new = valid ? c.lrc * c.v_old / c.v_new : c.lrc;
  const double e_new = valid ? e_pairs + lrc_new : c.energy;
  bool accept = false;
  if (valid) {
    // SimCalcs::acceptVolumeMove (SimulationStep.cpp:476-488)
    const double de = e_new - c.energy;
    double prob = B.bv.n_mol * (log(c.v_new) - log(c.v_old));
    prob -= (de + B.pressure * (c.v_new - c.v_old)) / B.bv.kT;
    prob = exp_fp64(prob);
    accept = prob >= c.u_accept;
  }
  if (B.tr_vol && c.vol_moves < B.tr_vol_cap) {
    mcgpu_volume_record r;
    r.step = c.steps_done;
    r.v_old = c.v_old;
    r.v_new = c.v_new;
    r.e_old = c.energy;
    r.e_new = e_new;
    r.u = c.u_accept;
    r.accepted = accept ? 1 : 0;
    r.reserved = 0;
    B.tr_vol[c.vol_moves] = r;
  }
  c.vol_moves++;
  if (accept) {
    c.vol_acc++;
    c.energy = e_new;
    c.lrc = lrc_new;
    for (int d = 0; d < 3; d++) c.L[d] = B.bv.L[d];
  } else {
    // the old edges, and the cell lists and mode from before the move
    for (int d = 0; d < 3; d++) B.bv.L[d] = c.L_old[d];
    const CellGrid cur = B.bv.cells;
    B.bv.cells = B.cells_alt;
    B.cells_alt = cur;
    B.bv.mode = B.mode_alt;
    item.undo = 1;
  }
  c.next_stop = c.steps_target < c.steps_done + B.vol_interval ? c.steps_target
                                                               : c.steps_done + B.vol_interval;
  c.status = c.steps_done >= c.steps_target ? kDone : kRunning;
}

// The full-energy pass over one box (admissions).
template <bool MIXED>
__global__ __launch_bounds__(256, 4) void k_energy_waves(const BatchBox* box, int split) {
  __shared__ FullShared sh;
  full_energy_block<MIXED>(box->bv, split, box->partial, nullptr, sh);
}

// Start energy of a newly added box: the fixed-order sum of its partials plus
// the offset (the LRC), or, for a box that continues from a resume record,
// that record's running energy.
__global__ __launch_bounds__(256) void k_start_energy(const BatchBox* box, BoxCtl* c, int split,
                                                      double offset, int resumed,
                                                      double energy) {
  __shared__ double red[4];
  const double s =
      block_sum<256>(full_sum<256>(box->partial, full_blocks(box->bv.n_mol, split)), red);
  if (threadIdx.x == 0) {
    c->energy = resumed ? energy : s + offset;
    c->start_energy = c->energy;
  }
}

// Entry blockIdx.x of a volume pass: the fixed-order sum of its
// partials at the new volume (as k_start_energy sums them),
// then the decision.
__global__ __launch_bounds__(256) void k_vol_settle(BatchBox* table, BoxCtl* ctl,
                                                    VolItem* items) {
  __shared__ double red[4];
  VolItem& item = items[blockIdx.x];
  BatchBox& B = table[item.slot];
  const double s = block_sum<256>(full_sum<256>(B.partial, full_blocks(B.bv.n_mol, 1)), red);
  if (threadIdx.x == 0) vol_decide(B, ctl[item.slot], item, s);
}

// Both precisions in one launch (a volume pass lists boxes of either): each
// block takes its entry's.
__global__ __launch_bounds__(256, 4) void k_energy_waves_any(const BatchBox* table,
                                                          const VolItem* items) {
  __shared__ FullShared sh;
  const BatchBox& B = table[items[blockIdx.y].slot];
  if (B.precision == MCGPU_MIXED)
    full_energy_block<true>(B.bv, 1, B.partial, nullptr, sh);
  else
    full_energy_block<false>(B.bv, 1, B.partial, nullptr, sh);
}

// Clears entry y's cell occupancies for its current geometry (block x's
// 256 cells), when the box is in cell mode.
__device__ __forceinline__ void clear_cells_block(const BoxView& bv) {
  if (bv.mode != MCGPU_NB_CELL) return;
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c < cells_total(bv.cells)) bv.cells.count[c] = 0;
  if (c == 0) bv.cells.overflow[0] = 0;
}

// NPT rescale of entry y: molecule m is translated so its first primary
// moves from p to f p (internal geometry untouched); its sites are backed up
// first and its primary mirror entries refreshed.  The entry's cell
// occupancies are cleared for the new geometry on the way (block x clears
// cells [256 x, 256 x + 256)).  A uniform box's block takes whole molecules
// (256 / len of them), one lane per site, so its loads and stores are
// contiguous: the first primaries' shifts go through LDS before any site is
// written.  Other boxes take one molecule per lane.
__global__ __launch_bounds__(256) void k_scale_multi(const BatchBox* table,
                                                     const VolItem* items) {
  __shared__ double shift[3][256];
  const VolItem it = items[blockIdx.y];
  const BatchBox& B = table[it.slot];
  const BoxView& bv = B.bv;
  clear_cells_block(bv);
  const double f = it.f;
  const int t = threadIdx.x;
  const int len = bv.uni_len;
  if (len > 0 && bv.single_primary) {
    const int per = 256 / len;  // molecules per block
    const int m0 = blockIdx.x * per;
    if (m0 >= bv.n_mol) return;
    const int nm = bv.n_mol - m0 < per ? bv.n_mol - m0 : per;
    if (t < nm) {
      const int m = m0 + t;
      const int p = m * len + bv.uni_p0;
      const double px = bv.x[p], py = bv.y[p], pz = bv.z[p];
      const double sx = px * f - px;
      const double sy = py * f - py;
      const double sz = pz * f - pz;
      shift[0][t] = sx;
      shift[1][t] = sy;
      shift[2][t] = sz;
      bv.px[m] = px + sx;
      bv.py[m] = py + sy;
      bv.pz[m] = pz + sz;
    }
    __syncthreads();
    if (t < nm * len) {
      const int s = m0 * len + t;
      const int k = t / len;
      const double x = bv.x[s], y = bv.y[s], z = bv.z[s];
      B.bx[s] = x;
      B.by[s] = y;
      B.bz[s] = z;
      bv.x[s] = x + shift[0][k];
      bv.y[s] = y + shift[1][k];
      bv.z[s] = z + shift[2][k];
    }
    return;
  }
  const int m = blockIdx.x * 256 + t;
  if (m >= bv.n_mol) return;
  const int p = bv.pidx[bv.mol_pidx_start[m]];
  const double sx = bv.x[p] * f - bv.x[p];
  const double sy = bv.y[p] * f - bv.y[p];
  const double sz = bv.z[p] * f - bv.z[p];
  const int s0 = bv.mol_start[m], s1 = s0 + bv.mol_len[m];
  for (int s = s0; s < s1; s++) {
    B.bx[s] = bv.x[s];
    B.by[s] = bv.y[s];
    B.bz[s] = bv.z[s];
    bv.x[s] += sx;
    bv.y[s] += sy;
    bv.z[s] += sz;
  }
  const int ps = bv.mol_pidx_start[m], pe = ps + bv.mol_pidx_count[m];
  for (int k = ps; k < pe; k++) {
    const int q = bv.pidx[k];
    bv.px[k] = bv.x[q];
    bv.py[k] = bv.y[q];
    bv.pz[k] = bv.z[q];
  }
}

// A rejected rescale undone: molecule m's sites and primaries restored (the
// decision put the cell lists from before the move back).  Blocks map to
// molecules as in k_scale_multi.
__global__ __launch_bounds__(256) void k_restore_multi(const BatchBox* table,
                                                       const VolItem* items) {
  if (!items[blockIdx.y].undo) return;
  const BatchBox& B = table[items[blockIdx.y].slot];
  const BoxView& bv = B.bv;
  const int t = threadIdx.x;
  const int len = bv.uni_len;
  if (len > 0 && bv.single_primary) {
    const int per = 256 / len;
    const int m0 = blockIdx.x * per;
    if (m0 >= bv.n_mol) return;
    const int nm = bv.n_mol - m0 < per ? bv.n_mol - m0 : per;
    if (t < nm * len) {
      const int s = m0 * len + t;
      bv.x[s] = B.bx[s];
      bv.y[s] = B.by[s];
      bv.z[s] = B.bz[s];
    }
    if (t < nm) {
      const int m = m0 + t;
      const int p = m * len + bv.uni_p0;
      bv.px[m] = B.bx[p];
      bv.py[m] = B.by[p];
      bv.pz[m] = B.bz[p];
    }
    return;
  }
  const int m = blockIdx.x * 256 + t;
  if (m >= bv.n_mol) return;
  const int s0 = bv.mol_start[m], s1 = s0 + bv.mol_len[m];
  for (int s = s0; s < s1; s++) {
    bv.x[s] = B.bx[s];
    bv.y[s] = B.by[s];
    bv.z[s] = B.bz[s];
  }
  const int ps = bv.mol_pidx_start[m], pe = ps + bv.mol_pidx_count[m];
  for (int k = ps; k < pe; k++) {
    const int q = bv.pidx[k];
    bv.px[k] = bv.x[q];
    bv.py[k] = bv.y[q];
    bv.pz[k] = bv.z[q];
  }
}

// Cell lists of every listed box in cell mode, built for the new geometry
// after k_scale_multi cleared the occupancies: by one work-group each, or
// assign, order for boxes beyond it (see cells.h).
__global__ __launch_bounds__(1024) void k_cells_build_multi(const BatchBox* table,
                                                            const VolItem* items) {
  __shared__ CellBuild sh;
  const BoxView& bv = table[items[blockIdx.x].slot].bv;
  if (bv.mode == MCGPU_NB_CELL) cells_build_block(bv, 0, nullptr, sh);
}

__global__ __launch_bounds__(256) void k_cells_assign_multi(const BatchBox* table,
                                                            const VolItem* items) {
  const BoxView& bv = table[items[blockIdx.y].slot].bv;
  if (bv.mode != MCGPU_NB_CELL) return;
  const int m = blockIdx.x * 256 + threadIdx.x;
  if (m < bv.n_mol) cells_assign_one(bv, m);
}

__global__ __launch_bounds__(256) void k_cells_sort_multi(const BatchBox* table,
                                                          const VolItem* items) {
  const BoxView& bv = table[items[blockIdx.y].slot].bv;
  if (bv.mode != MCGPU_NB_CELL) return;
  const int c = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  if (c < cells_total(bv.cells)) cells_sort_wave(bv.cells, c);
}

// ------------------------------------------------------------ host side

// Best-fit allocator over one device chunk (offsets, 256-byte aligned).
class Arena {
 public:
  ~Arena() {
    if (base_) (void)hipFree(base_);
  }
  int init(size_t bytes) {
    bytes = (bytes + 255) & ~size_t(255);
    MCGPU_HIP_TRY(hipMalloc(&base_, bytes));
    cap_ = bytes;
    free_[0] = bytes;
    return MCGPU_OK;
  }
  bool alloc(size_t bytes, size_t* off) {
    bytes = (bytes + 255) & ~size_t(255);
    auto best = free_.end();
    for (auto it = free_.begin(); it != free_.end(); ++it)
      if (it->second >= bytes && (best == free_.end() || it->second < best->second))
        best = it;
    if (best == free_.end()) return false;
    *off = best->first;
    const size_t rest = best->second - bytes;
    const size_t roff = best->first + bytes;
    free_.erase(best);
    if (rest) free_[roff] = rest;
    live_[*off] = bytes;
    used_ += bytes;
    peak_ = std::max(peak_, used_);
    return true;
  }
  void release(size_t off) {
    auto it = live_.find(off);
    if (it == live_.end()) return;
    size_t size = it->second;
    live_.erase(it);
    used_ -= size;
    auto nx = free_.lower_bound(off);
    if (nx != free_.end() && off + size == nx->first) {
      size += nx->second;
      nx = free_.erase(nx);
    }
    if (nx != free_.begin()) {
      auto pv = std::prev(nx);
      if (pv->first + pv->second == off) {
        pv->second += size;
        return;
      }
    }
    free_[off] = size;
  }
  char* base() const { return (char*)base_; }
  size_t used() const { return used_; }
  size_t peak() const { return peak_; }
  size_t capacity() const { return cap_; }

 private:
  void* base_ = nullptr;
  size_t cap_ = 0, used_ = 0, peak_ = 0;
  std::map<size_t, size_t> free_, live_;
};

// Offsets of one box's arrays inside its arena block.
struct BoxLayout {
  size_t x, y, z, px, py, pz, ms, ml, mps, mpc, meta, pidx, p64;
  size_t ccount, cslots, mcell, mslot, covf, vstale, vcount, partial, bx, by, bz, trm, trd,
      tra, trv;
  size_t ccount2, cslots2, mcell2, mslot2, covf2;  // NPT cell boxes: second set
  bool alt_cells;
  int64_t trv_cap;
  size_t upload;  // bytes of the arrays an admission uploads
  size_t bytes;
  int ncell, cap;
};

BoxLayout plan_layout(const mcgpu_box_desc& d, const mcgpu_run_params& p,
                      const ParamTable& pt) {
  BoxLayout L{};
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t o = off;
    off += (std::max<size_t>(bytes, 8) + 255) & ~size_t(255);
    return o;
  };
  const size_t ns = d.n_sites, nm = d.n_molecules, np = d.n_primary;
  // the arrays an admission uploads, first
  L.x = take(8 * ns);
  L.y = take(8 * ns);
  L.z = take(8 * ns);
  L.ms = take(4 * nm);
  L.ml = take(4 * nm);
  L.mps = take(4 * nm);
  L.mpc = take(4 * nm);
  L.meta = take(sizeof(MolMeta) * nm);
  L.pidx = take(4 * np);
  L.p64 = take(sizeof(SiteParam64) * pt.p64.size());
  L.covf = take(4);
  L.vstale = take(4);
  L.vcount = take(4);
  L.upload = off;
  L.px = take(8 * np);
  L.py = take(8 * np);
  L.pz = take(8 * np);
  L.ncell = 0;
  if (p.neighbor == MCGPU_NEIGHBOR_CELL) {
    // room for the grid of a box up to 26% larger in volume (NPT)
    double Lg[3];
    for (int k = 0; k < 3; k++) Lg[k] = d.box[k] * 1.08;
    int n[3], cn[3];
    double iw[3];
    cell_geometry(Lg, d.cutoff, pt.spread, n, iw);
    L.ncell = n[0] * n[1] * n[2];
    cell_geometry(d.box, d.cutoff, pt.spread, cn, iw);
    const int nc_now = cn[0] * cn[1] * cn[2];
    L.cap = ((int)std::ceil(3.0 * nm / nc_now) + 16 + 3) & ~3;
    L.ccount = take(4 * (size_t)L.ncell);
    L.cslots = take(4 * (size_t)L.ncell * L.cap);
  }
  L.mcell = take(4 * nm);
  L.mslot = take(4 * nm);
  L.alt_cells = L.ncell > 0 && p.ensemble == MCGPU_NPT;
  if (L.alt_cells) {
    L.ccount2 = take(4 * (size_t)L.ncell);
    L.cslots2 = take(4 * (size_t)L.ncell * L.cap);
    L.mcell2 = take(4 * nm);
    L.mslot2 = take(4 * nm);
    L.covf2 = take(4);
  }
  L.partial = take(8 * nm);
  if (p.ensemble == MCGPU_NPT) {
    L.bx = take(8 * ns);
    L.by = take(8 * ns);
    L.bz = take(8 * ns);
  }
  if (p.record_trace) {
    L.trm = take(4 * (size_t)p.steps);
    L.trd = take(8 * (size_t)p.steps);
    L.tra = take((size_t)p.steps);
    if (p.ensemble == MCGPU_NPT) {
      L.trv_cap = p.steps / p.volume_interval + 1;
      L.trv = take(sizeof(mcgpu_volume_record) * (size_t)L.trv_cap);
    }
  }
  L.bytes = off;
  return L;
}

// Per-move work of a box, estimated with the molecule density inside the
// cutoff sphere: candidates scanned, and steps of the pair sums.
struct MoveWork {
  double cand, pairs;
};

MoveWork move_work(const mcgpu_box_desc& d, int neighbor, int max_len) {
  const double V = d.box[0] * d.box[1] * d.box[2];
  const double rho = d.n_molecules / V;
  const double rc = d.cutoff;
  const double hits = std::min<double>(d.n_molecules - 1, 4.18879 * rc * rc * rc * rho);
  double cand = d.n_molecules;
  if (neighbor == MCGPU_NEIGHBOR_CELL) cand = std::min<double>(cand, 27.0 * rc * rc * rc * rho);
  int aw = 1;
  while (aw < max_len) aw *= 2;
  return {cand, hits * max_len * aw / 2};
}

// Work-group size of a box that has a compute unit to itself.  us a move with
// 4, 8 and 15 evaluating waves (FP64; MIXED, where it differs, after a slash):
//   all-pairs scan: water of 128 molecules 2.92 2.99 3.24, 400: 3.46 3.22 3.33,
//     600: 4.12 3.50 3.26, 1,000: 4.54 3.52 4.26, 1,900: 6.68 4.63 4.30, 2,000:
//     6.68 4.66 5.28, 4,096: 10.9 6.96 7.29; mixture of 500 5.86 4.77 4.88, 700:
//     6.33 5.10 4.78, 1,000: 6.78 5.14 5.91, 1,500: 8.42 6.38 6.08, 2,000: 9.63
//     6.96 7.26; 16-site bicyclic of 512 9.02 7.17 7.44 / 10.3 7.68 7.35, 950:
//     10.2 7.51 7.54 / 11.6 8.06 7.44, 2,000: 12.4 8.77 9.62 / 13.9 9.31 9.54
//   cells: water of 128 3.12 3.21 3.45, 400: 3.78 3.39 3.47, 600: 4.54 3.81 3.47,
//     1,000: 7.29 5.18 4.55, 4,096: 6.12 4.74 4.52; mixture of 300 6.71 5.27
//     5.20, 1,000: 9.82 7.19 6.27, 3,000: 10.4 7.57 6.43; bicyclic of 400 11.8
//     9.30 8.60 / 13.2 9.76 8.50, 4,000: 9.80 7.60 7.60 / 11.1 8.07 7.47
// Waves cost barriers and adding up, so a light move takes four.  An all-pairs
// scan costs its passes: of 512 candidates with 8 waves, two to a round (1.15 us
// a round, 0.8 for a last one of one pass), of 960 with 15, each a round (1.0
// us), which gain 0.1 us otherwise and more where the pair sums are FP32 (their
// conversions and branch keep a lane longer at a pair).  A scan of cells is a
// chain of two loads, so a candidate counts twice, and needs all the waves
// beyond a pass; in a box of one pass long pair sums do too.
int choose_group(const MoveWork& w, int neighbor, int n_mol, bool mixed) {
  const bool cells = neighbor == MCGPU_NEIGHBOR_CELL;
  if (cells && (n_mol > 512 || w.pairs > 2000.0)) return 2;
  if ((cells ? 2.0 : 1.0) * w.cand + w.pairs <= 1000.0) return 0;
  const int p8 = (n_mol + 511) / 512, p15 = (n_mol + 959) / 960;
  const double t8 = 1.15 * (p8 / 2) + 0.8 * (p8 % 2);
  const double t15 = 1.0 * p15 - 0.1 - (mixed ? w.pairs * 1e-4 : 0.0);
  return t15 < t8 ? 2 : 1;
}

}  // namespace mcgpu

using namespace mcgpu;

struct BatchSlot {
  bool used = false;
  size_t off = 0;
  BoxLayout lay{};
  mcgpu_run_params params{};
  int32_t n_pidx = 0;
  int32_t group = 0;   // preferred work-group size (estimate or tuner)
  double work = 0.0;   // per-move work (estimate)
  double spread = 0.0; // largest primary-to-first-primary distance
  int fault = 0;
  int64_t tune_key = 0;    // box class for the work-group-size tuner
  int trial = -1;          // group being measured for the class (-1: none)
  int64_t steps_at_launch = 0;
  // counters before this run (a box added from a resume record)
  int64_t base_steps = 0, base_acc = 0, base_vol = 0, base_vacc = 0;
  bool dirty = false;      // the device's control block is newer than h_ctl
  bool late = false;       // runs after its volume move in the tick in flight
};

// One captured tick launch: the persistent kernel of each work-group-size
// group over its active list, side by side; replayed while the grid sizes,
// sweep count and time budget are unchanged.
struct TickGraph {
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  int sweeps = -1;
  uint64_t version = 0;
  int grid[kGroups] = {};
};

// Host side of a batch.  Streams: `stream` carries the ticks and the
// read-back after them; `vstream`, beside each tick, the NPT volume moves of
// the boxes that reached a volume stop in the previous one (decided on the
// device) and then those boxes' own share of the tick (the late graph), which
// the read-back waits for (ev_vdone); `side[]` serve graph capture (the
// work-group-size groups of a tick run side by side); `sstream` admissions
// (their uploads, cells and start energy), which every tick waits for
// (ev_ready).
// Ownership: control blocks and generator states are the device's; the host
// mirrors them from each tick's read-back (merged for the boxes the tick
// ran) and writes a box's only when it sets the box up.
struct mcgpu_batch {
  hipStream_t stream = nullptr;
  hipStream_t side[kGroups - 1] = {};
  hipStream_t sstream = nullptr;
  hipStream_t vstream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr, fork = nullptr;
  hipEvent_t join[kGroups - 1] = {};
  hipEvent_t ev_ready = nullptr;  // set-up work queued so far is done
  hipEvent_t ev_vdone = nullptr;  // the volume branch of the tick is done
  Arena arena;
  int32_t max_boxes = 0;
  int device = 0;  // the device current when the batch was created
  int n_cu = 256;
  std::vector<BatchSlot> slots;
  BatchBox* d_table = nullptr;
  BatchBox* h_table = nullptr;  // pinned mirror (the host's copy)
  BoxCtl* d_ctl = nullptr;
  BoxCtl* h_ctl = nullptr;      // pinned mirror
  BoxCtl* h_ctl_rb = nullptr;   // pinned read-back of a tick
  Rng31* d_rng = nullptr;
  Rng31* h_rng = nullptr;       // pinned mirror
  Rng31* h_rng_rb = nullptr;    // pinned read-back of a tick
  // [2 * kGroups * (max_boxes + 1)]: per group [count, slots...], the
  // main lists then the late ones
  int32_t* d_active = nullptr;
  int32_t* h_active = nullptr;  // pinned
  std::vector<int32_t> next_active;  // the lists of the tick being set up
  std::vector<int> eff_group;        // work-group size of each box this tick
  std::vector<int> order;            // the tick's boxes in launch order
  VolItem* d_items = nullptr;   // [max_boxes] list of a volume pass
  VolItem* h_items = nullptr;   // pinned
  // pinned: admissions on their way in, up to stage_at, and coordinates on
  // their way out behind them; up to stage_used it has been used before
  char* h_stage = nullptr;
  char* d_stage = nullptr;
  size_t stage_at = 0, stage_used = 0;
  int admitted = 0;  // boxes, of which the first kStageFew
  long long* d_t0 = nullptr;    // wall clock at the start of the volume pass
  long long budget_ticks = 0;   // per-launch time limit (wall-clock ticks)
  double clock_khz = 100000.0;
  bool pending = false;         // a tick in flight
  std::vector<int> launched;    // slots of the tick in flight
  std::vector<int> late;        // of which after their volume move
  TickGraph main_graph, late_graph;
  uint64_t version = 1;  // bumped when the time budget changes
  // work-group-size tuner: per box class, moves per full tick at each size
  struct Tune {
    int best = -1;
    double moves[kGroups] = {};
    int samples[kGroups] = {};
    bool trialing = false;
  };
  std::map<int64_t, Tune> tune;
  bool autotune = true;
  // host seconds: waiting for ticks, volume moves, launching ticks
  double t_wait = 0.0, t_volume = 0.0, t_launch = 0.0;
  // timing
  double kernel_ms_sum = 0.0;
  int64_t kernel_launches = 0;
  bool timing_pending = false;
};

namespace {

double host_now() {
  return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch())
      .count();
}

// Pinned memory for admissions and downloads, allocated with the batch: one
// allocation of it costs 0.3-2.7 ms by its size, which a batch's first download
// or a large box's admission would pay.  Larger boxes go through it in pieces.
constexpr size_t kStageBytes = 4 << 20;
// Taking its pages for the first time costs 1.6 us each, 0.6 ms for the
// coordinates of 64,000 sites, which pays for itself over a few boxes: a batch's
// first kStageFew go in pieces of kStagePiece through the same pages, waiting for
// the device in between (a wait of about 15 us).
constexpr size_t kStagePiece = 256 << 10;
constexpr int kStageFew = 4;

int stage_alloc(mcgpu_batch* b) {
  if (hipHostMalloc((void**)&b->h_stage, kStageBytes, hipHostMallocMapped) != hipSuccess ||
      hipHostGetDevicePointer((void**)&b->d_stage, b->h_stage, 0) != hipSuccess) {
    set_error("pinned buffer allocation failed");
    return MCGPU_ERR_NOMEM;
  }
  return MCGPU_OK;
}

// Room for `bytes` (at most all of it) from stage_at on; from the front again
// when it is used up.  Before new pages are taken: kGo takes them, kWait waits
// until the set-up stream is done with the old ones, kLook looks whether it is
// (a look while the stream is busy costs an admission's 20 us).
enum class Stage { kGo, kWait, kLook };

int stage_room(mcgpu_batch* b, size_t bytes, Stage how) {
  const size_t end = b->stage_at + bytes;
  if (end <= b->stage_used || b->stage_at == 0) return MCGPU_OK;
  if (end <= kStageBytes && how != Stage::kWait) {
    if (how == Stage::kGo) return MCGPU_OK;
    if (hipStreamQuery(b->sstream) != hipSuccess) {
      (void)hipGetLastError();  // (not ready is no error to keep)
      return MCGPU_OK;
    }
  } else {
    MCGPU_HIP_TRY(hipStreamSynchronize(b->sstream));
  }
  b->stage_at = 0;
  return MCGPU_OK;
}

// Bytes [at, at + n) of an image that lies in host memory in parts, to or from
// the staging buffer.
struct ImagePart {
  size_t at;
  void* host;
  size_t bytes;
};

template <class Copy>
void for_image(const ImagePart* parts, int count, size_t at, size_t n, Copy copy) {
  for (int k = 0; k < count; k++) {
    const ImagePart& q = parts[k];
    const size_t lo = std::max(q.at, at), hi = std::min(q.at + q.bytes, at + n);
    if (lo < hi) copy(lo - at, (char*)q.host + (lo - q.at), hi - lo);
  }
}

int upload_ctl(mcgpu_batch* b, int s, hipStream_t st) {
  MCGPU_HIP_TRY(hipMemcpyAsync(b->d_ctl + s, b->h_ctl + s, sizeof(BoxCtl),
                               hipMemcpyHostToDevice, st));
  return MCGPU_OK;
}

char* slot_base(mcgpu_batch* b, int s) { return b->arena.base() + b->slots[s].off; }

// Cell geometry of slot s's current box into its descriptor (host copy):
// cell mode when the grid fits the allocation, else the all-molecule scan.
// Returns the cell count (0 without cells).
int slot_set_geometry(mcgpu_batch* b, int s) {
  BatchSlot& S = b->slots[s];
  BoxView& v = b->h_table[s].bv;
  if (S.lay.ncell == 0) {
    v.mode = MCGPU_NB_BRUTE;
    return 0;
  }
  int n[3];
  double iw[3];
  cell_geometry(v.L, b->h_table[s].cutoff, S.spread, n, iw);
  if (n[0] * n[1] * n[2] > S.lay.ncell) {
    v.mode = MCGPU_NB_BRUTE;
    return 0;
  }
  for (int k = 0; k < 3; k++) {
    v.cells.n[k] = n[k];
    v.cells.inv_w[k] = iw[k];
  }
  v.mode = MCGPU_NB_CELL;
  return n[0] * n[1] * n[2];
}

// The batched passes over the first k entries of a device list: per-molecule
// full-energy partials; cell lists for the current geometry (occupancies
// already cleared).
void launch_energy_partials(mcgpu_batch* b, const VolItem* items, int k, int max_mol,
                            hipStream_t st) {
  const dim3 grid((max_mol + 3) / 4, k);  // blocks past a box's molecules exit at once
  hipLaunchKernelGGL(k_energy_waves_any, grid, dim3(256), 0, st, b->d_table, items);
}

int launch_cells_pass(mcgpu_batch* b, const VolItem* items, int k, int max_mol,
                      int max_cells, hipStream_t st) {
  if (max_cells == 0) return MCGPU_OK;
  if (cells_build_fits(max_mol, max_cells)) {
    hipLaunchKernelGGL(k_cells_build_multi, dim3(k), dim3(1024), 0, st, b->d_table, items);
    MCGPU_HIP_TRY(hipGetLastError());
    return MCGPU_OK;
  }
  hipLaunchKernelGGL(k_cells_assign_multi, dim3((max_mol + 255) / 256, k), dim3(256), 0, st,
                     b->d_table, items);
  hipLaunchKernelGGL(k_cells_sort_multi, dim3((max_cells + 3) / 4, k), dim3(256), 0, st,
                     b->d_table, items);
  MCGPU_HIP_TRY(hipGetLastError());
  return MCGPU_OK;
}

// NPT volume moves of the boxes in `pend`, batched and decided on the
// device, queued on `st` at the start of the tick in which those boxes move
// on (beside the tick's other boxes): u1, u2 from each box's generator, the
// rescale (with backup), cells for the new geometry (in the box's second set
// of cell arrays, so that an undo only swaps the old lists back), the full
// energy, the decision, and the undo of rejected moves.  Semantics (the
// build's own; the reference's NPT path, Ensemble.cpp:9-28 /
// SimulationStep.cpp:476-518, always grows the box by 1.1 and never
// recomputes the energy):
//   V' = V + dv (2 u1 - 1), dv = delta V0 (V0 the volume at admission): a
//   fixed-width, symmetric step, so acceptVolumeMove's test is the whole
//   acceptance rule; molecules translated so first primaries scale by
//   f = (V'/V)^(1/3); V' then taken as the product of the new edges;
//   E' = E_pairs(V') + LRC V/V'; dE = E' - E, with E the box's running
//   energy (start energy plus accepted move dE); accept iff
//   exp(N ln(V'/V) - (dE + P (V' - V)) / kT) >= u2 (SimulationStep.cpp:
//   476-488), and then the running energy becomes E' exactly.  A proposal
//   V' <= 0 is rejected.
int queue_volume_moves(mcgpu_batch* b, const std::vector<int>& pend, hipStream_t st) {
  int rc;
  const int K = (int)pend.size();
  for (int k = 0; k < K; k++) b->h_items[k] = VolItem{pend[k], 0, 1.0};
  MCGPU_HIP_TRY(hipMemcpyAsync(b->d_items, b->h_items, sizeof(VolItem) * K,
                               hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_vol_begin, dim3((K + 63) / 64), dim3(64), 0, st, b->d_table, b->d_ctl,
                     b->d_items, K);
  int max_mol = 0, max_cells = 0, scale_blocks = 0;
  for (int s : pend) {
    const BoxView& v = b->h_table[s].bv;
    max_mol = std::max(max_mol, v.n_mol);
    max_cells = std::max(max_cells, b->slots[s].lay.ncell);
    // k_scale_multi and k_restore_multi: whole molecules per block for
    // uniform boxes
    const int per = v.uni_len > 0 && v.single_primary ? 256 / v.uni_len : 256;
    scale_blocks = std::max(scale_blocks, (v.n_mol + per - 1) / per);
  }
  // blocks for the occupancies too (at most the allocated cells)
  const int clear_blocks = (max_cells + 255) / 256;
  const int rescale_grid = std::max(scale_blocks, clear_blocks);
  hipLaunchKernelGGL(k_scale_multi, dim3(rescale_grid, K), dim3(256), 0, st, b->d_table,
                     b->d_items);
  MCGPU_HIP_TRY(hipGetLastError());
  if ((rc = launch_cells_pass(b, b->d_items, K, max_mol, max_cells, st))) return rc;
  launch_energy_partials(b, b->d_items, K, max_mol, st);
  hipLaunchKernelGGL(k_vol_settle, dim3(K), dim3(256), 0, st, b->d_table, b->d_ctl,
                     b->d_items);
  hipLaunchKernelGGL(k_restore_multi, dim3(scale_blocks, K), dim3(256), 0, st, b->d_table,
                     b->d_items);
  MCGPU_HIP_TRY(hipGetLastError());
  return MCGPU_OK;
}

// Work-group-size tuner.  Per box class (neighbour source, pair precision,
// largest molecule, molecule count in quarter-octaves) the first box of the
// class runs one tick at each work-group size; all boxes of a tick get the
// same time budget, so the moves it made in a full tick measure its speed
// at that size.  The fastest size is kept for the class; until then other
// boxes of the class use the density estimate (choose_group).
int64_t tune_key_of(const mcgpu_box_desc& d, const mcgpu_run_params& p, int max_len) {
  const int64_t nb = (int64_t)std::lround(4.0 * std::log2((double)std::max(d.n_molecules, 1)));
  return ((int64_t)p.neighbor * 4 + p.precision) * 1000000 + (int64_t)max_len * 1000 + nb;
}

void tune_sample(mcgpu_batch* b, int s) {
  BatchSlot& S = b->slots[s];
  // a box that took its volume move first ran a shortened tick
  if (S.trial < 0 || S.late) return;
  const BoxCtl& c = b->h_ctl[s];
  const int64_t moved = c.steps_done - S.steps_at_launch;
  // only full ticks measure speed: the box ran until the time budget
  if (c.status != kRunning || moved < 1 || c.steps_done >= c.next_stop) return;
  auto& T = b->tune[S.tune_key];
  T.moves[S.trial] += (double)moved;
  T.samples[S.trial]++;
  int next = -1;
  for (int g = 0; g < kGroups; g++)
    if (T.samples[g] == 0) {
      next = g;
      break;
    }
  if (next >= 0) {
    S.trial = next;
    S.group = next;
    return;
  }
  int best = 0;
  for (int g = 1; g < kGroups; g++)
    if (T.moves[g] / T.samples[g] > T.moves[best] / T.samples[best]) best = g;
  T.best = best;
  T.trialing = false;
  S.trial = -1;
  for (int k = 0; k < b->max_boxes; k++)
    if (b->slots[k].used && b->slots[k].tune_key == S.tune_key) b->slots[k].group = best;
}

// Tick boundary: consumes a finished tick (its read-back merged for the
// boxes it ran, its volume branch included).  Boxes that reached a volume
// stop in it stay at kVolumePending until the next tick takes their volume
// move.  Without a tick in flight it does nothing.
int batch_boundary(mcgpu_batch* b) {
  if (!b->pending) return MCGPU_OK;
  const double t0 = host_now();
  MCGPU_HIP_TRY(hipStreamSynchronize(b->stream));
  b->t_wait += host_now() - t0;
  b->pending = false;
  for (int s : b->launched) {
    b->h_ctl[s] = b->h_ctl_rb[s];
    b->h_rng[s] = b->h_rng_rb[s];
    b->slots[s].dirty = false;
    if (b->budget_ticks > 0) tune_sample(b, s);
    b->slots[s].late = false;
  }
  if (b->timing_pending) {
    float ms = 0.f;
    MCGPU_HIP_TRY(hipEventElapsedTime(&ms, b->ev0, b->ev1));
    b->kernel_ms_sum += ms;
    b->kernel_launches++;
    b->timing_pending = false;
  }
  b->launched.clear();
  b->late.clear();
  return MCGPU_OK;
}

// Whether the tick in flight runs slot s.
bool in_flight(const mcgpu_batch* b, int s) {
  return b->pending && std::find(b->launched.begin(), b->launched.end(), s) != b->launched.end();
}

// Control blocks of slots set up since their last tick, from the device.
int refresh_dirty(mcgpu_batch* b, int only_slot) {
  bool any = false;
  for (int s = 0; s < b->max_boxes; s++)
    if (b->slots[s].used && b->slots[s].dirty && (only_slot < 0 || s == only_slot)) {
      if (!any) MCGPU_HIP_TRY(hipStreamSynchronize(b->sstream));
      any = true;
      MCGPU_HIP_TRY(hipMemcpy(b->h_ctl + s, b->d_ctl + s, sizeof(BoxCtl),
                              hipMemcpyDeviceToHost));
      b->slots[s].dirty = false;
    }
  return MCGPU_OK;
}

// Everything queued is done and every mirror is current.  The mirrors take each
// tick's read-back and hold what a box was set up with, so only boxes set up
// since their last tick have to be read (reading every control block and
// generator on each call took two copies, 40 of a download's 75 us).
int batch_quiesce(mcgpu_batch* b) {
  int rc;
  if ((rc = batch_boundary(b))) return rc;
  if (b->launched.empty()) return refresh_dirty(b, -1);
  // a tick that failed half-way: the device's state for every box
  MCGPU_HIP_TRY(hipStreamSynchronize(b->stream));
  MCGPU_HIP_TRY(hipStreamSynchronize(b->vstream));
  MCGPU_HIP_TRY(hipStreamSynchronize(b->sstream));
  MCGPU_HIP_TRY(hipMemcpy(b->h_ctl, b->d_ctl, sizeof(BoxCtl) * b->max_boxes,
                          hipMemcpyDeviceToHost));
  MCGPU_HIP_TRY(hipMemcpy(b->h_rng, b->d_rng, sizeof(Rng31) * b->max_boxes,
                          hipMemcpyDeviceToHost));
  for (BatchSlot& S : b->slots) S.dirty = false;
  return MCGPU_OK;
}

void free_slot(mcgpu_batch* b, int s) {
  if (!b->slots[s].used) return;
  if (b->slots[s].trial >= 0) {
    auto it = b->tune.find(b->slots[s].tune_key);
    if (it != b->tune.end()) it->second.trialing = false;
  }
  b->arena.release(b->slots[s].off);
  b->slots[s] = BatchSlot();
}

}  // namespace

extern "C" int mcgpu_batch_create(int32_t max_boxes, size_t budget,
                                  mcgpu_batch** out) {
  if (!out || max_boxes < 1) {
    set_error("mcgpu_batch_create: bad argument");
    return MCGPU_ERR_INVALID;
  }
  *out = nullptr;
  int rc = ensure_device();
  if (rc) return rc;
  auto* b = new (std::nothrow) mcgpu_batch();
  if (!b) return MCGPU_ERR_NOMEM;
  b->max_boxes = max_boxes;
  if (hipGetDevice(&b->device) != hipSuccess) b->device = 0;
  b->slots.resize(max_boxes);
  if (budget == 0) {
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) != hipSuccess) fr = size_t(8) << 30;
    budget = std::min(fr / 4, size_t(64) << 30);
  }
  auto fail = [&](int code) {
    mcgpu_batch_destroy(b);
    return code;
  };
  if ((rc = b->arena.init(budget)) || (rc = stage_alloc(b))) return fail(rc);
  {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, b->device) ==
            hipSuccess &&
        cus > 0)
      b->n_cu = cus;
  }
  int dev = 0, khz = 0;
  if (hipGetDevice(&dev) == hipSuccess &&
      hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) == hipSuccess &&
      khz > 0)
    b->clock_khz = khz;
  const size_t M = max_boxes;
  bool ok = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) == hipSuccess &&
            hipStreamCreateWithFlags(&b->sstream, hipStreamNonBlocking) == hipSuccess &&
            hipStreamCreateWithFlags(&b->vstream, hipStreamNonBlocking) == hipSuccess &&
            hipEventCreate(&b->ev0) == hipSuccess && hipEventCreate(&b->ev1) == hipSuccess &&
            hipEventCreateWithFlags(&b->fork, hipEventDisableTiming) == hipSuccess &&
            hipEventCreateWithFlags(&b->ev_ready, hipEventDisableTiming) == hipSuccess &&
            hipEventCreateWithFlags(&b->ev_vdone, hipEventDisableTiming) == hipSuccess;
  for (int g = 0; ok && g < kGroups - 1; g++)
    ok = hipStreamCreateWithFlags(&b->side[g], hipStreamNonBlocking) == hipSuccess &&
         hipEventCreateWithFlags(&b->join[g], hipEventDisableTiming) == hipSuccess;
  ok = ok && hipMalloc(&b->d_table, sizeof(BatchBox) * M) == hipSuccess &&
       hipMalloc(&b->d_ctl, sizeof(BoxCtl) * M) == hipSuccess &&
       hipMalloc(&b->d_rng, sizeof(Rng31) * M) == hipSuccess &&
       hipMalloc(&b->d_active, sizeof(int32_t) * 2 * kGroups * (M + 1)) == hipSuccess &&
       hipMalloc(&b->d_items, sizeof(VolItem) * M) == hipSuccess &&
       hipMalloc(&b->d_t0, sizeof(long long)) == hipSuccess &&
       hipHostMalloc((void**)&b->h_table, sizeof(BatchBox) * M, 0) == hipSuccess &&
       hipHostMalloc((void**)&b->h_ctl, sizeof(BoxCtl) * M, 0) == hipSuccess &&
       hipHostMalloc((void**)&b->h_ctl_rb, sizeof(BoxCtl) * M, 0) == hipSuccess &&
       hipHostMalloc((void**)&b->h_rng, sizeof(Rng31) * M, 0) == hipSuccess &&
       hipHostMalloc((void**)&b->h_rng_rb, sizeof(Rng31) * M, 0) == hipSuccess &&
       hipHostMalloc((void**)&b->h_active, sizeof(int32_t) * 2 * kGroups * (M + 1), 0) ==
           hipSuccess &&
       hipHostMalloc((void**)&b->h_items, sizeof(VolItem) * M, 0) == hipSuccess;
  if (!ok) {
    set_error("mcgpu_batch_create: allocation failed");
    return fail(MCGPU_ERR_NOMEM);
  }
  std::memset(b->h_table, 0, sizeof(BatchBox) * M);
  std::memset(b->h_ctl, 0, sizeof(BoxCtl) * M);
  // empty active lists on both sides: a tick uploads a group's list only
  // when it differs from what the device holds (h_active mirrors d_active)
  std::memset(b->h_active, 0, sizeof(int32_t) * 2 * kGroups * (M + 1));
  if (hipMemset(b->d_active, 0, sizeof(int32_t) * 2 * kGroups * (M + 1)) != hipSuccess) {
    set_error("mcgpu_batch_create: allocation failed");
    return fail(MCGPU_ERR_HIP);
  }
  std::memset(b->h_rng, 0, sizeof(Rng31) * M);
  for (size_t s = 0; s < M; s++) b->h_ctl[s].status = kDone;
  if (hipMemcpy(b->d_ctl, b->h_ctl, sizeof(BoxCtl) * M, hipMemcpyHostToDevice) != hipSuccess) {
    set_error("mcgpu_batch_create: upload failed");
    return fail(MCGPU_ERR_HIP);
  }
  *out = b;
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_destroy(mcgpu_batch* b) {
  if (!b) return MCGPU_OK;
  for (hipStream_t s : {b->stream, b->vstream, b->side[0], b->side[1], b->sstream})
    if (s) (void)hipStreamSynchronize(s);
  for (TickGraph* G : {&b->main_graph, &b->late_graph}) {
    if (G->exec) (void)hipGraphExecDestroy(G->exec);
    if (G->graph) (void)hipGraphDestroy(G->graph);
  }
  for (void* p : {(void*)b->d_table, (void*)b->d_ctl, (void*)b->d_rng, (void*)b->d_active,
                  (void*)b->d_items, (void*)b->d_t0})
    if (p) (void)hipFree(p);
  for (void* p : {(void*)b->h_table, (void*)b->h_ctl, (void*)b->h_ctl_rb, (void*)b->h_rng,
                  (void*)b->h_rng_rb, (void*)b->h_active, (void*)b->h_items, (void*)b->h_stage})
    if (p) (void)hipHostFree(p);
  for (hipEvent_t e : {b->ev0, b->ev1, b->fork, b->ev_ready, b->ev_vdone})
    if (e) (void)hipEventDestroy(e);
  for (hipEvent_t e : b->join)
    if (e) (void)hipEventDestroy(e);
  for (hipStream_t s : {b->stream, b->vstream, b->side[0], b->side[1], b->sstream})
    if (s) (void)hipStreamDestroy(s);
  delete b;
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_bind_thread(mcgpu_batch* b) {
  if (!b) return MCGPU_ERR_INVALID;
  MCGPU_HIP_TRY(hipSetDevice(b->device));
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_set_tick_budget(mcgpu_batch* b, double microseconds) {
  if (!b || microseconds < 0) return MCGPU_ERR_INVALID;
  b->budget_ticks = (long long)(microseconds * b->clock_khz / 1000.0);
  b->version++;
  return MCGPU_OK;
}

extern "C" int mcgpu_box_footprint(const mcgpu_box_desc* d,
                                   const mcgpu_run_params* p, size_t* bytes) {
  if (!d || !p || !bytes) return MCGPU_ERR_INVALID;
  const std::string why = validate_desc(*d);
  if (!why.empty()) {
    set_error("mcgpu_box_footprint: " + why);
    return MCGPU_ERR_INVALID;
  }
  const ParamTable pt = build_param_table(*d);
  *bytes = plan_layout(*d, *p, pt).bytes;
  return MCGPU_OK;
}

// Admission: the box's arrays are uploaded and its cells, start energy and
// control block set up on the set-up stream, beside a tick in flight (a
// tick only touches the boxes it runs); the box joins the next tick.  With
// a resume record r the box continues that record's generator stream,
// running energy, LRC and NPT schedule.
static int batch_add_impl(mcgpu_batch* b, const mcgpu_box_desc* d, const mcgpu_run_params* p,
                          const mcgpu_resume_state* r, int32_t* slot_out) {
  if (!b || !d || !p || !slot_out) return MCGPU_ERR_INVALID;
  if (r && (r->rng_front < 0 || r->rng_front > 30 || r->rng_rear < 0 || r->rng_rear > 30 ||
            (r->rng_front - r->rng_rear + 31) % 31 != 3 || r->steps_done < 0)) {
    set_error("mcgpu_batch_add_resumed: bad resume record");
    return MCGPU_ERR_INVALID;
  }
  const std::string why = validate_desc(*d);
  if (!why.empty()) {
    set_error("mcgpu_batch_add: " + why);
    return MCGPU_ERR_INVALID;
  }
  if ((p->precision != MCGPU_FP64 && p->precision != MCGPU_MIXED) ||
      (p->ensemble != MCGPU_NVT && p->ensemble != MCGPU_NPT) || p->steps < 0 ||
      (p->neighbor != MCGPU_NEIGHBOR_BRUTE && p->neighbor != MCGPU_NEIGHBOR_CELL) ||
      (p->ensemble == MCGPU_NPT && (p->volume_interval < 1 || !(p->max_volume_delta > 0) ||
                                    !(p->max_volume_delta < 0.5)))) {
    set_error("mcgpu_batch_add: bad run parameters");
    return MCGPU_ERR_INVALID;
  }
  int rc;
  int s = -1;
  for (int k = 0; k < b->max_boxes; k++)
    if (!b->slots[k].used) {
      s = k;
      break;
    }
  if (s < 0) {
    set_error("mcgpu_batch_add: no free slot");
    return MCGPU_ERR_NOMEM;
  }
  const ParamTable pt = build_param_table(*d);
  if ((int)pt.p64.size() > kParamCap) {
    set_error("mcgpu_batch_add: more than " + std::to_string(kParamCap) +
              " distinct site-parameter entries");
    return MCGPU_ERR_INVALID;
  }
  const BoxLayout L = plan_layout(*d, *p, pt);
  size_t off = 0;
  if (!b->arena.alloc(L.bytes, &off)) {
    set_error("mcgpu_batch_add: HBM budget exhausted");
    return MCGPU_ERR_NOMEM;
  }
  BatchSlot& S = b->slots[s];
  S = BatchSlot();
  S.used = true;
  S.off = off;
  S.lay = L;
  S.params = *p;
  S.n_pidx = d->n_primary;
  S.spread = pt.spread;
  const MoveWork mw = move_work(*d, p->neighbor, pt.max_len);
  S.group = choose_group(mw, p->neighbor, d->n_molecules, p->precision == MCGPU_MIXED);
  S.work = mw.cand + mw.pairs;
  S.tune_key = tune_key_of(*d, *p, pt.max_len);
  if (b->autotune && b->budget_ticks > 0) {
    auto& T = b->tune[S.tune_key];
    if (T.best >= 0) {
      S.group = T.best;
    } else if (!T.trialing) {  // this box measures the class
      T.trialing = true;
      for (int g = 0; g < kGroups; g++)
        if (T.samples[g] == 0) {
          S.trial = S.group = g;
          break;
        }
    }
  }
  char* base = b->arena.base() + off;
  BatchBox& E = b->h_table[s];
  E = BatchBox{};
  BoxView& v = E.bv;
  v.x = gmem((double*)(base + L.x));
  v.y = gmem((double*)(base + L.y));
  v.z = gmem((double*)(base + L.z));
  v.px = gmem((double*)(base + L.px));
  v.py = gmem((double*)(base + L.py));
  v.pz = gmem((double*)(base + L.pz));
  v.mol_start = gmem((int32_t*)(base + L.ms));
  v.mol_len = gmem((int32_t*)(base + L.ml));
  v.mol_pidx_start = gmem((int32_t*)(base + L.mps));
  v.mol_pidx_count = gmem((int32_t*)(base + L.mpc));
  v.meta = gmem((MolMeta*)(base + L.meta));
  v.single_primary = pt.single_primary;
  v.pidx = gmem((int32_t*)(base + L.pidx));
  v.p64 = gmem((SiteParam64*)(base + L.p64));
  v.n_mol = d->n_molecules;
  v.n_site = d->n_sites;
  v.max_len = pt.max_len;
  v.uni_len = pt.uni_len;
  v.uni_param = pt.uni_param;
  v.uni_p0 = pt.uni_p0;
  v.n_param = (int32_t)pt.p64.size();
  v.mode = MCGPU_NB_BRUTE;
  for (int k = 0; k < 3; k++) v.L[k] = d->box[k];
  v.cutoff2 = d->cutoff * d->cutoff;
  v.reach2 = reach2_of(pt.reach);
  v.kT = d->kT;
  v.cells.count = gmem((int32_t*)(base + L.ccount));
  v.cells.slots = gmem((int32_t*)(base + L.cslots));
  v.cells.mol_cell = gmem((int32_t*)(base + L.mcell));
  v.cells.mol_slot = gmem((int32_t*)(base + L.mslot));
  v.cells.overflow = gmem((int32_t*)(base + L.covf));
  v.cells.cap = L.cap;
  E.cells_alt = v.cells;
  if (L.alt_cells) {
    E.cells_alt.count = gmem((int32_t*)(base + L.ccount2));
    E.cells_alt.slots = gmem((int32_t*)(base + L.cslots2));
    E.cells_alt.mol_cell = gmem((int32_t*)(base + L.mcell2));
    E.cells_alt.mol_slot = gmem((int32_t*)(base + L.mslot2));
    E.cells_alt.overflow = gmem((int32_t*)(base + L.covf2));
  }
  E.mode_alt = MCGPU_NB_BRUTE;
  v.verlet.stale = gmem((int32_t*)(base + L.vstale));
  v.verlet.count = gmem((int32_t*)(base + L.vcount));
  E.rng = b->d_rng + s;
  E.max_t = d->max_translate;
  E.max_r = d->max_rotate;
  E.precision = p->precision;
  E.record = p->record_trace ? 1 : 0;
  E.partial = (double*)(base + L.partial);
  E.bx = (double*)(base + L.bx);
  E.by = (double*)(base + L.by);
  E.bz = (double*)(base + L.bz);
  E.pressure = p->pressure;
  // fixed-width volume step: a symmetric proposal, so the acceptance test
  // needs no Hastings factor
  E.dv = p->max_volume_delta * (d->box[0] * d->box[1] * d->box[2]);
  if (r && r->volume_step > 0) E.dv = r->volume_step;
  E.cutoff = d->cutoff;
  E.spread = pt.spread;
  E.vol_interval = p->volume_interval;
  E.ncell_cap = L.ncell;
  E.tr_mol = (int32_t*)(base + L.trm);
  E.tr_de = (double*)(base + L.trd);
  E.tr_acc = (int8_t*)(base + L.tra);
  E.tr_vol = L.trv_cap > 0 ? (mcgpu_volume_record*)(base + L.trv) : nullptr;
  E.tr_vol_cap = L.trv_cap;
  if (r) {
    for (int k = 0; k < 31; k++) b->h_rng[s].s[k] = r->rng_words[k];
    b->h_rng[s].f = r->rng_front;
    b->h_rng[s].r = r->rng_rear;
    S.base_steps = r->steps_done;
    S.base_acc = r->accepted;
    S.base_vol = r->volume_moves;
    S.base_vacc = r->volume_accepted;
  } else {
    rng31_seed(b->h_rng[s], p->seed);
  }
  BoxCtl& c = b->h_ctl[s];
  c = BoxCtl{};
  for (int k = 0; k < 3; k++) c.L[k] = d->box[k];
  c.lrc = r ? r->lrc : p->energy_offset;
  c.steps_target = p->steps;
  c.next_stop = p->steps;
  if (p->ensemble == MCGPU_NPT) {
    // volume moves after every volume_interval moves since the first start;
    // one due where a previous run stopped comes first
    const int64_t prior = r ? r->steps_done : 0;
    const int64_t due = (r && r->volume_pending) ? 0 : p->volume_interval - prior % p->volume_interval;
    c.next_stop = std::min<int64_t>(p->steps, due);
  }
  c.status = p->steps > 0 ? kRunning : kDone;
  const hipStream_t st = b->sstream;
  const int ncell = p->neighbor == MCGPU_NEIGHBOR_CELL ? slot_set_geometry(b, s) : 0;
  // the sources are the caller's (and this call's) arrays: packed here, and
  // fetched by the device when it gets there
  const size_t ns = d->n_sites, nm = d->n_molecules;
  int32_t zero = 0;
  const ImagePart parts[] = {{L.x, (void*)d->x, 8 * ns},
                             {L.y, (void*)d->y, 8 * ns},
                             {L.z, (void*)d->z, 8 * ns},
                             {L.ms, (void*)d->mol_start, 4 * nm},
                             {L.ml, (void*)d->mol_len, 4 * nm},
                             {L.mps, (void*)d->mol_pidx_start, 4 * nm},
                             {L.mpc, (void*)d->mol_pidx_count, 4 * nm},
                             {L.meta, (void*)pt.meta.data(), sizeof(MolMeta) * nm},
                             {L.pidx, (void*)d->primary_index, 4 * (size_t)d->n_primary},
                             {L.p64, (void*)pt.p64.data(), sizeof(SiteParam64) * pt.p64.size()},
                             {L.covf, &zero, 4},
                             {L.vstale, &zero, 4},
                             {L.vcount, &zero, 4}};
  // (behind a tick in flight the set-up stream may wait for long)
  const bool few = b->admitted < kStageFew && !b->pending;
  b->admitted += b->admitted < kStageFew;
  const size_t piece = (few ? kStagePiece : kStageBytes) - kAdmitHead;
  for (size_t at = 0; at < L.upload;) {
    const size_t n = std::min(L.upload - at, piece);
    const bool wait = few && n >= kStagePiece / 4;  // (few pages cost less)
    if ((rc = stage_room(b, kAdmitHead + n, wait ? Stage::kWait : Stage::kGo))) {
      free_slot(b, s);
      return rc;
    }
    AdmitHead* head = (AdmitHead*)(b->h_stage + b->stage_at);
    head->box = E;
    head->ctl = c;
    head->rng = b->h_rng[s];
    char* arrays = (char*)head + kAdmitHead;
    for_image(parts, (int)std::size(parts), at, n,
              [&](size_t to, const char* from, size_t k) { std::memcpy(arrays + to, from, k); });
    const unsigned blocks = (unsigned)std::min<size_t>((n + 4095) / 4096, 1024);
    hipLaunchKernelGGL(k_admit, dim3(blocks), dim3(256), 0, st,
                       (const AdmitHead*)(b->d_stage + b->stage_at), b->d_table + s, b->d_ctl + s,
                       b->d_rng + s, base + at, n);
    b->stage_at += kAdmitHead + n;
    b->stage_used = std::max(b->stage_used, b->stage_at);
    at += n;
  }
  bool signalled = false;
  rc = hipGetLastError() != hipSuccess ? MCGPU_ERR_HIP
       : ncell > 0 ? launch_cells_build(v, S.n_pidx, nullptr, HostSignal{nullptr, 0},
                                        &signalled, st)
                   : launch_refresh_primary(v, S.n_pidx, st);
  if (rc) {
    set_error("mcgpu_batch_add: upload failed");
    free_slot(b, s);
    return rc;
  }
  // start energy: the full-energy pass over this one box
  const int split = full_split(v.n_mol);
  const dim3 grid(full_blocks(v.n_mol, split));
  if (p->precision == MCGPU_MIXED)
    hipLaunchKernelGGL(k_energy_waves<true>, grid, dim3(256), 0, st,
                       (const BatchBox*)(b->d_table + s), split);
  else
    hipLaunchKernelGGL(k_energy_waves<false>, grid, dim3(256), 0, st,
                       (const BatchBox*)(b->d_table + s), split);
  hipLaunchKernelGGL(k_start_energy, dim3(1), dim3(256), 0, st, (const BatchBox*)(b->d_table + s),
                     b->d_ctl + s, split, p->energy_offset, r ? 1 : 0, r ? r->energy : 0.0);
  MCGPU_HIP_TRY(hipGetLastError());
  S.dirty = true;  // the device now holds the start energy
  *slot_out = s;
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_add(mcgpu_batch* b, const mcgpu_box_desc* d,
                               const mcgpu_run_params* p, int32_t* slot_out) {
  return batch_add_impl(b, d, p, nullptr, slot_out);
}

extern "C" int mcgpu_batch_add_resumed(mcgpu_batch* b, const mcgpu_box_desc* d,
                                       const mcgpu_run_params* p, const mcgpu_resume_state* r,
                                       int32_t* slot_out) {
  if (!r) return MCGPU_ERR_INVALID;
  return batch_add_impl(b, d, p, r, slot_out);
}

extern "C" int mcgpu_batch_get_resume(mcgpu_batch* b, int32_t s, mcgpu_resume_state* out) {
  if (!b || !out || s < 0 || s >= b->max_boxes || !b->slots[s].used) {
    set_error("mcgpu_batch_get_resume: bad slot");
    return MCGPU_ERR_RANGE;
  }
  int rc = batch_quiesce(b);
  if (rc) return rc;
  const BatchSlot& S = b->slots[s];
  const BoxCtl& c = b->h_ctl[s];
  const Rng31& g = b->h_rng[s];
  *out = mcgpu_resume_state{};
  for (int k = 0; k < 31; k++) out->rng_words[k] = g.s[k];
  out->rng_front = g.f;
  out->rng_rear = g.r;
  out->steps_done = S.base_steps + c.steps_done;
  out->accepted = S.base_acc + c.accepted;
  out->volume_moves = S.base_vol + c.vol_moves;
  out->volume_accepted = S.base_vacc + c.vol_acc;
  out->energy = c.energy;
  out->lrc = c.lrc;
  out->ensemble = S.params.ensemble;
  out->volume_interval = S.params.volume_interval;
  out->pressure = S.params.pressure;
  const int vi = S.params.volume_interval;
  if (S.params.ensemble == MCGPU_NPT && vi > 0) {
    out->volume_step = b->h_table[s].dv;
    out->volume_pending = out->steps_done > 0 && out->steps_done % vi == 0 &&
                          out->volume_moves < out->steps_done / vi;
  }
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_remove(mcgpu_batch* b, int32_t s) {
  if (!b || s < 0 || s >= b->max_boxes || !b->slots[s].used) {
    set_error("mcgpu_batch_remove: bad slot");
    return MCGPU_ERR_RANGE;
  }
  // a tick in flight without this box touches neither its control block nor
  // its arena block (its read-back copies the block but merges launched
  // slots only), so only a tick that runs it is waited for
  int rc;
  if (in_flight(b, s) && (rc = batch_boundary(b))) return rc;
  if (b->slots[s].dirty) MCGPU_HIP_TRY(hipStreamSynchronize(b->sstream));
  b->h_ctl[s] = BoxCtl{};
  b->h_ctl[s].status = kDone;
  if ((rc = upload_ctl(b, s, b->sstream))) return rc;
  free_slot(b, s);
  return MCGPU_OK;
}

namespace {

// Replays G on `st` (the late graph on the volume stream, after the volume
// pass), capturing it again when the grids, sweep count or time budget
// changed; e0 and e1 (optional) are recorded around the replay.  Every group
// is launched, with its list's count rounded up to a multiple of 32
// work-groups (32 at least; surplus work-groups exit at once), and a grid is
// kept while it is at most twice what the list needs, so a graph survives
// most admissions, retirements and volume stops: capturing and instantiating
// one takes the host a few hundred microseconds, during which the device
// would idle.
int launch_tick_graph(mcgpu_batch* b, TickGraph& G, bool late, hipStream_t st,
                      const int n[kGroups], int sweeps, hipEvent_t e0, hipEvent_t e1) {
  const int stride = b->max_boxes + 1;
  const int32_t* act = b->d_active + (late ? kGroups * stride : 0);
  int grid[kGroups];
  bool same = G.exec && G.version == b->version && G.sweeps == sweeps;
  for (int g = 0; g < kGroups; g++) {
    const int need = std::min(b->max_boxes, (std::max(n[g], 1) + 31) & ~31);
    const int cur = G.exec ? G.grid[g] : 0;
    grid[g] = cur >= need && cur <= 2 * need ? cur : need;
    same = same && G.grid[g] == grid[g];
  }
  if (!same) {
    if (G.exec) MCGPU_HIP_TRY(hipGraphExecDestroy(G.exec));
    if (G.graph) MCGPU_HIP_TRY(hipGraphDestroy(G.graph));
    G.exec = nullptr;
    G.graph = nullptr;
    using K = void (*)(const BatchBox*, BoxCtl*, const int32_t*, int, long long,
                       const long long*);
    const K kern[2][kGroups] = {
        {k_batch<0, false>, k_batch<1, false>, k_batch<2, false>},
        {k_batch<0, true>, k_batch<1, true>, k_batch<2, true>}};
    // the branch on `st` starts first, the others 10-30 us later: the largest
    // groups lead
    const hipStream_t on[kGroups] = {b->side[1], b->side[0], st};
    MCGPU_HIP_TRY(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    MCGPU_HIP_TRY(hipEventRecord(b->fork, st));
    for (int g = 1; g < kGroups; g++)
      MCGPU_HIP_TRY(hipStreamWaitEvent(b->side[g - 1], b->fork, 0));
    for (int g = kGroups - 1; g >= 0; g--)
      hipLaunchKernelGGL(kern[late][g], dim3(grid[g]), dim3(group_threads(g)), 0, on[g],
                         b->d_table, b->d_ctl, act + g * stride, sweeps, b->budget_ticks,
                         (const long long*)b->d_t0);
    for (int g = 1; g < kGroups; g++) {
      MCGPU_HIP_TRY(hipEventRecord(b->join[g - 1], b->side[g - 1]));
      MCGPU_HIP_TRY(hipStreamWaitEvent(st, b->join[g - 1], 0));
    }
    MCGPU_HIP_TRY(hipStreamEndCapture(st, &G.graph));
    MCGPU_HIP_TRY(hipGraphInstantiate(&G.exec, G.graph, nullptr, nullptr, 0));
    G.version = b->version;
    G.sweeps = sweeps;
    for (int g = 0; g < kGroups; g++) G.grid[g] = grid[g];
  }
  if (e0) MCGPU_HIP_TRY(hipEventRecord(e0, st));
  MCGPU_HIP_TRY(hipGraphLaunch(G.exec, st));
  if (e1) MCGPU_HIP_TRY(hipEventRecord(e1, st));
  return MCGPU_OK;
}

// Uploads the active lists of one side (main or late) that changed.  The
// previous tick, and so its uploads from h_active, has completed (the
// boundary waited for it).
int upload_lists(mcgpu_batch* b, bool late, hipStream_t st) {
  const int stride = b->max_boxes + 1;
  const size_t base = late ? (size_t)kGroups * stride : 0;
  for (int g = 0; g < kGroups; g++) {
    const int32_t* want = &b->next_active[base + g * stride];
    const size_t words = 1 + (size_t)want[0];
    int32_t* h = b->h_active + base + g * stride;
    if (std::memcmp(h, want, sizeof(int32_t) * words) == 0) continue;
    std::memcpy(h, want, sizeof(int32_t) * words);
    MCGPU_HIP_TRY(hipMemcpyAsync(b->d_active + base + g * stride, h, sizeof(int32_t) * words,
                                 hipMemcpyHostToDevice, st));
  }
  return MCGPU_OK;
}

}  // namespace

// One tick: every running box advances up to `sweeps` moves in one graph
// launch; beside it, on the volume stream, the boxes that reached a volume
// stop in the previous tick take their volume move and then advance in the
// late graph until the same deadline.  The previous tick is consumed first;
// with sync the call returns after this tick is consumed too.
extern "C" int mcgpu_batch_run(mcgpu_batch* b, int32_t sweeps, int32_t sync) {
  if (!b || sweeps < 1) return MCGPU_ERR_INVALID;
  int rc = batch_boundary(b);
  if (rc) return rc;
  const int stride = b->max_boxes + 1;
  b->launched.clear();
  b->late.clear();
  for (int s = 0; s < b->max_boxes; s++) {
    const BatchSlot& S = b->slots[s];
    const int32_t st = b->h_ctl[s].status;
    if (!S.used || (st != kRunning && st != kVolumePending)) continue;
    b->launched.push_back(s);
    b->slots[s].steps_at_launch = b->h_ctl[s].steps_done;
    if (st == kVolumePending) {
      b->late.push_back(s);
      b->slots[s].late = true;
    }
  }
  if (b->launched.empty()) return MCGPU_OK;
  // Work-group sizes of this tick: each box's preferred one, unless the
  // boxes need more compute units than some XCD has.  Then every box
  // takes the smallest groups, which share compute units, so that up to 512
  // boxes are resident at once: with larger ones oversubscribed, groups wait for
  // whole units and run in rounds (a tick limited to 5 ms of 220 boxes of the
  // middle size and 100 small ones took 10.2 ms, of 220 and 60 5.1), and groups
  // of two sizes fragment them (us
  // for 2,000 moves of 512 water boxes of 64-4,096 molecules: 18,600 all
  // small, 18,500 with the 256 heaviest at the middle size).  A first round of
  // work-groups takes one unit each and the next starts over with the first
  // unit, so the heaviest boxes lead and their units' second boxes are the
  // lightest (17,900 us; work-groups in slot order 18,600; 17,300 since later
  // changes).  Boxes measured by the tuner keep their size.
  std::vector<int>& eff = b->eff_group;
  eff.assign(b->max_boxes, 0);
  int n[2][kGroups] = {};
  for (int s : b->launched) {
    eff[s] = b->slots[s].group;
    n[b->slots[s].late][eff[s]]++;
  }
  const int xcds = std::max(1, b->n_cu / kXcdUnits);
  int demand = 0;  // units of the XCD that takes the most of each launch
  for (int g = 0; g < kGroups; g++)
    for (int side = 0; side < 2; side++) {
      const int groups = (n[side][g] + xcds - 1) / xcds;
      demand += (groups + kGroupResident[g] - 1) / kGroupResident[g];
    }
  std::vector<int>& order = b->order;
  order = b->launched;
  if (demand * xcds > b->n_cu) {
    const int cu = b->n_cu, total = (int)order.size();
    std::stable_sort(order.begin(), order.end(),
                     [&](int x, int y) { return b->slots[x].work > b->slots[y].work; });
    for (int s : order)
      if (b->slots[s].trial < 0) eff[s] = 0;
    for (int i = cu; i < total; i += 2 * cu)
      std::reverse(order.begin() + i, order.begin() + std::min(total, i + cu));
  }
  std::vector<int32_t>& act = b->next_active;
  act.assign((size_t)2 * kGroups * stride, 0);
  for (auto& side : n) std::fill(std::begin(side), std::end(side), 0);
  for (int s : order) {
    const int side = b->slots[s].late ? 1 : 0;
    const size_t at = (size_t)(side * kGroups + eff[s]) * stride;
    act[at + 1 + n[side][eff[s]]++] = s;
  }
  for (int side = 0; side < 2; side++)
    for (int g = 0; g < kGroups; g++) act[(size_t)(side * kGroups + g) * stride] = n[side][g];
  const double tl = host_now();
  // set-up work queued so far (admissions) first
  MCGPU_HIP_TRY(hipEventRecord(b->ev_ready, b->sstream));
  const bool any_main = b->late.size() < b->launched.size();
  const bool any_late = !b->late.empty();
  double tv = 0.0;
  // Order: the volume branch's clock stamp (the late boxes' tick start), the
  // main graph, then the rest of the branch, so that both sides start
  // together and the main graph waits for as little host work as possible.
  if (any_late) {
    MCGPU_HIP_TRY(hipStreamWaitEvent(b->vstream, b->ev_ready, 0));
    hipLaunchKernelGGL(k_stamp_clock, dim3(1), dim3(1), 0, b->vstream, b->d_t0);
    MCGPU_HIP_TRY(hipGetLastError());
  }
  MCGPU_HIP_TRY(hipStreamWaitEvent(b->stream, b->ev_ready, 0));
  if (any_main &&
      ((rc = upload_lists(b, false, b->stream)) ||
       (rc = launch_tick_graph(b, b->main_graph, false, b->stream, n[0], sweeps, b->ev0,
                               b->ev1))))
    return rc;
  if (any_late) {
    if ((rc = upload_lists(b, true, b->vstream))) return rc;
    const double t1 = host_now();
    if ((rc = queue_volume_moves(b, b->late, b->vstream))) return rc;
    tv = host_now() - t1;
    b->t_volume += tv;
    if ((rc = launch_tick_graph(b, b->late_graph, true, b->vstream, n[1], sweeps, nullptr,
                                nullptr)))
      return rc;
    MCGPU_HIP_TRY(hipEventRecord(b->ev_vdone, b->vstream));
    MCGPU_HIP_TRY(hipStreamWaitEvent(b->stream, b->ev_vdone, 0));
  }
  // read-back of the launched boxes' control blocks and generators into
  // staging (slots up to the highest launched one; the boundary merges the
  // launched slots only)
  const size_t nrb = (size_t)b->launched.back() + 1;
  MCGPU_HIP_TRY(hipMemcpyAsync(b->h_ctl_rb, b->d_ctl, sizeof(BoxCtl) * nrb,
                               hipMemcpyDeviceToHost, b->stream));
  MCGPU_HIP_TRY(hipMemcpyAsync(b->h_rng_rb, b->d_rng, sizeof(Rng31) * nrb,
                               hipMemcpyDeviceToHost, b->stream));
  b->pending = true;
  b->timing_pending = any_main;
  b->t_launch += host_now() - tl - tv;
  if (sync) return batch_boundary(b);
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_host_seconds(mcgpu_batch* b, double* wait, double* volume,
                                        double* launch) {
  if (!b) return MCGPU_ERR_INVALID;
  if (wait) *wait = b->t_wait;
  if (volume) *volume = b->t_volume;
  if (launch) *launch = b->t_launch;
  return MCGPU_OK;
}

namespace {

// A slot's statistics from its host mirror.
void stats_from_mirror(const mcgpu_batch* b, int s, mcgpu_box_stats* out) {
  const BoxCtl& c = b->h_ctl[s];
  out->steps_done = c.steps_done;
  out->accepted = c.accepted;
  out->volume_moves = c.vol_moves;
  out->volume_accepted = c.vol_acc;
  out->energy = c.energy;
  out->start_energy = c.start_energy;
  out->work_candidates = c.work_cand;
  out->work_sites = c.work_sites + c.work_self;
  out->neighbor_fallbacks = c.fallbacks;
  for (int k = 0; k < 3; k++) out->box[k] = c.L[k];
  out->done = c.status == kDone;
  out->fault = c.fault ? c.fault : b->slots[s].fault;
}

}  // namespace

extern "C" int mcgpu_batch_stats(mcgpu_batch* b, int32_t s, mcgpu_box_stats* out) {
  if (!b || !out || s < 0 || s >= b->max_boxes || !b->slots[s].used) {
    set_error("mcgpu_batch_stats: bad slot");
    return MCGPU_ERR_RANGE;
  }
  int rc = batch_boundary(b);
  if (rc || (rc = refresh_dirty(b, s))) return rc;
  stats_from_mirror(b, s, out);
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_peek(mcgpu_batch* b, int32_t s, mcgpu_box_stats* out) {
  if (!b || !out || s < 0 || s >= b->max_boxes || !b->slots[s].used) {
    set_error("mcgpu_batch_peek: bad slot");
    return MCGPU_ERR_RANGE;
  }
  if (b->slots[s].dirty) {
    if (!in_flight(b, s)) {
      int rc = refresh_dirty(b, s);
      if (rc) return rc;
    } else {
      // admitted just before the tick in flight, which writes its control
      // block: only the start energy is read (after the set-up stream, which
      // computes it; the tick stores it back unchanged), and the box is
      // reported as before its first move
      MCGPU_HIP_TRY(hipStreamSynchronize(b->sstream));
      MCGPU_HIP_TRY(hipMemcpy(&b->h_ctl[s].start_energy, &b->d_ctl[s].start_energy,
                              sizeof(double), hipMemcpyDeviceToHost));
      b->h_ctl[s].energy = b->h_ctl[s].start_energy;
    }
  }
  stats_from_mirror(b, s, out);
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_download(mcgpu_batch* b, int32_t s, double* x,
                                    double* y, double* z) {
  if (!b || s < 0 || s >= b->max_boxes || !b->slots[s].used || !x || !y || !z) {
    set_error("mcgpu_batch_download: bad argument");
    return MCGPU_ERR_RANGE;
  }
  int rc = batch_quiesce(b);
  if (rc) return rc;
  // the three arrays lie one after another in the box's block: one copy, to
  // pinned memory (a copy to pageable memory goes through the runtime's own
  // staging, three times)
  const BoxView& v = b->h_table[s].bv;
  const size_t nb = 8 * (size_t)v.n_site;
  const BoxLayout& L = b->slots[s].lay;
  const size_t span = L.z - L.x + nb;
  const ImagePart parts[] = {{0, x, nb}, {L.y - L.x, y, nb}, {L.z - L.x, z, nb}};
  for (size_t at = 0; at < span;) {
    const size_t n = std::min(span - at, kStageBytes);
    if ((rc = stage_room(b, n, Stage::kLook))) return rc;
    const char* from = b->h_stage + b->stage_at;  // not kept past this call
    MCGPU_HIP_TRY(hipMemcpyAsync((void*)from, (const char*)v.x + at, n, hipMemcpyDeviceToHost,
                                 b->stream));
    MCGPU_HIP_TRY(hipStreamSynchronize(b->stream));
    for_image(parts, 3, at, n,
              [&](size_t to, char* host, size_t k) { std::memcpy(host, from + to, k); });
    b->stage_used = std::max(b->stage_used, b->stage_at + n);
    at += n;
  }
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_trace(mcgpu_batch* b, int32_t s, int32_t* mol,
                                 double* delta, int8_t* acc, int64_t cap,
                                 int64_t* n) {
  if (!b || s < 0 || s >= b->max_boxes || !b->slots[s].used || !n) {
    set_error("mcgpu_batch_trace: bad argument");
    return MCGPU_ERR_RANGE;
  }
  int rc = batch_quiesce(b);
  if (rc) return rc;
  const BatchBox& E = b->h_table[s];
  if (!E.record) {
    set_error("mcgpu_batch_trace: box was added without record_trace");
    return MCGPU_ERR_STATE;
  }
  const int64_t k = std::min<int64_t>(cap, b->h_ctl[s].steps_done);
  if (k > 0) {
    if (mol) MCGPU_HIP_TRY(hipMemcpyAsync(mol, E.tr_mol, 4 * k, hipMemcpyDeviceToHost, b->stream));
    if (delta) MCGPU_HIP_TRY(hipMemcpyAsync(delta, E.tr_de, 8 * k, hipMemcpyDeviceToHost, b->stream));
    if (acc) MCGPU_HIP_TRY(hipMemcpyAsync(acc, E.tr_acc, k, hipMemcpyDeviceToHost, b->stream));
    MCGPU_HIP_TRY(hipStreamSynchronize(b->stream));
  }
  *n = k;
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_volume_trace(mcgpu_batch* b, int32_t s,
                                        mcgpu_volume_record* out, int64_t cap,
                                        int64_t* n) {
  if (!b || s < 0 || s >= b->max_boxes || !b->slots[s].used || !n) {
    set_error("mcgpu_batch_volume_trace: bad argument");
    return MCGPU_ERR_RANGE;
  }
  int rc = batch_quiesce(b);
  if (rc) return rc;
  const BatchBox& E = b->h_table[s];
  if (!E.tr_vol) {
    set_error("mcgpu_batch_volume_trace: box is not NPT or was added without record_trace");
    return MCGPU_ERR_STATE;
  }
  const int64_t k = std::min<int64_t>(std::min<int64_t>(cap, E.tr_vol_cap),
                                      b->h_ctl[s].vol_moves);
  if (k > 0 && out) {
    MCGPU_HIP_TRY(hipMemcpyAsync(out, E.tr_vol, sizeof(mcgpu_volume_record) * k,
                                 hipMemcpyDeviceToHost, b->stream));
    MCGPU_HIP_TRY(hipStreamSynchronize(b->stream));
  }
  *n = k;
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_kernel_ms(mcgpu_batch* b, double* avg_ms,
                                     int64_t* launches) {
  if (!b || !avg_ms || !launches) return MCGPU_ERR_INVALID;
  int rc = batch_boundary(b);
  if (rc) return rc;
  *launches = b->kernel_launches;
  *avg_ms = b->kernel_launches ? b->kernel_ms_sum / b->kernel_launches : 0.0;
  b->kernel_ms_sum = 0.0;
  b->kernel_launches = 0;
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_memory(mcgpu_batch* b, size_t* used, size_t* peak,
                                  size_t* capacity) {
  if (!b) return MCGPU_ERR_INVALID;
  if (used) *used = b->arena.used();
  if (peak) *peak = b->arena.peak();
  if (capacity) *capacity = b->arena.capacity();
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_set_autotune(mcgpu_batch* b, int32_t on) {
  if (!b) return MCGPU_ERR_INVALID;
  b->autotune = on != 0;
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_tuning(mcgpu_batch* b, int64_t* keys, int32_t* threads,
                                  double* moves_per_tick, int32_t cap, int32_t* n) {
  if (!b || !n) return MCGPU_ERR_INVALID;
  int k = 0;
  for (const auto& kv : b->tune) {
    if (kv.second.best < 0) continue;
    if (k < cap) {
      if (keys) keys[k] = kv.first;
      if (threads) threads[k] = kGroupNT[kv.second.best];
      for (int g = 0; moves_per_tick && g < kGroups; g++)
        moves_per_tick[kGroups * k + g] =
            kv.second.samples[g] ? kv.second.moves[g] / kv.second.samples[g] : 0.0;
    }
    k++;
  }
  *n = k;
  return MCGPU_OK;
}

extern "C" int mcgpu_batch_group(mcgpu_batch* b, int32_t s, int32_t* threads) {
  if (!b || !threads || s < 0 || s >= b->max_boxes || !b->slots[s].used)
    return MCGPU_ERR_RANGE;
  *threads = kGroupNT[b->slots[s].group];
  return MCGPU_OK;
}
