// glibc random_r TYPE_3 generator state and steps, usable from host and
// device code.  MathLibrary.cpp:27-33 (seed/randomReal) draws from it via
// srand/rand; keeping a per-box copy on the device lets batched boxes
// reproduce the reference's trial-move sequence without host round trips.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define MCGPU_HD __host__ __device__
#else
#define MCGPU_HD
#endif

namespace mcgpu {

// 31 state words, front index f and rear index r = f - 3 (mod 31).
// rand(): state[f] += state[r]; return the new word >> 1.
struct Rng31 {
  int32_t s[31];
  int32_t f;
  int32_t r;
};

MCGPU_HD inline int32_t rng31_next(Rng31& g) {
  const uint32_t v = (uint32_t)g.s[g.f] + (uint32_t)g.s[g.r];
  g.s[g.f] = (int32_t)v;
  g.f = (g.f == 30) ? 0 : g.f + 1;
  g.r = (g.r == 30) ? 0 : g.r + 1;
  return (int32_t)(v >> 1);
}

// srand(seed): Park-Miller words via Schrage's decomposition, 310 discards.
MCGPU_HD inline void rng31_seed(Rng31& g, uint32_t seed) {
  if (seed == 0) seed = 1;
  int32_t word = (int32_t)seed;
  g.s[0] = word;
  for (int i = 1; i < 31; i++) {
    const long long hi = word / 127773;
    const long long lo = word % 127773;
    long long w = 16807 * lo - 2836 * hi;
    if (w < 0) w += 2147483647;
    word = (int32_t)w;
    g.s[i] = word;
  }
  g.f = 3;
  g.r = 0;
  for (int i = 0; i < 310; i++) (void)rng31_next(g);
}

// A launch's place in its generator's stream, which it draws ahead, 31 positions
// at a time, into a ring of kRing entries (position i in entry i mod kRing):
// pos, the current move's first draw, and head, the position after the last
// drawn.  The front index and the ring entry follow from pos modulo 31 and 64,
// so both positions are taken back by the least common multiple when pos passes
// it, and a launch may make any number of moves.
constexpr int kRing = 64;
constexpr int kStreamWrap = 31 * kRing;
struct StreamAt {
  int pos = 0;
  int head = 0;
};

// A move of `draws` draws is done (8, and 1 when it took its uniform).
MCGPU_HD inline void stream_advance(StreamAt& a, int draws) {
  a.pos += draws;
  if (a.pos >= kStreamWrap) {
    a.pos -= kStreamWrap;
    a.head -= kStreamWrap;
  }
}

// Whether the next 31 positions are to be drawn while a move is evaluated: the
// next move starts at pos + 8 or pos + 9 and its successor's draws end before
// that plus 17.  The ring then still holds the move's uniform, at pos + 8, 30 or
// more positions behind the new head.
MCGPU_HD inline bool stream_low(const StreamAt& a) { return a.head < a.pos + 26; }

// The generator's front index at pos, from the one at the launch's start.
MCGPU_HD inline int stream_front(const StreamAt& a, int start) { return (start + a.pos) % 31; }

// MathLibrary.cpp:31-33: (end - start) * ((Real)rand() / RAND_MAX) + start
MCGPU_HD inline double random_real(int32_t r, double start, double end) {
#if defined(__clang__)
#pragma clang fp contract(off)
#endif
  return (end - start) * ((double)r / 2147483647) + start;
}

}  // namespace mcgpu
