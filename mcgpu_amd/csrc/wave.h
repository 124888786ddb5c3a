// Wavefront primitives for CDNA (wave64): DPP reductions and scans, lane
// reads of 64-bit values, and the glibc TYPE_3 generator held across the
// lanes of one wave.
//
// DPP (data-parallel primitives) moves values between lanes inside the VALU
// pipeline, so a reduction step costs a few cycles instead of an LDS round
// trip (ds_bpermute, which __shfl_* compiles to).  Controls used (GFX9 DPP
// encoding): quad_perm [1,0,3,2] = 0xb1, quad_perm [2,3,0,1] = 0x4e,
// row_shr:n = 0x110 | n, row_ror:n = 0x120 | n.  Every DPP move here starts
// from 0 in the destination, so a lane whose source lies outside its row
// reads 0.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mcgpu {

__device__ __forceinline__ int wlane() { return threadIdx.x & 63; }

template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, false);
}

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = dpp_i32<CTRL>((int)(b & 0xffffffffll));
  const int hi = dpp_i32<CTRL>((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Value of lane `lane` (wave-uniform index) for every lane.
__device__ __forceinline__ int readlane_i32(int v, int lane) {
  return __builtin_amdgcn_readlane(v, lane);
}
__device__ __forceinline__ double readlane_f64(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// Sum over the 64 lanes in a fixed order; the result is wave-uniform.
// Within each 16-lane row: pairs, quads, then rotations by 4 and 8 leave the
// row sum in every lane of the row; the four row sums (read at lanes 0, 16,
// 32, 48) are added as (r0 + r1) + (r2 + r3).
__device__ __forceinline__ double wave_sum_f64(double v) {
  v += dpp_f64<0xb1>(v);
  v += dpp_f64<0x4e>(v);
  v += dpp_f64<0x124>(v);
  v += dpp_f64<0x128>(v);
  const double r0 = readlane_f64(v, 0), r1 = readlane_f64(v, 16);
  const double r2 = readlane_f64(v, 32), r3 = readlane_f64(v, 48);
  return (r0 + r1) + (r2 + r3);
}

__device__ __forceinline__ unsigned wave_sum_u32(unsigned v) {
  v += (unsigned)dpp_i32<0xb1>((int)v);
  v += (unsigned)dpp_i32<0x4e>((int)v);
  v += (unsigned)dpp_i32<0x124>((int)v);
  v += (unsigned)dpp_i32<0x128>((int)v);
  return (unsigned)readlane_i32((int)v, 0) + (unsigned)readlane_i32((int)v, 16) +
         (unsigned)readlane_i32((int)v, 32) + (unsigned)readlane_i32((int)v, 48);
}

// Inclusive prefix sum over the 64 lanes (lane order).  Rows are scanned by
// shifts of 1, 2, 4, 8 (Hillis-Steele); the totals of the preceding rows are
// then added from lanes 15, 31, 47.
__device__ __forceinline__ int wave_incl_scan_i32(int v) {
  v += dpp_i32<0x111>(v);
  v += dpp_i32<0x112>(v);
  v += dpp_i32<0x114>(v);
  v += dpp_i32<0x118>(v);
  const int t0 = readlane_i32(v, 15);
  const int t1 = readlane_i32(v, 31);
  const int t2 = readlane_i32(v, 47);
  const int row = wlane() >> 4;
  v += (row >= 1 ? t0 : 0) + (row >= 2 ? t1 : 0) + (row >= 3 ? t2 : 0);
  return v;
}

// Inclusive prefix sum over the 16 lanes of each row.
__device__ __forceinline__ int wave_incl_row_i32(int v) {
  v += dpp_i32<0x111>(v);
  v += dpp_i32<0x112>(v);
  v += dpp_i32<0x114>(v);
  v += dpp_i32<0x118>(v);
  return v;
}

// Largest of the lanes' values (all >= 0), wave-uniform.
__device__ __forceinline__ int wave_max_i32(int v) {
  auto mx = [](int a, int b) { return a > b ? a : b; };
  v = mx(v, dpp_i32<0xb1>(v));
  v = mx(v, dpp_i32<0x4e>(v));
  v = mx(v, dpp_i32<0x124>(v));
  v = mx(v, dpp_i32<0x128>(v));
  return mx(mx(readlane_i32(v, 0), readlane_i32(v, 16)),
            mx(readlane_i32(v, 32), readlane_i32(v, 48)));
}

// Number of set flags in lanes below this one (ballot + mbcnt).
__device__ __forceinline__ int wave_rank(unsigned long long ballot) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(ballot >> 32),
                                   __builtin_amdgcn_mbcnt_lo((unsigned)ballot, 0u));
}

// Value of lane `lane` (any lane's own index) for every lane.
__device__ __forceinline__ int shuffle_i32(int v, int lane) {
  return __builtin_amdgcn_ds_bpermute(lane << 2, v);
}

// The two values' sums over the 64 lanes, at once and in a fixed order: swaps
// between wave halves leave a's lane pairs summed in lanes 0..31 and b's in
// lanes 32..63, DPP sums each 16-lane row.  Row r holds its sum in every lane:
// rows 0 and 1 add up to a's total, rows 2 and 3 to b's.
__device__ __forceinline__ double wave_row_sums(double a, double b) {
  typedef unsigned uint2v __attribute__((ext_vector_type(2)));
  const uint2v lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a),
                                                     (unsigned)__double2loint(b), false, false);
  const uint2v hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a),
                                                     (unsigned)__double2hiint(b), false, false);
  double v = __hiloint2double((int)hi.x, (int)lo.x) + __hiloint2double((int)hi.y, (int)lo.y);
  v += dpp_f64<0xb1>(v);
  v += dpp_f64<0x4e>(v);
  v += dpp_f64<0x124>(v);
  v += dpp_f64<0x128>(v);
  return v;
}

// a: the value of lane 0, b: of lane 32, in every lane, after rows 0 and 1 and
// rows 2 and 3 of v (each row's lanes alike) have been added.
__device__ __forceinline__ void wave_half_totals(double v, double& a, double& b) {
  typedef unsigned uint2v __attribute__((ext_vector_type(2)));
  uint2v lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(v),
                                               (unsigned)__double2loint(v), false, false);
  uint2v hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(v),
                                               (unsigned)__double2hiint(v), false, false);
  v = __hiloint2double((int)hi.x, (int)lo.x) + __hiloint2double((int)hi.y, (int)lo.y);
  lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(v), (unsigned)__double2loint(v),
                                        false, false);
  hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(v), (unsigned)__double2hiint(v),
                                        false, false);
  a = __hiloint2double((int)hi.x, (int)lo.x);
  b = __hiloint2double((int)hi.y, (int)lo.y);
}

// Largest of the lanes' values (all >= 0) and sum, over each half of the wave,
// in every lane of the half.
__device__ __forceinline__ void half_max_sum_i32(int v, int& mx, int& sum) {
  typedef unsigned uint2v __attribute__((ext_vector_type(2)));
  auto big = [](int a, int b) { return a > b ? a : b; };
  int m = v, t = v;
  m = big(m, dpp_i32<0xb1>(m));
  t += dpp_i32<0xb1>(t);
  m = big(m, dpp_i32<0x4e>(m));
  t += dpp_i32<0x4e>(t);
  m = big(m, dpp_i32<0x124>(m));
  t += dpp_i32<0x124>(t);
  m = big(m, dpp_i32<0x128>(m));
  t += dpp_i32<0x128>(t);
  const uint2v pm = __builtin_amdgcn_permlane16_swap((unsigned)m, (unsigned)m, false, false);
  const uint2v pt = __builtin_amdgcn_permlane16_swap((unsigned)t, (unsigned)t, false, false);
  mx = big((int)pm.x, (int)pm.y);
  sum = (int)pt.x + (int)pt.y;
}

// Inclusive prefix sum over each half of the wave.
__device__ __forceinline__ int half_incl_scan_i32(int v) {
  const int k = wlane() & 31;
  v = wave_incl_row_i32(v);
  const int first = shuffle_i32(v, (wlane() & 32) + 15);
  return k >= 16 ? v + first : v;
}

// A window of a glibc random_r TYPE_3 stream across one wave: lane k < 31 holds
// word H - 31 + k, H the position of the next word.  Drawing word by word is
// a chain of lane reads; a word is the sum of the words 31 and 3 before it, so
// the next 31 words are running sums, with stride 3, of the window (its last
// three words added to the first three sums): four doubling steps.
__device__ __forceinline__ int stream_next31(int w) {
  const int k = wlane();
  int y = w;
  const int c = shuffle_i32(w, 28 + k);
  y += k < 3 ? c : 0;
#pragma unroll
  for (int d = 3; d < 31; d *= 2) {
    const int b = shuffle_i32(y, k - d);
    y += k >= d ? b : 0;
  }
  return y;
}

// The window d <= 28 positions earlier (word n = word n + 31 - word n + 28).
__device__ __forceinline__ int stream_back(int w, int d) {
  const int k = wlane();
  const int in = shuffle_i32(w, k - d);
  const int a = shuffle_i32(w, k + 31 - d), b = shuffle_i32(w, k + 28 - d);
  return k >= d ? in : a - b;
}

}  // namespace mcgpu
