// cth_sweep.h: the forward stripe sweep shared by the phase-1 DP (dp.hip) and
// the MAP kernels (map.hip).
//
// A stripe is 64 query rows, one per lane of a wavefront; the wavefront
// sweeps the template's columns along anti-diagonals, lane l one column
// behind lane l-1.  The sweep runs in phases of 32 steps: in phase k lane l
// visits columns 32k-1-l .. 32k+30-l, so that every 32x32 block of the
// reference starts and ends with a phase, its boundary rules apply at phase
// starts only, and the steps inside a phase need no tests.
//
// The stripes of one pair run on up to W wavefronts of a workgroup, stripe s
// on wavefront s mod W, kLag phases behind stripe s-1, with a barrier after
// every phase.  Stripe s-1 has then stored a column of its bottom row, and
// finished with that column of the buffer of maxima (cth_flow.h), at least
// one barrier before stripe s reads it; no two stripes touch one column in
// the same phase (two phases of lag would not do).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cth_dev.h"

constexpr int kSweepLag = 3;

// phases of one stripe (the last ends the upper half-wavefront's last block)
__host__ __device__ __forceinline__ int sweep_phases(int lt) { return ((lt + 31) >> 5) + 2; }

// the phase of the pair's schedule in which stripe s starts
__host__ __device__ __forceinline__ int sweep_start(int s, int W, int P) {
  const int round = s / W, period = P > kSweepLag * W ? P : kSweepLag * W;
  return round * period + (s - round * W) * kSweepLag;
}

// Column transitions: a ring of the wavefront's last 128 columns in LDS, each
// column as two float4 (MM, MI, IM, II and MD, DM, DD), the ring's first 32
// columns again behind its end so that a lane's 32 columns of a phase are
// consecutive and a step's reads are two ds_read_b128 at immediate offsets.
// The reads cost no VALU; handing seven values from lane to lane each step
// costs seven DPP moves and the copies that feed lane 0.
constexpr int kRing = 128, kRingCols = kRing + 32;
constexpr int kRingBytes = 2 * kRingCols * 16;

// field order of the two halves of a column's entry
enum { kT0MM = 0, kT0MI, kT0IM, kT0II, kT1MD = 0, kT1DM, kT1DD };

// The loads of the ring's 32 columns from C on, for profile transitions at
// vector tb (lanes 0..31 one column's first half each, lanes 32..63 the
// second).  Columns before the profile get `before`, columns past it
// `after`.
struct ring_block {
  float4 v;
};
__device__ __forceinline__ ring_block ring_load(const cth_dpset& db, int64_t tb, int lt, int C, float before,
                                                float after) {
  const int lane = threadIdx.x & 63, c = C + (lane & 31);
  const bool hi = lane >= 32, in = 0 <= c && c < lt;
  const float out = c < 0 ? before : after;
  const int64_t at = tb + (in ? c : 0);
  ring_block b;
  b.v = make_float4(out, out, out, out);
  if (in) {
    const float* const t = db.trn + at;
    b.v.x = t[(hi ? CTH_MD : CTH_MM) * db.ldtr];
    b.v.y = hi ? t[CTH_DM * db.ldtr] : t[CTH_MI * db.ldtr + 1];
    b.v.z = t[(hi ? CTH_DD : CTH_IM) * db.ldtr];
    b.v.w = hi ? 0.0f : t[CTH_II * db.ldtr + 1];
  }
  return b;
}
__device__ __forceinline__ void ring_store(float4* ring, int C, const ring_block& b) {
  const int lane = threadIdx.x & 63, slot = C & (kRing - 1);
  float4* const at = ring + (lane >= 32 ? kRingCols : 0) + slot + (lane & 31);
  *at = b.v;
  if (slot == 0) at[kRing] = b.v;
}

// Barrier of the workgroup's wavefronts that orders their LDS accesses only
// (__syncthreads would also wait for the loads in flight).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// byte offset of an LDS object
__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}

// the neighbour row's value: lane l takes lane l-1's v, lane 0 keeps old
__device__ __forceinline__ float dpp_shr1(float old_lane0, float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old_lane0),
                                                               __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, false));
}

__device__ __forceinline__ int corner_maxlen(int lq, int lt) {
  int m = (int)rintf(CTH_CORNERPRC * (float)(lq > lt ? lq : lt));
  return m > CTH_MAXCORNER ? CTH_MAXCORNER : m;
}

// The columns of query row y outside the matrix's ignored corners, as lo ..
// hi (empty when lo > hi).  The corners are the cells with lq <= y + edge and
// x <= edge + y - lq, and those with lt - edge + y <= x and y < edge.
__device__ __forceinline__ void valid_columns(int lq, int lt, int edge, int y, int& lo, int& hi) {
  lo = lq <= y + edge ? max(0, edge + y - lq + 1) : 0;
  hi = y < edge ? min(lt - 1, lt - edge + y - 1) : lt - 1;
}
__device__ __forceinline__ bool in_valid_area(int lq, int lt, int edge, int y, int x) {
  int lo, hi;
  valid_columns(lq, lt, edge, y, lo, hi);
  return 0 <= y && y < lq && lo <= x && x <= hi;
}
