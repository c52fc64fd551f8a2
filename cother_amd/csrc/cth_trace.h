// cth_trace.h: a wavefront's walk over the traceback bytes of one pair, shared
// by the phase-1 finalisation (dp.hip) and the MAP traceback (map.hip).
//
// Walked by one lane, each step waits for its byte from memory: ~0.3 us a
// step, of which the other lanes take no part (120 us for paths of 250 steps,
// 330 us for 1500 paths of up to 372).  Here the wavefront copies a tile of
// 64 rows x up to 61 columns up to the walk's position into LDS, and takes a
// whole run of equal moves at once: lane k looks at the k-th cell ahead in
// each direction, and the first lane whose cell differs ends the run.  The
// path comes out in chunks, one step per lane, so that what is done with its
// cells (scores, residues, rows of the alignment) is done for a chunk at a
// time, its loads together.  1500 such paths take 24 us, the others 8 to 15.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cth_consts.h"

constexpr int kTracePitch = 17;                     // dwords of a tile row: 64 bytes, and 4 to spread the banks
constexpr int kTraceTileBytes = 64 * kTracePitch * 4;

// Walk from (x, y) until a stop cell or the matrix's edge; x and y end there.
// btck: the pair's byte of row 0, column 0; rows are ldsc bytes apart, a
// multiple of 4 below 2^32.  tile: kTraceTileBytes of LDS of this wavefront's own.
// chunk(cnt, px, py, move) is called for every kChunk steps of the path and
// for the rest: lane l < cnt has step l's cell and move.  kDiag: steps are the
// diagonal ones only.  Each turn of the loop takes a step at least, so the
// walk ends.
template <int kChunk, bool kDiag, class Chunk>
__device__ __forceinline__ void trace_walk(const uint8_t* __restrict__ btck, int64_t ldsc, int& x, int& y,
                                           uint32_t* tile, Chunk&& chunk) {
  const int lane = threadIdx.x & 63;
  const uint8_t* const bytes = reinterpret_cast<const uint8_t*>(tile);
  constexpr int kRow = 4 * kTracePitch;
  x = __builtin_amdgcn_readfirstlane(x);
  y = __builtin_amdgcn_readfirstlane(y);
  int have = 0, px = 0, py = 0, pb = CTH_BT_STOP;
  int ty = 0, c0 = 0, al = 0;  // the tile: row of its first line, first column, its offset in a line
  bool loaded = false;
  while (x >= 0 && y >= 0) {
    if (!loaded || ty - y > 63 || x < c0) {
      ty = y;
      c0 = x > 60 ? x - 60 : 0;
      const uint8_t* const p = btck + (int64_t)ty * ldsc + c0;
      al = (int)(reinterpret_cast<uintptr_t>(p) & 3);
      const int d = lane & 15;
      // rows above 0 and dwords beyond column x's repeat the last, unused
      const uint8_t* const line = p - al + 4 * min(d, (x - c0 + al) >> 2);
      uint32_t v[16];
#pragma unroll
      for (int i = 0; i < 16; i++)
        v[i] = *reinterpret_cast<const uint32_t*>(line - (uint64_t)(uint32_t)min(4 * i + (lane >> 4), ty) * (uint32_t)ldsc);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int i = 0; i < 16; i++) tile[(4 * i + (lane >> 4)) * kTracePitch + d] = v[i];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      loaded = true;
    }
    // the cells ahead: lane k the k-th, if it lies in the tile
    const int r = ty - y, c = x - c0;
    const bool rin = r + lane <= 63 && lane <= y, cin = lane <= c;
    const int at = r * kRow + al + c;
    const int left = cin ? bytes[at - lane] : CTH_BT_STOP;
    const int up = rin ? bytes[at + lane * kRow] : CTH_BT_STOP;
    const int diag = rin && cin ? bytes[at + lane * (kRow - 1)] : CTH_BT_STOP;
    const int b = __builtin_amdgcn_readfirstlane(left);  // lane 0's: the cell itself
    if (b == CTH_BT_STOP) break;
    const uint64_t same = b == CTH_BT_LEFT ? __builtin_amdgcn_ballot_w64(left == CTH_BT_LEFT)
                          : b == CTH_BT_UP ? __builtin_amdgcn_ballot_w64(up == CTH_BT_UP)
                                           : __builtin_amdgcn_ballot_w64(diag == b);
    int run = ~same ? __builtin_ctzll(~same) : 64;
    const int dx = b == CTH_BT_UP ? 0 : 1, dy = b == CTH_BT_LEFT ? 0 : 1;
    if (!kDiag || (b != CTH_BT_UP && b != CTH_BT_LEFT)) {
      run = min(run, kChunk - have);
      const int k = lane - have;
      if (0 <= k && k < run) { px = x - k * dx; py = y - k * dy; pb = b; }
      have += run;
    }
    x -= run * dx;
    y -= run * dy;
    if (have == kChunk) {
      chunk(kChunk, px, py, pb);
      have = 0;
    }
  }
  if (have) chunk(have, px, py, pb);
}
