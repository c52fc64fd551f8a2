// dp.hip: phase-1 profile-profile DP with traceback, and its finalisation.
//
// k_dp computes, for one template profile per workgroup, the five-state
// local DP of ExecDP_Btck_Unroll32x (cudp/CuBatchDP_init_btck.cu:65-494)
// over the whole Lq x Lt matrix, as the stripe sweep of cth_sweep.h: the 64
// lanes of a wavefront own 64 consecutive query rows and sweep the
// anti-diagonals of the stripe; each step a lane takes its upper neighbour's
// state from lane-1 by a DPP wave_shr:1 move, and the stripes of a pair run
// on wavefronts of one workgroup.  Cell values and the maximum with its cell
// equal the reference's (dp_pair below).
//
// Bound by VALU issue together with the LDS of its rows: 43 VALU instructions per
// step (56 with traceback) in 37 (52) issue slots, which fill 73% of the cycles of a
// first pass of 128,000 pairs at 2.3 wavefronts a SIMD, 56% of one of 6000 pairs and
// 40% of a traceback pass of 1500, whose ends have few pairs in flight (counters in
// profiles/k_dp_pmc.txt).  Measured against one wavefront per pair with the boundary tests
// and the transitions' lane-to-lane moves in every step (~190 VALU): first
// pass of 128,000 pairs of 99 x 231 positions 16.6 -> 5.7 ms; a query of 2000
// positions against 130 templates of 1000-3000, whose rows were in global
// memory, 177 -> 5.9 ms for both passes; 250 positions against 4000 templates
// (median 220) 4.6 -> 0.92 ms.
//
// k_dpfin restates FinalizeDPPro (cudp/CuBatchDP_final.cu:61-292): pass
// test against the score threshold, traceback from the maximum, correlation
// bonus over DIAG scores in 32-score chunks (each chunk reduced in the
// reference's xor-butterfly order), signed square root, positive-score count
// and begin coordinates.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "cth_batch.h"
#include "cth_flow.h"
#include "cth_dev.h"
#include "cth_dp.h"
#include "cth_sweep.h"
#include "cth_trace.h"

namespace {

constexpr float kLog0 = CTH_LOG0;
// transitions of the columns past the profile: no path through them reaches
// a positive match state, however large the maximum so far
constexpr float kPast = -1e30f;

// LDS of one workgroup of W wavefronts: each wavefront's transition ring and,
// where the boundary rows are in global memory, its stages of 32 columns of
// the row above (read) and of its own bottom row (written); else the pair's
// boundary row of lt + 33 columns (MM, MI, IM, DN as float4, ND) and the
// buffer of maxima (value and cell per column).
constexpr int kStage = 32;
__host__ __device__ constexpr size_t dp_wave_lds(bool grow) { return kRingBytes + (grow ? 2 * kStage * 20 : 0); }
__host__ __device__ constexpr size_t dp_row_lds(int lt, bool grow) {
  return grow ? 0 : (size_t)20 * (lt + 33) + (size_t)8 * lt;
}

// the max the recursion takes.  kSel: the reference's select a < b ? b : a,
// whose result differs from the hardware's max only for NaN operands (and in
// the sign of a zero, which no result depends on); the hardware's max runs
// when neither set can give a NaN (cth_dpset.finite)
template <bool kSel>
__device__ __forceinline__ float mx(float a, float b) {
  if constexpr (kSel) return a < b ? b : a;
  else return __builtin_fmaxf(a, b);
}

// the state of a lane: its last column's cells, and what the diagonal
// predecessors (the row above's cells of the column before) contribute, aMM
// and aMI with the row's MM transition added already
struct dp_state {
  float cMM, cMI, cIM, cDN, cND;
  float aMM, aMI, pIM, pDN, pND;
};

// One step (one cell per lane) with the row's transitions qt, the column's T0
// and T1, the score S and the row above's b0, b1 for lane 0.  Sums are taken
// in the reference's order; max(a, b) + c stands for max(a + c, b + c), which
// is the same number (rounding is monotone), except for kSel, where a NaN
// could tell them apart.
template <bool kTrace, bool kSel>
__device__ __forceinline__ int dp_step(dp_state& d, const float* qt, const float4& T0, const float4& T1, float S,
                                       const float4& b0, float b1) {
  const float uMM = dpp_shr1(b0.x, d.cMM), uMI = dpp_shr1(b0.y, d.cMI), uIM = dpp_shr1(b0.z, d.cIM);
  const float uDN = dpp_shr1(b0.w, d.cDN), uND = dpp_shr1(b1, d.cND);
  float nMM, nIM;
  if constexpr (kSel) {
    float v = d.aMI + T0.z;
    v = mx<kSel>(v, d.pIM + qt[CTH_IM] + T0.x);
    v = mx<kSel>(v, d.pDN + qt[CTH_DM] + T0.x);
    v = mx<kSel>(v, d.pND + qt[CTH_MM] + T1.y);
    v = mx<kSel>(v, d.aMM + T0.x);
    nMM = mx<kSel>(v + S, 0.0f);
    nIM = mx<kSel>(d.cMM + qt[CTH_MI] + T0.x, d.cIM + qt[CTH_II] + T0.x);
  } else {
    const float m1 = mx<kSel>(mx<kSel>(d.aMM, d.pIM + qt[CTH_IM]), d.pDN + qt[CTH_DM]) + T0.x;
    const float v = mx<kSel>(mx<kSel>(m1, d.aMI + T0.z), d.pND + qt[CTH_MM] + T1.y);
    nMM = mx<kSel>(v + S, 0.0f);
    nIM = mx<kSel>(d.cMM + qt[CTH_MI], d.cIM + qt[CTH_II]) + T0.x;
  }
  d.aMM = uMM + qt[CTH_MM];
  d.aMI = uMI + qt[CTH_MM];
  const float nMI = mx<kSel>(d.aMM + T0.y, d.aMI + T0.w);
  const float nDN = mx<kSel>(uMM + qt[CTH_MD], uDN + qt[CTH_DD]);
  const float nND = mx<kSel>(d.cMM + T1.x, d.cND + T1.z);
  int bk = 0;
  if constexpr (kTrace) {
    float m = nMM;
    bk = nMM != 0.0f ? CTH_BT_DIAG : CTH_BT_STOP;
    if (m < nMI) { m = nMI; bk = CTH_BT_UP; }
    if (m < nIM) { m = nIM; bk = CTH_BT_LEFT; }
    if (m < nDN) { m = nDN; bk = CTH_BT_UP; }
    if (m < nND) { m = nND; bk = CTH_BT_LEFT; }
  }
  d.cMM = nMM; d.cMI = nMI; d.cIM = nIM; d.cDN = nDN; d.cND = nND;
  d.pIM = uIM; d.pDN = uDN; d.pND = uND;
  return bk;
}

// eight consecutive columns of a lane's score row, two dword-aligned 16-byte
// loads.  Every lane reads its own row, so a load touches a cache line per
// lane, and fewer, wider loads take the texture path and L1 far fewer
// requests.  The loads are not guarded: the buffer is readable 8 floats to
// either side, and what lies outside the profile is replaced at its use.
struct score8 {
  float v[8];
};
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ score8 score_load8(const float* at) {
  const float4u a = *reinterpret_cast<const float4u*>(at), b = *reinterpret_cast<const float4u*>(at + 4);
  return {{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}};
}

// Store lane 63's cells of step j to its bottom row in LDS (outA, outB: byte
// offsets of step 0's column): the lanes are chosen by exec inside one asm
// block, because a branch around the stores would keep the compiler from
// issuing the next step's LDS reads ahead of them (LDS accesses execute in
// issue order, so its own waits stay sufficient).  mask: 1 << 63, or 0 where
// no column is stored.
__device__ __forceinline__ void store_bottom(uint32_t outA, uint32_t outB, uint64_t mask, const dp_state& d) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  const f4 v = {d.cMM, d.cMI, d.cIM, d.cDN};
  asm volatile(
      "s_mov_b64 exec, %4\n\t"
      "ds_write_b128 %0, %2\n\t"
      "ds_write_b32 %1, %3\n\t"
      "s_mov_b64 exec, -1"
      :
      : "v"(outA), "v"(outB), "v"(v), "v"(d.cND), "s"(mask));
}

// Eight steps, j0 .. j0+7 of a phase.  ring: the lane's column of step j0;
// inA, inB: the row above from that step's column of lane 0; outA, outB: the
// bottom row's columns, stored by lane 63 (mask); crel: the column of
// step j0 relative to the row's first valid one, span: the last valid one
// relative to it.  kFix: scores outside the valid columns are -9 (cells of
// the ignored corners and outside the matrix, CuBatchDP_init_btck.cu:245).
// mv, ms: the lane's running maximum and the step that set it (kSel: at
// columns c + j in 0 .. clt-1 only; else no match state outside them is
// positive, CTH_SET_FINITE and kPast).
template <bool kTrace, bool kSel, bool kFix>
__device__ __forceinline__ void dp_steps8(dp_state& d, const float* qt, int j0, const float4* __restrict__ ring,
                                          const float4* __restrict__ inA, const float* __restrict__ inB,
                                          uint32_t outA, uint32_t outB, uint64_t mask, int crel,
                                          uint32_t span, int c, uint32_t clt, const score8& sc, float& mv, int& ms,
                                          uint32_t* bk) {
  if constexpr (kTrace) bk[0] = bk[1] = 0;
  int ml = -1;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const float4 T0 = ring[j], T1 = ring[kRingCols + j];
    const float4 b0 = inA[j];
    const float b1 = inB[j];
    float S = sc.v[j];
    if constexpr (kFix) S = (uint32_t)(crel + j) <= span ? S : CTH_OUTSCORE;
    const int b = dp_step<kTrace, kSel>(d, qt, T0, T1, S, b0, b1);
    if constexpr (kTrace) bk[j >> 2] |= (uint32_t)b << (8 * (j & 3));
    bool up = mv < d.cMM;
    if constexpr (kSel) up = up && (uint32_t)(c + j) < clt;
    ml = up ? j : ml;
    mv = up ? d.cMM : mv;
    store_bottom(outA + 16 * j, outB + 4 * j, mask, d);
  }
  ms = ml >= 0 ? j0 + ml : ms;
}

// The DP of query qp against template profile p on a workgroup of W
// wavefronts, whose scores begin at scores[colp] (row stride ldsc);
// traceback bytes to btck at the same offsets (kTrace).  lds: the
// workgroup's dynamic LDS (W dp_wave_lds + dp_row_lds bytes); grow: 7 x lt
// floats of global memory for the boundary row and the buffer of maxima
// (kGlobalRow).  The maximum and its cell follow the reference's buffer (see
// below); valid in every lane of wavefront 0.
//
// The reference (ExecDP_Btck_Unroll32x, cudp/CuBatchDP_init_btck.cu:246-263,
// 328, 436-464) computes 32x32 oblique blocks; thread tx of a block starting
// at column x0 in the block row of query rows 32b..32b+31 takes row
// 32b+31-tx, columns x0+tx .. x0+tx+31, keeps the first cell of a larger MM
// value (strict <), seeded from the buffer at column x0+tx-1, and at the
// block's end writes the buffer at column x0+tx+ndx (ndx = 31, but 0 for a
// block whose column x0+31 is past the end and lt-x0-32 for the block that
// covers the end; block row 0 overwrites, later ones keep the buffer's
// value unless it is smaller).  FinalizeDPPro (cudp/CuBatchDP_final.cu:
// 100-142) reduces the last 64 columns.  Here lane l of stripe s is row
// 64s+l of block row 2s + l/32 with tx = 31 - l%32; its blocks start and end
// with the phases, x0 = 32(k-1) - (32 for the upper half-wavefront) in phase
// k.  At a block end the lower half-wavefront writes before the upper one
// (its block row's blocks run two launches ahead, so where the right-edge
// writes of both meet a column, the lower one's comes first); every buffer
// column then sees its block rows' writes and reads in the reference's
// order.  Lanes past the query's end take part as the reference's threads of
// those rows do.
//
// Cells outside the matrix: the reference's rows start at column -1-(q mod
// 32) with zero states, which is where lane l's phase 0 (lower half) or 1
// (upper half) starts; rows q = 31 mod 32 see zeros left and upper-left at
// column 0, the first column of lane 31's phase 1 and lane 63's phase 2; rows
// q = 0 mod 32 see zeros above at negative columns, which are the zeroed
// states of lane 31 at that point.  So the states are zeroed at three phase
// starts, and the steps need no tests.  What lanes compute past the
// profile's end stays out of the maxima (kPast) and reaches no cell inside.
//
// Cost: 18 adds (two issue together), 7 max, 5 DPP moves and 3 instructions
// for the maximum per step, against ~190 VALU with the boundary tests,
// transitions handed from lane to lane, selects for max and score selection
// in every step.
template <bool kTrace, bool kGlobalRow, bool kSel>
__device__ __forceinline__ void dp_pair(const cth_dpset& q, int qp, const cth_dpset& db, int p, int64_t colp,
                                        int64_t ldsc, const float* __restrict__ scores, uint8_t* __restrict__ btck,
                                        float4* lds, float* grow, int W, float& best_out, uint32_t& bestxy_out) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lq = q.len[qp], lt = db.len[p];
  const int64_t qb = q.dist[qp] + qp;      // query transition vector 0
  const int64_t tb = db.dist[p] + p;       // template transition vector 0
  const int edge = corner_maxlen(lq, lt);
  const int ns = (lq + 63) >> 6, P = sweep_phases(lt);
  const int hi = lane & 32;           // 32 for the upper half-wavefront
  const int tx = 31 - (lane & 31);    // the reference's thread in its block
  float4* const wl = lds + w * (dp_wave_lds(kGlobalRow) / 16);
  float4* const ring = wl;
  // the pair's row and buffer: column c of the row at index c + 1 (index 0,
  // column -1, stays zero)
  float4* const rowA = kGlobalRow ? nullptr : lds + W * (dp_wave_lds(false) / 16);
  float* const rowB = reinterpret_cast<float*>(rowA + (lt + 33));
  float* const bmv = kGlobalRow ? grow + 5 * (int64_t)lt : rowB + (lt + 33);
  uint32_t* const bmc = reinterpret_cast<uint32_t*>(bmv + lt);
  // stages of the global row
  float4* const sinA = wl + kRingBytes / 16;
  float* const sinB = reinterpret_cast<float*>(sinA + kStage);
  float4* const soutA = sinA + kStage + kStage / 4;
  float* const soutB = reinterpret_cast<float*>(soutA + kStage);
  // the first stripe's row above: zeros
  if constexpr (!kGlobalRow) {
    for (int k = threadIdx.x; k < lt + 33; k += 64 * W) {
      rowA[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      rowB[k] = 0.0f;
    }
    lds_barrier();
  }
  // a zero in a vector register: LDS addresses built on it are not rebuilt
  // from scalar registers at every access
  int vzero;
  asm("v_mov_b32 %0, 0" : "=v"(vzero));
  const int G = sweep_start(ns - 1, W, P) + P;
  // this wavefront's current stripe
  int s = w, gs = sweep_start(w, W, P);
  float qt[CTH_NTRN];
  dp_state d;
  float mv = 0.0f;
  uint32_t mc = 0;
  int y = 0, lo = 0, hc = 0;
  const float* srow = scores;
  score8 nxt{};
  for (int g = 0; g < G; g++) {
    const int k = g - gs;
    if (k >= 0 && s < ns) {
      const int cf = 32 * k - 1 - lane;  // the lane's first column of the phase
      const int band = 2 * s + (hi >> 5);   // block row of this lane
      const int yb = 32 * band + 31;        // its last query row
      const bool bandok = 32 * band < lq;   // the block row takes part
      if (k == 0) {
        y = (s << 6) + lane;
        const bool rowok = y < lq;
        valid_columns(lq, lt, edge, y, lo, hc);
        if (hc < lo) lo = hc = 1 << 30;                  // no valid column
        if (!rowok) { lo = -(1 << 30); hc = 1 << 30; }  // what its cells hold reaches nothing
        const int64_t at = qb + (rowok ? y : 0);
        qt[CTH_MM] = q.trn[CTH_MM * q.ldtr + at];
        qt[CTH_MI] = q.trn[CTH_MI * q.ldtr + at + 1];
        qt[CTH_MD] = q.trn[CTH_MD * q.ldtr + at];
        qt[CTH_IM] = q.trn[CTH_IM * q.ldtr + at];
        qt[CTH_II] = q.trn[CTH_II * q.ldtr + at + 1];
        qt[CTH_DM] = q.trn[CTH_DM * q.ldtr + at];
        qt[CTH_DD] = q.trn[CTH_DD * q.ldtr + at];
        srow = scores + (int64_t)(rowok ? y : lq - 1) * ldsc + colp;
        nxt = score_load8(srow + max(cf, -8));
        const ring_block r0 = ring_load(db, tb, lt, -64, kLog0, kPast), r1 = ring_load(db, tb, lt, -32, kLog0, kPast),
                         r2 = ring_load(db, tb, lt, 0, kLog0, kPast);
        ring_store(ring, -64, r0);
        ring_store(ring, -32, r1);
        ring_store(ring, 0, r2);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront", "local");
        mv = 0.0f;
        mc = 0u;
      }
      // zero states: at the stripe's start, and where the boundary rules ask
      if (k < 3 && (k == 0 || lane >= (k == 1 ? 31 : 63))) {
        d.cMM = d.cMI = d.cIM = d.cDN = d.cND = 0.0f;
        d.aMM = d.aMI = 0.0f + qt[CTH_MM];
        d.pIM = d.pDN = d.pND = 0.0f;
      }
      // a block starts: seed from the buffer at the column before
      const int x0 = 32 * (k - 1) - hi;
      const bool blk = bandok && -32 <= x0 && x0 < lt;
      if (blk) {
        const int xs = x0 + tx - 1;
        const bool in = 0 <= xs && xs < lt;
        mv = in ? bmv[xs] : 0.0f;
        mc = in ? bmc[xs] : 0u;
      }
      const float mv0 = mv;
      int ms = -1;
      // the next phase's transitions (in the ring after this phase's steps)
      const ring_block nring = ring_load(db, tb, lt, 32 * k + 32, kLog0, kPast);
      // the row above from lane 0's first column on, the bottom row from lane
      // 63's (columns past the profile carry what no cell inside reads)
      const float4* inA;
      const float* inB;
      uint32_t outA, outB;
      const int kb = k < (lt >> 5) ? k : (lt >> 5);
      if constexpr (kGlobalRow) {
        if (lane < kStage) {
          const int c = 32 * k - 1 + lane;
          float v[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
          if (s > 0 && 0 <= c && c < lt) {
#pragma unroll
            for (int i = 0; i < 5; i++) v[i] = grow[(int64_t)i * lt + c];
          }
          sinA[lane] = make_float4(v[0], v[1], v[2], v[3]);
          sinB[lane] = v[4];
        }
        inA = sinA + vzero; inB = sinB + vzero;
        outA = lds_offset(soutA); outB = lds_offset(soutB);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup", "local");
      } else {
        inA = rowA + 32 * kb + vzero; inB = rowB + 32 * kb + vzero;
        outA = lds_offset(rowA) + 16 * (32 * k - 63); outB = lds_offset(rowB) + 4 * (32 * k - 63);
      }
      const uint64_t mask = __builtin_amdgcn_readfirstlane(k) >= 2 ? 1ull << 63 : 0ull;  // (scalar)
      const float4* const rg = ring + (cf & (kRing - 1));
      const bool fix = __builtin_amdgcn_ballot_w64(cf < lo || cf + 31 > hc) != 0;
      const int crel = cf - lo;
      const uint32_t span = (uint32_t)(hc - lo);
      // (with traceback 16 steps a turn: a lane's bytes go to its own row, so a
      // store touches 64 cache lines however few bytes it has: 372 positions
      // against 1500 templates 0.80 -> 0.70 ms)
      constexpr int kTurn = kTrace ? 16 : 8;
      for (int j0 = 0; j0 < 32 && 32 * k - 64 + j0 < lt; j0 += kTurn) {
        uint32_t bk[kTurn / 4];
#pragma unroll
        for (int h = 0; h < kTurn; h += 8) {
          const int jh = j0 + h;
          const score8 cur = nxt;
          nxt = score_load8(srow + max(-8, min(cf + jh + 8, lt)));
          if (fix)
            dp_steps8<kTrace, kSel, true>(d, qt, jh, rg + jh, inA + jh, inB + jh, outA + 16 * jh, outB + 4 * jh, mask,
                                          crel + jh, span, cf + jh, (uint32_t)lt, cur, mv, ms, bk + h / 4);
          else
            dp_steps8<kTrace, kSel, false>(d, qt, jh, rg + jh, inA + jh, inB + jh, outA + 16 * jh, outB + 4 * jh, mask,
                                           0, 0u, cf + jh, (uint32_t)lt, cur, mv, ms, bk + h / 4);
        }
        if constexpr (kTrace) {
          if (y < lq) {
            const int c = cf + j0;
            uint8_t* const at = btck + (int64_t)y * ldsc + colp + c;
            if (0 <= c && c + kTurn - 1 < lt) {
              memcpy(at, bk, kTurn);
            } else {
#pragma unroll
              for (int j = 0; j < kTurn; j++)
                if (0 <= c + j && c + j < lt) at[j] = (uint8_t)(bk[j >> 2] >> (8 * (j & 3)));
            }
          }
        }
      }
      // the asm stores are not counted by the compiler's waits
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
      // rows past the query's end computed on whatever lies there
      if (y >= lq) mv = mv0;
      else if (ms >= 0) mc = ((uint32_t)(cf + ms) << 16) | (uint32_t)y;
      ring_store(ring, 32 * k + 32, nring);
      // a block ends: write the buffer, the lower half-wavefront first
      const int wc = flow_write_column(x0, tx, lt);
      const bool wr = blk && flow_block_iters(x0, yb, lq, lt) >= 1 && 0 <= wc && wc < lt;
      if (wr && hi == 0 && (band == 0 || bmv[wc] < mv)) {
        bmv[wc] = mv;
        bmc[wc] = mc;
      }
      flow_phase<kGlobalRow>();
      if (wr && hi != 0 && bmv[wc] < mv) {
        bmv[wc] = mv;
        bmc[wc] = mc;
      }
      if constexpr (kGlobalRow) {
        const int c = 32 * k - 64 + lane;
        if (lane < kStage && k >= 2 && c < lt) {
          const float4 a = soutA[lane];
          grow[c] = a.x;
          grow[(int64_t)lt + c] = a.y;
          grow[(int64_t)2 * lt + c] = a.z;
          grow[(int64_t)3 * lt + c] = a.w;
          grow[(int64_t)4 * lt + c] = soutB[lane];
        }
      }
      if (k == P - 1) {
        s += W;
        gs = sweep_start(s, W, P);
      }
    }
    if constexpr (kGlobalRow) __syncthreads();
    else lds_barrier();
  }
  // FinalizeDPPro's reduction of the buffer's last 64 columns
  if (w == 0) flow_final(bmv, bmc, lt, best_out, bestxy_out);
}

// wavefronts of the largest workgroup
constexpr int kMaxWaves = 8;

template <bool kTrace, bool kGlobalRow, bool kSel>
__global__ __launch_bounds__(64 * kMaxWaves) void k_dp(cth_dpset q, int qp, cth_dpset db, int pbase,
                                                       const int* __restrict__ plist, int64_t col0, int64_t ldsc,
                                                       const float* __restrict__ scores, uint8_t* __restrict__ btck,
                                                       cth_dpres* __restrict__ res, float* __restrict__ grow,
                                                       int64_t growstride) {
  extern __shared__ float4 lds_dp[];
  const int p = plist ? plist[blockIdx.x] : pbase + blockIdx.x;
  float best = 0.0f;
  uint32_t bestxy = 0;
  dp_pair<kTrace, kGlobalRow, kSel>(q, qp, db, p, db.dist[p] - col0, ldsc, scores, btck, lds_dp,
                                    kGlobalRow ? grow + (int64_t)blockIdx.x * growstride : nullptr,
                                    (int)(blockDim.x >> 6), best, bestxy);
  if (threadIdx.x == 0) {
    res[blockIdx.x].maxsc = best;
    res[blockIdx.x].maxxy = bestxy;
  }
}

// Batched phase 1: a persistent grid works through n pairs (or the *count
// pairs listed in list), each workgroup taking the next pair from the device
// counter next; pair pairs[i] of query bq[pairs[i].b] reads that query's
// scores (and writes its traceback bytes) at the query's offset; res is per
// pair.  Pairs come in the order given (longest first), so the longest DPs
// start first.
//
// No branch in this loop depends on the lane: every lane of wavefront 0 takes
// part in the fetch (lane 0 adds 1, the others 0, so lane 0's old value is
// the pair) and the others read it from LDS.  A fetch under
// `if (threadIdx.x == 0)` lets the compiler thread that loop-invariant branch
// across the back edge, which leaves lanes 1..63 in a second copy of the loop
// that never fetches again (they re-run the first pair forever).
template <bool kTrace, bool kGlobalRow, bool kSel>
__global__ __launch_bounds__(64 * kMaxWaves) void k_dp_batch(
    cth_dpset q, cth_dpset db, const cth_bquery* __restrict__ bq, const cth_bpair* __restrict__ pairs,
    const int* __restrict__ list, const int* __restrict__ count, int n, int* __restrict__ next, int64_t ldsc,
    const float* __restrict__ scores, uint8_t* __restrict__ btck, cth_dpres* __restrict__ res,
    float* __restrict__ grow, int64_t growstride) {
  extern __shared__ float4 lds_dp[];
  __shared__ int s_next;
  const int nj = count ? *count : n;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  for (;;) {
    if (w == 0) s_next = __builtin_amdgcn_readfirstlane(atomicAdd(next, threadIdx.x == 0 ? 1 : 0));
    __syncthreads();
    // uniform: scalar loads of the pair and query
    const int k = __builtin_amdgcn_readfirstlane(s_next);
    if (k >= nj) break;
    const int i = list ? list[k] : k;
    const cth_bpair pr = pairs[i];
    const cth_bquery Q = bq[pr.b];
    float best = 0.0f;
    uint32_t bestxy = 0;
    dp_pair<kTrace, kGlobalRow, kSel>(q, Q.qp, db, pr.p, db.dist[pr.p], ldsc, scores + Q.off,
                                      kTrace ? btck + Q.off : nullptr, lds_dp,
                                      kGlobalRow ? grow + (int64_t)blockIdx.x * growstride : nullptr,
                                      (int)(blockDim.x >> 6), best, bestxy);
    if (w == 0) {
      // flow_final leaves the same maximum in every lane
      res[i].maxsc = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, best)));
      res[i].maxxy = (uint32_t)__builtin_amdgcn_readfirstlane((int)bestxy);
    }
    __syncthreads();
  }
}

// FinalizeDPPro for one profile, by a wavefront: pass test against scorethld,
// traceback from the maximum, correlation bonus, signed square root,
// positive-score count and begin coordinates into r (in every lane).  The
// bonus takes the path's scores 32 at a time, v[n] (((v[n-4] + v[n-3]) +
// v[n-2]) + v[n-1]) summed by an xor butterfly.
__device__ __forceinline__ void dpfin_pair(const cth_dpset& db, int p, int64_t colp, int64_t ldsc, const float* __restrict__ scores,
                           const uint8_t* __restrict__ btck, float scorethld, cth_dpres& r, uint32_t* tile) {
  r.passed = 0; r.score = 0.0f; r.psts = 0; r.beg = 0;
  if (r.maxsc <= scorethld) return;
  const int lane = threadIdx.x & 63;
  int x = (int)(r.maxxy >> 16), y = (int)(r.maxxy & 0xffff);
  int psts = 0;
  float sum = 0.0f, last = 0.0f;  // last: the 32 scores before
  trace_walk<32, true>(btck + colp, ldsc, x, y, tile, [&](int cnt, int px, int py, int) {
    const float v = lane < cnt ? scores[(int64_t)py * ldsc + colp + px] : 0.0f;
    psts += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v > 0.0f));
    float before[4];
    for (int j = 1; j <= 4; j++) {
      const float here = __shfl(v, lane - j & 31), prev = __shfl(last, lane - j & 31);
      before[j - 1] = lane >= j ? here : prev;
    }
    float t = lane < cnt ? v * (((before[3] + before[2]) + before[1]) + before[0]) : 0.0f;
    for (int off = 16; off >= 1; off >>= 1) t += __shfl_xor(t, off);
    sum += __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, t)));
    last = v;
  });
  sum *= 0.5f;
  sum = sum < 0.0f ? -sqrtf(-sum) : sqrtf(sum);
  const float score = r.maxsc + sum;
  r.psts = psts;
  r.beg = ((uint32_t)(x + 1) << 16) | (uint32_t)(y + 1);
  r.score = score;
  r.passed = scorethld < score ? 1 : 0;
}

// one wavefront per profile
__global__ __launch_bounds__(64) void k_dpfin(cth_dpset db, int pbase, const int* __restrict__ plist, int64_t col0,
                                              int64_t ldsc, const float* __restrict__ scores,
                                              const uint8_t* __restrict__ btck, float scorethld,
                                              cth_dpres* __restrict__ res) {
  __shared__ uint32_t tile[kTraceTileBytes / 4];
  const int p = plist ? plist[blockIdx.x] : pbase + blockIdx.x;
  cth_dpres r = res[blockIdx.x];
  dpfin_pair(db, p, db.dist[p] - col0, ldsc, scores, btck, scorethld, r, tile);
  if (threadIdx.x == 0) res[blockIdx.x] = r;
}

// Batched finalisation over the *count pairs listed in list (persistent, a
// wavefront per pair at a time), each against its query's threshold.
__global__ __launch_bounds__(64) void k_dpfin_batch(cth_dpset db, const cth_bquery* __restrict__ bq,
                                                    const cth_bpair* __restrict__ pairs, const int* __restrict__ list,
                                                    const int* __restrict__ count, int64_t ldsc,
                                                    const float* __restrict__ scores,
                                                    const uint8_t* __restrict__ btck, cth_dpres* __restrict__ res) {
  __shared__ uint32_t tile[kTraceTileBytes / 4];
  const int nj = *count;
  for (int k = blockIdx.x; k < nj; k += gridDim.x) {
    const int i = list[k];
    const cth_bpair pr = pairs[i];
    const cth_bquery Q = bq[pr.b];
    cth_dpres r = res[i];
    dpfin_pair(db, pr.p, db.dist[pr.p], ldsc, scores + Q.off, btck + Q.off, Q.scorethld, r, tile);
    if (threadIdx.x == 0) res[i] = r;
  }
}

__global__ void k_selftest_dpp(int* out) {
  const float v = (float)threadIdx.x;
  out[threadIdx.x] = (int)dpp_shr1(-1.0f, v);
}

}  // namespace

// Lane-layout check of the DPP wave_shr:1 move the DP kernel relies on:
// out[l] = l-1 for l >= 1, out[0] = -1.
extern "C" int cth_selftest_dpp(int* host_out64) {
  int* d = nullptr;
  CTH_HIP_CHECK(hipMalloc(&d, 64 * sizeof(int)));
  hipLaunchKernelGGL(k_selftest_dpp, dim3(1), dim3(64), 0, 0, d);
  CTH_HIP_CHECK(hipGetLastError());
  CTH_HIP_CHECK(hipMemcpy(host_out64, d, 64 * sizeof(int), hipMemcpyDeviceToHost));
  CTH_HIP_CHECK(hipFree(d));
  return 0;
}

// Bytes of global boundary rows a launch over np profiles of at most ltmax
// positions needs (0 when the rows fit the LDS).
extern "C" size_t cth_dp_row_bytes(int np, int ltmax) {
  return ltmax > CTH_DP_GLOBAL_FROM ? sizeof(float) * 7 * (size_t)ltmax * (size_t)(np > 0 ? np : 0) : 0;
}

namespace {

// Wavefronts per pair of np pairs of queries of lq positions and profiles of
// ltmean positions on average, ltmax at most.  One per stripe gives the
// shortest schedule of a pair (the phases until its last stripe ends), which is
// what few pairs take: 600 positions against 1300 templates 0.69 ms with eight,
// 0.82 with three.  But from a third of a stripe's phases on a wavefront waits
// for the stripe above, and it takes registers and LDS from other pairs.
// Taken is the number of phases that is least for all pairs: a compute unit's
// share (of the device's ncu) over those that fit it, plus half as many again as the longest pair's,
// which few others accompany and which start first (databases are sorted).  372
// positions against 1500 templates (235 on average, up to 700), with
// traceback (8 bytes a store): 0.8 ms with three or four, 1.19 with six; 600 against 6000
// without: 2.0 with three, 2.8 with eight.  Five to seven where there are more
// stripes load the four SIMDs unevenly (800 against 3000: 2.17 ms, with eight
// 1.77, with three 1.36).
int dp_waves(int lq, int ltmean, int ltmax, int np, bool global, bool trace, int ncu) {
  constexpr size_t kUnitLds = (size_t)160 << 10;
  const int unit = trace ? 12 : 16;  // wavefronts a compute unit holds, by their registers
  const int ns = std::max(1, (lq + 63) / 64), most = std::min(kMaxWaves, ns);
  auto schedule = [&](int W, int lt) { return sweep_start(ns - 1, W, sweep_phases(lt)) + sweep_phases(lt); };
  int best = most;
  double least = 0.0;
  for (int W = most; W >= 1; W = std::min(W - 1, 4)) {
    const size_t lds = W * dp_wave_lds(global) + dp_row_lds(ltmax, global);
    const int fit = std::max(1, std::min((int)(kUnitLds / lds), unit / W));
    const double t = (double)np / (ncu * fit) * schedule(W, ltmean) + 1.5 * schedule(W, ltmax);
    if (W == most || t < least) {
      least = t;
      best = W;
    }
  }
  return best;
}

bool dp_select(const cth_dpset* q, const cth_dpset* db) { return !cth_finite_scores(q, db); }

template <bool kTrace, bool kGlobalRow>
void dp_launch(const cth_dpset* q, int qp, const cth_dpset* db, int p0, const int* plist, int np, int W, size_t lds,
               int64_t col0, int64_t ldsc, const float* scores, uint8_t* btck, cth_dpres* res, float* grow,
               int64_t growstride, hipStream_t st) {
  if (dp_select(q, db))
    hipLaunchKernelGGL((k_dp<kTrace, kGlobalRow, true>), dim3(np), dim3(64 * W), lds, st, *q, qp, *db, p0, plist, col0,
                       ldsc, scores, btck, res, grow, growstride);
  else
    hipLaunchKernelGGL((k_dp<kTrace, kGlobalRow, false>), dim3(np), dim3(64 * W), lds, st, *q, qp, *db, p0, plist, col0,
                       ldsc, scores, btck, res, grow, growstride);
}

template <bool kTrace, bool kGlobalRow>
void dp_launch_batch(const cth_dpset* q, const cth_dpset* db, const cth_bquery* bq, const cth_bpair* pairs,
                     const int* list, const int* count, int n, int* next, int W, size_t lds, int grid, int64_t ldsc,
                     const float* scores, uint8_t* btck, cth_dpres* res, float* grow, int64_t growstride,
                     hipStream_t st) {
  if (dp_select(q, db))
    hipLaunchKernelGGL((k_dp_batch<kTrace, kGlobalRow, true>), dim3(grid), dim3(64 * W), lds, st, *q, *db, bq, pairs,
                       list, count, n, next, ldsc, scores, btck, res, grow, growstride);
  else
    hipLaunchKernelGGL((k_dp_batch<kTrace, kGlobalRow, false>), dim3(grid), dim3(64 * W), lds, st, *q, *db, bq, pairs,
                       list, count, n, next, ldsc, scores, btck, res, grow, growstride);
}

}  // namespace

// Phase 1 for np profiles (query qp of lq positions): p0 + k, or plist[k]
// (device array of absolute indices) when plist is not NULL, of at most ltmax
// positions and about ltmean on average; res[k] receives
// profile k's record.  scores: readable 8 floats to either side of its
// [lq][ldsc].  btck NULL: no traceback bytes (maximum and its coordinates
// only); finalize: run the finalisation (needs btck).  grow:
// cth_dp_row_bytes(np, ltmax) bytes of device memory when ltmax exceeds
// CTH_DP_GLOBAL_FROM (else unused).
extern "C" int cth_launch_dp_list(const cth_dpset* q, int qp, int lq, const cth_dpset* db, int p0, const int* plist,
                                  int np, int ltmean, int ltmax, int64_t col0, int64_t ldsc, const float* scores,
                                  uint8_t* btck, float scorethld, int finalize, cth_dpres* res, float* grow,
                                  hipStream_t st) {
  if (np <= 0) return 0;
  if (finalize && !btck) { cth_set_error("dp: finalisation needs the traceback"); return -1; }
  if (finalize && ldsc % 4) { cth_set_error("dp: rows of %lld traceback bytes", (long long)ldsc); return -1; }
  if (ltmax > CTH_MAXCOLUMNS) { cth_set_error("dp: profile length %d over %d", ltmax, CTH_MAXCOLUMNS); return -1; }
  const bool global = ltmax > CTH_DP_GLOBAL_FROM;
  if (global && !grow) { cth_set_error("dp: profile length %d needs global boundary rows", ltmax); return -1; }
  int dev = 0, ncu = 0;
  CTH_HIP_CHECK(hipGetDevice(&dev));
  CTH_HIP_CHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  const int W = dp_waves(lq, ltmean, ltmax, np, global, btck != nullptr, ncu);
  const size_t lds = W * dp_wave_lds(global) + dp_row_lds(ltmax, global);
  const int64_t gs = (int64_t)7 * ltmax;
  if (global) {
    if (btck)
      dp_launch<true, true>(q, qp, db, p0, plist, np, W, lds, col0, ldsc, scores, btck, res, grow, gs, st);
    else
      dp_launch<false, true>(q, qp, db, p0, plist, np, W, lds, col0, ldsc, scores, btck, res, grow, gs, st);
  } else {
    if (btck)
      dp_launch<true, false>(q, qp, db, p0, plist, np, W, lds, col0, ldsc, scores, btck, res, nullptr, 0, st);
    else
      dp_launch<false, false>(q, qp, db, p0, plist, np, W, lds, col0, ldsc, scores, btck, res, nullptr, 0, st);
  }
  CTH_HIP_CHECK(hipGetLastError());
  if (finalize) {
    hipLaunchKernelGGL(k_dpfin, dim3(np), dim3(64), 0, st, *db, p0, plist, col0, ldsc, scores, btck, scorethld, res);
    CTH_HIP_CHECK(hipGetLastError());
  }
  return 0;
}

// Host check of the rule for the wavefronts per pair, on a device of ncu compute units.
extern "C" int cth_selftest_dp_waves(int lq, int ltmean, int ltmax, int np, int trace, int ncu) {
  return dp_waves(lq, ltmean, ltmax, np, ltmax > CTH_DP_GLOBAL_FROM, trace != 0, ncu);
}

extern "C" int cth_launch_dp(const cth_dpset* q, int qp, int lq, const cth_dpset* db, int p0, int np, int ltmean,
                             int ltmax, int64_t col0, int64_t ldsc, const float* scores, uint8_t* btck,
                             float scorethld, cth_dpres* res, float* grow, hipStream_t st) {
  return cth_launch_dp_list(q, qp, lq, db, p0, nullptr, np, ltmean, ltmax, col0, ldsc, scores, btck, scorethld, 1, res,
                            grow, st);
}

// Bytes of global boundary rows a batched launch of `grid` workgroups needs.
extern "C" size_t cth_dp_batch_row_bytes(int grid, int ltmax) { return cth_dp_row_bytes(grid, ltmax); }

// Batched phase 1 (k_dp_batch) on a persistent grid of `grid` workgroups of W
// wavefronts: the first pass over n pairs (list NULL, btck NULL), or the
// traceback pass over the *count pairs of list followed by their
// finalisation (btck not NULL).  next: a device counter that starts at zero;
// ltmax: the database's longest profile; scores as in cth_launch_dp_list;
// grow: cth_dp_batch_row_bytes(grid, ltmax) bytes.
extern "C" int cth_launch_dp_batch(const cth_dpset* q, const cth_dpset* db, const cth_bquery* bq,
                                   const cth_bpair* pairs, const int* list, const int* count, int n, int* next,
                                   int ltmax, int64_t ldsc, const float* scores, uint8_t* btck, cth_dpres* res,
                                   float* grow, int grid, int W, hipStream_t st) {
  if (grid < 1) return 0;
  if (W < 1 || W > kMaxWaves) { cth_set_error("dp batch: %d wavefronts per pair", W); return -1; }
  if (btck && ldsc % 4) { cth_set_error("dp batch: rows of %lld traceback bytes", (long long)ldsc); return -1; }
  const bool global = ltmax > CTH_DP_GLOBAL_FROM;
  if (global && !grow) { cth_set_error("dp batch: profile length %d needs global boundary rows", ltmax); return -1; }
  const size_t lds = W * dp_wave_lds(global) + dp_row_lds(ltmax, global);
  const int64_t gs = (int64_t)7 * ltmax;
  if (global) {
    if (btck)
      dp_launch_batch<true, true>(q, db, bq, pairs, list, count, n, next, W, lds, grid, ldsc, scores, btck, res, grow,
                                  gs, st);
    else
      dp_launch_batch<false, true>(q, db, bq, pairs, list, count, n, next, W, lds, grid, ldsc, scores, btck, res, grow,
                                   gs, st);
  } else {
    if (btck)
      dp_launch_batch<true, false>(q, db, bq, pairs, list, count, n, next, W, lds, grid, ldsc, scores, btck, res,
                                   nullptr, 0, st);
    else
      dp_launch_batch<false, false>(q, db, bq, pairs, list, count, n, next, W, lds, grid, ldsc, scores, btck, res,
                                    nullptr, 0, st);
  }
  CTH_HIP_CHECK(hipGetLastError());
  if (btck && list) {
    hipLaunchKernelGGL(k_dpfin_batch, dim3(grid), dim3(64), 0, st, *db, bq, pairs, list, count, ldsc, scores, btck,
                       res);
    CTH_HIP_CHECK(hipGetLastError());
  }
  return 0;
}
