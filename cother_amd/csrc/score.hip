// score.hip: the score-matrix stage on gfx950.
//
// For a query profile against a contiguous range of template positions, every
// cell of
//   S[i,j]   = Init + (SS + CVS) + DDMS
//   mod[i,j] = (SS + CVS - 0.5*CVSWGT) + (DDMS - 0.2*DDMSWGT)
// in the order the reference's three kernels accumulate them
// (cusco/CuBatchScoreMatrix.cu:236-396: CalcSM_Init_SMEMUnroll2x writes S,
// CalcSM_SSSS_CVS2S_SMEMUnroll2x_2 adds SS+CVS and writes mod,
// CalcSM_DDMS2S_SMEMUnroll2x_h2 adds DDMS to both when it is non-zero).
//
// k_score_plain writes all but the distance-match term; where a cell can have
// one, k_score_ddms adds it to both matrices afterwards (the order of the
// sums is the reference's, and the 16 bytes a cell that pass through memory
// once more are nothing beside the scan's time).
#include <float.h>

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "cth_batch.h"
#include "cth_dev.h"
#include "cth_math.h"
#include "cth_mfma.h"

namespace {

constexpr int kCols = 64;  // template columns per workgroup of the plain kernel (one per lane)

// The distance-match scan's workgroup: 256 cells, one per lane, as 32, 16 or
// 8 query rows (the fewest that hold the tile's) x 8, 16 or 32 template
// columns, whose lists are in LDS (eight workgroups a compute unit).
constexpr int kDThreads = 256, kDRows = 32, kDRowsMin = 8;
constexpr int kDColsMin = kDThreads / kDRows;
constexpr int kDLists = kDRows + kDColsMin;
static_assert(kDRowsMin + kDThreads / kDRowsMin <= kDLists, "lists of the lowest tile");
constexpr int kListEntries = 112;  // entries of a list the scan reads (0..111)
constexpr int kListPitch = 4 * 113;  // LDS bytes per list: lists fall on different banks
constexpr float kSumScale = 0x1p-6f;  // of the distance-match sums (a segment's stays below 1)

struct DdmsLds {
  // Lists as the pair table's byte rows (query lists, first) and byte columns
  // (template lists), a word per entry: the entry in the low half-word, the
  // one after next, with which the scan takes it, in the high one.  Entry 0
  // is the length.
  uint8_t list[kDLists * kListPitch];
  float dms[22 * 22];  // the pair scores times kSumScale
};

__device__ __forceinline__ float ss_lookup(const float* ss, int row, int col) {
  if (row < col) { int x = row; row = col; col = x; }
  if (row) col += row + ((row * (row - 1)) >> 1);
  return ss[col + 2];
}

// A segment's coordinates as packed words: begin B = QB | PB << 11 and end
// E = QE | PE << 11.  Every index is below 256, so with kEndBias = 0x200 in
// each 11-bit half, (E + kEndBias) - B = 0x200 + (end - begin) per half with
// no borrow between the halves, and bit 9 of the half is set exactly when
// end >= begin.  Packed words stay below 2^22, so a float 2^23 + W holds W
// exactly and its bits are kMagic + W: the kernel computes a candidate's
// begin as one fma on floats (an instruction that dual-issues) and takes its
// bits, and every word it compares carries the same kMagic, which cancels in
// each difference of a test.  The register keeps each entry as
// nb = kEndBias - B and ce = E + kEndBias (with kMagic), so that both
// differences of a test are one add or subtract from a segment's B and E.
constexpr uint32_t kPack = 0x801u;        // one index step on both axes
constexpr float kPackF = 2049.0f;
constexpr uint32_t kEndBias = 0x00100200u;
constexpr uint32_t kMagic = 0x4b000000u;  // the bits of 2^23
// entries that intersect nothing: begins 255, ends 0
constexpr uint32_t kNoBeginN = kEndBias - (kMagic + 0x0007f8ffu), kNoEnd = kMagic + kEndBias;

// the AND that is zero when segment s (begin sb, end se) does not intersect
// register entry c (nb, ce): on the query or the template axis the byte-wise
// max of the begins is <= the min of the ends
// (CuBatchScoreMatrix_ddms2s.cuh:141-153), i.e. (begin <= end within each
// segment) ce >= sb and se >= cb
__device__ __forceinline__ uint32_t overlap(uint32_t sb, uint32_t se, uint32_t nb, uint32_t ce) {
  // the three-input and as one instruction (left to itself the compiler
  // shares (ce - sb) & kEndBias between tests at the cost of an extra and)
  return __builtin_amdgcn_bitop3_b32(ce - sb, se + nb, kEndBias, 0x80);
}

// Lane masks of the comparisons of the scan: as masks each comparison is made
// once (as booleans the compiler repeats those whose negation is also used)
// and their combinations are scalar.
__device__ __forceinline__ uint64_t mask_ge(float a, float b) { return __builtin_amdgcn_fcmpf(a, b, 3); }
__device__ __forceinline__ uint64_t mask_gt(float a, float b) { return __builtin_amdgcn_fcmpf(a, b, 2); }
__device__ __forceinline__ uint64_t mask_zero(uint32_t a) { return __builtin_amdgcn_uicmp(a, 0u, 32); }
__device__ __forceinline__ bool in_mask(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// The three best segment scores m0 >= m1 >= m2 whose coordinates do not
// intersect, m0's and m1's with their coordinates.  An empty entry holds
// FLT_MIN: every comparison with a segment's sum (at least 2^-99) falls as
// with 0, and in the final sum it vanishes beside a sum or the intercept.
struct ddms_register {
  float m0, m1, m2;
  uint32_t nb0, ce0, nb1, ce1;
};
// RegisterMaxDDMScore (CuBatchScoreMatrix_ddms2s.cuh:168-261) for the lanes
// whose segment s >= m2 (begin sb, end se) changes the register; masks: ge0
// s >= m0, ge1 s >= m1, n0 and n1 s does not intersect m0, m1.  The
// reference's three cases:
//  s >= m0: s becomes m0; the old m0 becomes m1 and the old m1 m2 (dropped if
//           it intersects s), unless the old m0 intersects s: then it drops,
//           the old m1 stays m1 unless it intersects s, and m2 is empty;
//  m1 <= s < m0, s not intersecting m0: s becomes m1, the old m1 becomes m2
//           unless it intersects s;
//  m2 <= s < m1, s intersecting neither m0 nor m1: s becomes m2.
// So where s >= m0 the two change places, and what is left is inserted at m1
// or not.  Only m0's and m1's coordinates are ever tested, so m2's are not
// kept; an empty entry may keep stale coordinates (a test with it only
// decides between two empty values), and no segment intersects the initial
// ones (kNoBeginN, kNoEnd).
//
// One asm block whose assignments choose their lanes by exec: a move per
// value where selects take up to two conditional moves, and no branches (a
// branch around each case's few moves costs more than the moves).
__device__ __forceinline__ void register_max(ddms_register& R, float s, uint32_t sb, uint32_t se, uint64_t ge0,
                                             uint64_t ge1, uint64_t n0, uint64_t n1) {
  uint32_t nb = kEndBias - sb, ce = se + kEndBias;
  const float rest = in_mask(n1) ? R.m1 : FLT_MIN;
  const uint64_t insert = (ge0 & n0) | (~ge0 & ge1), self = ge0 & ~n0, low = ~(ge0 | ge1);
  uint64_t all;
  asm volatile(
      "s_mov_b64 %[all], exec\n\t"
      "s_and_b64 exec, %[all], %[ge0]\n\t"
      "v_swap_b32 %[s], %[m0]\n\t"
      "v_swap_b32 %[nb], %[nb0]\n\t"
      "v_swap_b32 %[ce], %[ce0]\n\t"
      "s_and_b64 exec, %[all], %[insert]\n\t"
      "v_mov_b32 %[m2], %[rest]\n\t"
      "v_mov_b32 %[m1], %[s]\n\t"
      "v_mov_b32 %[nb1], %[nb]\n\t"
      "v_mov_b32 %[ce1], %[ce]\n\t"
      "s_and_b64 exec, %[all], %[self]\n\t"
      "v_mov_b32 %[m1], %[rest]\n\t"
      "v_mov_b32 %[m2], 0x00800000\n\t"
      "s_and_b64 exec, %[all], %[low]\n\t"
      "v_mov_b32 %[m2], %[s]\n\t"
      "s_mov_b64 exec, %[all]"
      : [all] "=&s"(all), [s] "+v"(s), [nb] "+v"(nb), [ce] "+v"(ce), [m0] "+v"(R.m0), [m1] "+v"(R.m1),
        [m2] "+v"(R.m2), [nb0] "+v"(R.nb0), [ce0] "+v"(R.ce0), [nb1] "+v"(R.nb1), [ce1] "+v"(R.ce1)
      : [rest] "v"(rest), [ge0] "s"(ge0), [insert] "s"(insert), [self] "s"(self), [low] "s"(low)
      : "scc");
}

// CalcDDMS2ScoreSMEMh2<2,true,2> (cusco/CuBatchScoreMatrix_ddms2s_h2.cuh:435-500):
// upper diagonals j = len2>>2 .. 0 step 2, lower diagonals i = len1>>2 .. 1
// step 2; per diagonal a Kadane scan in steps of 4 cells where cells 2 and 4
// are exact pair scores and cells 1 and 3 their means; per 4-cell step the
// best qualifying segment (length >= DSTSEGM) goes to the top-3 register.
//
// What counts is the number of VALU instructions: the SIMD issues two per
// slot, of two wavefronts, one of which has to be a plain FP32 add, multiply
// or fma (source modifiers and clamp included), a u32 add, a logic op or a
// move.  The sums are kept scaled by 2^-6 (an exact scaling: no value comes
// near the denormals), which puts every segment's sum below 1 (at most 102
// cells of at most 0.5), so that one add with the clamp modifier is
// max(sum + x, 0) with the reference's one rounding.  Per cell, with x the
// cell's scaled pair score (or, for the interpolated cells, 0.5 (a + b),
// whose halving is exact and joins the sum in one fma), dd = the segment's
// begin minus the cell index (an integer value, <= 0) and big = 2^126:
//   nz   = clamp(u * big)          1 when the previous sum is > 0, else 0
//                                  (positive sums are far above 2^-126)
//   dd   = fma(nz, dd, -nz)        dd - 1, or 0 where the segment restarts
//   u    = clamp(u + x)
// and, where some lane of the wavefront can have a candidate in the step,
//   cand = u * clamp(-dd - 4)      u if the segment has at least DSTSEGM = 6
//                                  cells (dd <= -5), else 0
// and the step's best is the max of its four candidates: the reference takes
// a cell when its sum exceeds the best so far, i.e. the first cell reaching
// the max.  The clamp at 0 differs from the reference's select only in the
// sign of a zero sum, and a zero is never registered.  The top-3 register
// holds scaled sums too (scaling commutes with every comparison and with the
// rounding of the final sum, which is scaled back exactly).
#define CTH_DDMS_CELL(U, DD, SUM, UOUT, DDOUT)                                \
  const float nz##UOUT = __builtin_amdgcn_fmed3f((U) * big, 0.0f, 1.0f);      \
  const float DDOUT = fmaf(nz##UOUT, DD, -nz##UOUT);                          \
  const float UOUT = __builtin_amdgcn_fmed3f(SUM, 0.0f, 1.0f);
// one 4-cell step, cells K0+1..K0+4 relative to the base ib, with the pair
// scores S0, S2, S4 of cells K0 (the previous step's last cell), K0+2 and
// K0+4, and FB the float 2^23 + the packed coordinates of cell K0+1 on both
// axes.  Where no lane has a sum or a positive score in the step every sum
// stays 0 (and dd, which then counts for nothing, as it is).  A candidate's
// segment has 6 cells or more at a cell of the step, so at least 3 at its
// first (dd1 <= -2): where no lane's has, the step ends there.  The begin and
// end of the step's best are recovered only when it can be registered.  Three levels: the
// step's best is a candidate when it reaches m2 (empty most of the time: a
// growing best segment drops it); a candidate whose segment already meets m0
// with its end at the step's first cell and that scores below m0 is dropped
// after one intersection test, before its end cell is selected (most
// candidates are of this kind: segments of neighbouring diagonals through
// the same region); the rest take the full test, and the update runs for a
// wavefront only when one of its lanes really changes its register.  The
// empty asm statements keep the candidate's packed words in registers:
// without them the compiler folds their sums into each test as
// scalar-operand adds, which issue one per cycle.
#define CTH_DDMS_4CELL(S0, S2, S4, FB)                                        \
  if (mask_gt(fmaxf(fmaxf(u, S2), S4), 0.0f) != 0) {                          \
    const float t1 = S0 + S2, t3 = S2 + S4;                                   \
    CTH_DDMS_CELL(u, dd, fmaf(t1, 0.5f, u), u1, dd1)                          \
    CTH_DDMS_CELL(u1, dd1, u1 + S2, u2, dd2)                                  \
    CTH_DDMS_CELL(u2, dd2, fmaf(t3, 0.5f, u2), u3, dd3)                       \
    CTH_DDMS_CELL(u3, dd3, u3 + S4, u4, dd4)                                  \
    u = u4;                                                                   \
    dd = dd4;                                                                 \
    if (mask_ge(-2.0f, dd1) != 0) {                                           \
    const float cd1 = u1 * __builtin_amdgcn_fmed3f(-dd1 - 4.0f, 0.0f, 1.0f);  \
    const float cd2 = u2 * __builtin_amdgcn_fmed3f(-dd2 - 4.0f, 0.0f, 1.0f);  \
    const float cd3 = u3 * __builtin_amdgcn_fmed3f(-dd3 - 4.0f, 0.0f, 1.0f);  \
    const float cd4 = u4 * __builtin_amdgcn_fmed3f(-dd4 - 4.0f, 0.0f, 1.0f);  \
    const float scom = fmaxf(fmaxf(cd1, cd2), fmaxf(cd3, cd4));               \
    if (in_mask(mask_ge(scom, R.m2))) {                                       \
      /* the step's first cell on both axes, packed (with kMagic) */          \
      const uint32_t base = __float_as_uint(FB);                              \
      /* begin: the candidate's segment has DSTSEGM or more cells at a cell   \
         of this step, so it runs at the step's first cell, whose dd gives    \
         its begin: 2^23 + first cell + dd1 (1 + 2^11), exact in float */     \
      uint32_t sb = __float_as_uint(fmaf(dd1, packf, FB));                    \
      asm("" : "+v"(sb));                                                     \
      /* the end lies in cells 1..4 and an intersection, once there, stays as \
         the end grows: a segment that meets m0 ending at cell 1 meets it at  \
         its end, and below m0 it cannot change the register */               \
      const uint64_t ge0 = mask_ge(scom, R.m0);                               \
      if (in_mask(ge0 | mask_zero(overlap(sb, base, R.nb0, R.ce0)))) {        \
        /* end: the first of cells 1..4 reaching scom, the cell k + 1 after   \
           the first, as 2^23 + first cell + k (1 + 2^11); n_k = 1 where cell \
           k is below scom and 0 at scom (scom >= cd_k, and the scaled sums   \
           are multiples of 2^-105, so a difference is 0 or scaled by 2^120   \
           at least 1), so k = n1 (1 + n2 (1 + n3)):                          \
           fmas that dual-issue, where compares and selects do not */         \
        const float sbig = scom * big2;                                       \
        const float n1 = __builtin_amdgcn_fmed3f(fmaf(cd1, -big2, sbig), 0.0f, 1.0f); \
        const float n2 = __builtin_amdgcn_fmed3f(fmaf(cd2, -big2, sbig), 0.0f, 1.0f); \
        const float n3 = __builtin_amdgcn_fmed3f(fmaf(cd3, -big2, sbig), 0.0f, 1.0f); \
        uint32_t se = __float_as_uint(fmaf(n1, fmaf(n2, fmaf(n3, packf, packf), packf), FB)); \
        asm("" : "+v"(se));                                                   \
        const uint64_t free0 = mask_zero(overlap(sb, se, R.nb0, R.ce0));      \
        const uint64_t free1 = mask_zero(overlap(sb, se, R.nb1, R.ce1));      \
        const uint64_t ge1 = mask_ge(scom, R.m1);                             \
        if (in_mask(ge0 | (free0 & (ge1 | free1))))                           \
          register_max(R, scom, sb, se, ge0, ge1, free0, free1);              \
      }                                                                       \
    }                                                                         \
    }                                                                         \
  }
// eight cells (two steps) from entry O on; the pair scores of the step after
// are loaded one step ahead (lists are padded).  GUARD: whether the second
// step is due.
#define CTH_DDMS_8CELL(O, GUARD)                                              \
  {                                                                           \
    const uint32_t a6 = lds_u32(lds, qo + 4 * (O + 6)) + lds_u32(lds, to + 4 * (O + 6)); \
    const float n2 = pair(lds, a6 & low), n4 = pair(lds, a6 >> 16);           \
    CTH_DDMS_4CELL(s0, s2, s4, O ? fb + O * kPackF : fb)                      \
    const uint32_t a10 = lds_u32(lds, qo + 4 * (O + 10)) + lds_u32(lds, to + 4 * (O + 10)); \
    const float p2 = pair(lds, a10 & low), p4 = pair(lds, a10 >> 16);         \
    if (GUARD) CTH_DDMS_4CELL(s4, n2, n4, fb + (O + 4) * kPackF)              \
    s0 = n4;                                                                  \
    s2 = p2;                                                                  \
    s4 = p4;                                                                  \
  }
#define CTH_DDMS_ADVANCE(N)                                                   \
  fb += N * kPackF;                                                           \
  qo += 4 * N;                                                                \
  to += 4 * N;                                                                \
  asm("" : "+v"(qo), "+v"(to));

// The scan reads everything from the workgroup's LDS block by byte offsets
// held in vector registers.  One add of two list words gives the table
// offsets of two pairs.  kDms: the pair-score table in the block
constexpr int kDms = (int)offsetof(DdmsLds, dms);
__device__ __forceinline__ uint32_t lds_u32(const char* lds, int off) {
  return *reinterpret_cast<const uint32_t*>(lds + off);
}
__device__ __forceinline__ float pair(const char* lds, uint32_t off) {
  return *reinterpret_cast<const float*>(lds + kDms + off);
}

// The shortest and the longest list of the wavefront's cells on each axis
// (of the cells whose lists both reach DSTSEGM).
struct ddms_lens {
  int qmin, qmax, tmin, tmax;
};

// lds: the workgroup's block; qr, tr: byte offsets of the lane's query and
// template lists; len1, len2: their lengths, at least DSTSEGM
__device__ __forceinline__ float ddms_cell(const char* lds, int qr, int tr, int len1, int len2, const ddms_lens& n) {
  ddms_register R{FLT_MIN, FLT_MIN, FLT_MIN, kNoBeginN, kNoEnd, kNoBeginN, kNoEnd};
  // 2^126, 1 + 2^11 and 2^120 in vector registers: as scalar operands they
  // would keep the multiplies and fmas off the second issue slot (the
  // half-word mask the ands)
  float big, packf, big2;
  asm("v_mov_b32 %0, 0x7e800000" : "=v"(big));
  asm("v_mov_b32 %0, 0x7b800000" : "=v"(big2));  // 2^120
  uint32_t low;
  asm("v_mov_b32 %0, 0xffff" : "=v"(low));
  asm("v_mov_b32 %0, %1" : "=v"(packf) : "i"(__builtin_bit_cast(uint32_t, kPackF)));
  // a diagonal of `cells` cells from the entries at byte offsets qo and to on,
  // `first` its cell 1 as 2^23 + packed coordinates; full: cells that every
  // lane's diagonal has, whose steps are taken without a test of the lane's
  // end.  The offsets advance by one iteration at a time in vector registers.
  auto diagonal = [&](int qo, int to, uint32_t first, int cells, int full) {
    const uint32_t a0 = lds_u32(lds, qo) + lds_u32(lds, to), a4 = lds_u32(lds, qo + 16) + lds_u32(lds, to + 16);
    float s0 = pair(lds, a0 & low), s2 = pair(lds, a0 >> 16), s4 = pair(lds, a4 & low);
    float u = __builtin_amdgcn_fmed3f(s0, 0.0f, 1.0f);  // max(s0, 0)
    float dd = 0.0f, fb = __uint_as_float(first);
    asm("" : "+v"(qo), "+v"(to));
    int ib = 0;
    for (; ib + 12 < full; ib += 16) {
      CTH_DDMS_8CELL(0, true)
      CTH_DDMS_8CELL(8, true)
      CTH_DDMS_ADVANCE(16)
    }
    for (; ib < cells; ib += 8) {
      CTH_DDMS_8CELL(0, ib + 4 < cells)
      CTH_DDMS_ADVANCE(8)
    }
  };
  // upper diagonals, j = len2>>2 .. 0 step 2: query index i with template index
  // j + i; lower ones, i = len1>>2 .. 1: query index i + j with template index
  // j.  (len - (len >> 2) grows with len, so the shortest lists give the
  // shortest diagonals.)
  {
    int j = len2 >> 2, to = tr + 4 * (1 + j), left = len2 - j;
    uint32_t first = kMagic + kPack + ((uint32_t)j << 11);
    int most = n.tmin - (n.tmin >> 2);
    for (int k = n.tmax >> 3; k >= 0; k--) {
      if (j >= 0) diagonal(qr + 4, to, first, min(len1, left), min(n.qmin, most));
      j -= 2; to -= 8; left += 2; most += 2;
      first -= 2u << 11;
    }
  }
  {
    int i = len1 >> 2, qo = qr + 4 * (1 + i), left = len1 - i;
    uint32_t first = kMagic + kPack + (uint32_t)i;
    int most = n.qmin - (n.qmin >> 2);
    for (int k = ((n.qmax >> 2) + 1) >> 1; k > 0; k--) {
      if (i >= 1) diagonal(qo, tr + 4, first, min(left, len2), min(most, n.tmin));
      i -= 2; qo -= 8; left += 2; most += 2;
      first -= 2u;
    }
  }
  float s = 0.0f;
  s += R.m0;
  s += R.m1;
  s += R.m2;
  s *= 1.0f / kSumScale;  // the register holds scaled sums
  s = fmaf(CTH_DDMS_SLOPE * CTH_DDMS_SCALE, s, CTH_DDMS_ICEPT);
  return s * CTH_DDMSWGT;
}
#undef CTH_DDMS_CELL
#undef CTH_DDMS_4CELL
#undef CTH_DDMS_8CELL
#undef CTH_DDMS_ADVANCE

// Adds the distance-match term to the matrices that k_score_plain wrote.
//
// A wavefront covers 32 query rows x 2 template columns, each lane a cell with
// its own two lists (a tile of fewer rows, as many as the next power of two
// and more columns).  A part of a step runs when any of the wavefront's lanes
// needs it, and the lists of neighbouring positions are alike, on the query's
// side most of all.  Replayed with the synthetic lists, of a wavefront's steps
// as 1 x 64, 8 x 8, 16 x 4 and 32 x 2 cells
//   86, 55, 49, 47%  have a sum or a positive score,
//   75, 42, 37, 34%  reach the candidate test,
//   31, 23, 21, 20%  change a register;
// 64 x 1 would be 43, 31 and 19%, but its query lists take the LDS of eight
// workgroups.
//
// Bound by VALU issue: by the counters 15,500 instructions a wavefront in 9,400
// issue slots of its 9,800 cycles (1 x 64 cells with every step's arithmetic
// taken: 25,300 in 14,700).  The score stage of 250 positions against 4000
// templates (median 220) takes 61.1 ms.  With one loop over both kinds of
// diagonals, whose starts are then built anew each time, 61.9; with 16 x 4
// cells, lists read an entry at a time and no test for a step without sums
// 73.4; with 16 rows and words of two 16-bit entries added by SDWA (which issue
// alone) 68.4.  Workgroups of 512 lanes: 67.0 against 65.9 (a wavefront's place
// waits for the seven others).  Tiles of the fewest rows that hold a query's
// last ones: 40 positions against 6000 templates 5.05 ms, with 32 x 8 tiles
// alone 6.4.
// kBatch: the row tiles of several queries in one launch, ytab[blockIdx.y /
// ysplit] giving query and first row of ysplit tiles of kDRows rows.
template <bool kBatch>
__global__ __launch_bounds__(kDThreads) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_score_ddms(
    cth_dpset q, int qp, cth_dpset db, int64_t col0, int ncols, int64_t ldsc, const cth_tables* __restrict__ tabs,
    float* __restrict__ scores, float* __restrict__ mods, const int32_t* __restrict__ qoff,
    const cth_bytile* __restrict__ ytab, int ysplit, const cth_bquery* __restrict__ bq) {
  __shared__ DdmsLds L;
  const int tid = threadIdx.x;
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  int row0 = blockIdx.y * kDRows;
  if constexpr (kBatch) {
    const cth_bytile t = ytab[blockIdx.y / ysplit];
    const cth_bquery Q = bq[t.b];
    qp = Q.qp;
    row0 = t.row0 + (int)(blockIdx.y % ysplit) * kDRows;
    scores += Q.off;
    mods += Q.off;
  }
  const int rows = min(kDRows, q.len[qp] - row0);
  if (rows <= 0) return;
  // rows of a wavefront's cells, as a shift (a wavefront's columns lie within
  // the tile's), and the tile's columns; workgroups past the last one leave
  const int tqs = max(6 - __builtin_ctz(kDThreads / kDRowsMin), rows > 1 ? 32 - __builtin_clz(rows - 1) : 0);
  const int cols = kDThreads >> max(tqs, __builtin_ctz(kDRowsMin));
  const int c0 = blockIdx.x * cols;
  if (c0 >= ncols) return;
  const int64_t q0 = q.dist[qp] + row0;
  for (int k = tid; k < 22 * 22; k += kDThreads) L.dms[k] = kSumScale * tabs->dms[k];
  for (int k = tid; k < rows * 128; k += kDThreads) {
    const int r = k >> 7, e = k & 127;
    if (e < kListEntries)
      *reinterpret_cast<int32_t*>(&L.list[r * kListPitch + 4 * e]) = qoff[(size_t)(q0 + r) * CTH_DDSTRIDE + e];
  }
  // template values (<= 21) times 4; the length byte stays
  const int t0 = rows * kListPitch;
  for (int k = tid; k < cols * 32; k += kDThreads) {
    const int c = k >> 5, d = k & 31;
    if (d >= kListEntries / 4) continue;
    uint32_t v = 0, v1 = 0;  // (an empty list)
    if (c0 + c < ncols) {
      const uint32_t* const src = reinterpret_cast<const uint32_t*>(db.dd + (size_t)(col0 + c0 + c) * CTH_DDSTRIDE);
      v = src[d];
      v1 = src[d + 1];
    }
    v = d == 0 ? (v & 0xffu) | ((v & 0xffffff00u) << 2) : v << 2;
    v1 <<= 2;
    uint32_t* const dst = reinterpret_cast<uint32_t*>(&L.list[t0 + c * kListPitch + 16 * d]);
    // bytes 0 and 2, 1 and 3, 2 and 4, 3 and 5
    dst[0] = __builtin_amdgcn_perm(v1, v, 0x0c020c00u);
    dst[1] = __builtin_amdgcn_perm(v1, v, 0x0c030c01u);
    dst[2] = __builtin_amdgcn_perm(v1, v, 0x0c040c02u);
    dst[3] = __builtin_amdgcn_perm(v1, v, 0x0c050c03u);
  }
  __syncthreads();

  const int r = lane >> (6 - tqs), c = (w << (6 - tqs)) + (lane & (63 >> tqs));
  if ((w << (6 - tqs)) >= cols) return;
  const char* const lds = reinterpret_cast<const char*>(&L);
  const int qr = kListPitch * min(r, rows - 1), tr = t0 + kListPitch * c;
  const int len1 = (int)(lds_u32(lds, qr) & 0xff), len2 = (int)(lds_u32(lds, tr) & 0xff);
  const bool on = r < rows && c0 + c < ncols && len1 >= CTH_DSTSEGM && len2 >= CTH_DSTSEGM;
  ddms_lens n{on ? len1 : CTH_MAXDST, on ? len1 : 0, on ? len2 : CTH_MAXDST, on ? len2 : 0};
  for (int o = 32; o >= 1; o >>= 1) {
    n.qmin = min(n.qmin, __shfl_xor(n.qmin, o));
    n.qmax = max(n.qmax, __shfl_xor(n.qmax, o));
    n.tmin = min(n.tmin, __shfl_xor(n.tmin, o));
    n.tmax = max(n.tmax, __shfl_xor(n.tmax, o));
  }
  if (!on) return;
  n.qmin = __builtin_amdgcn_readfirstlane(n.qmin);
  n.qmax = __builtin_amdgcn_readfirstlane(n.qmax);
  n.tmin = __builtin_amdgcn_readfirstlane(n.tmin);
  n.tmax = __builtin_amdgcn_readfirstlane(n.tmax);
  const float d = ddms_cell(lds, qr, tr, len1, len2, n);
  if (d != 0.0f) {
    const int64_t at = (int64_t)(row0 + r) * ldsc + c0 + c;
    scores[at] = scores[at] + d;
    mods[at] = mods[at] + fmaf(-CTH_DDMSSHIFT, CTH_DDMSWGT, d);
  }
}

// The score matrices without the DDMS term.  A workgroup covers a tile of
// query rows (every fourth row per wavefront) of 64 template columns, each
// lane holding its column in registers: frequencies, denominators and their
// reciprocals, context vector (128 VGPRs, 4 wavefronts per SIMD).  A row's
// values are uniform and come by scalar loads from the query's record
// (k_query_records).
//
// Bound by VALU issue: ~205 instructions a row, of which a third find a partner (a
// scalar operand keeps an instruction from issuing with another wavefront's); 97%
// of its cycles issue (profiles/k_dp_pmc.txt).
// With the rows staged in LDS and the frequencies and context vectors there
// too, the LDS returned ~250 cycles of data per row and wavefront, four of
// which share it: 2.7e9 cells took 22.0 ms, this form in 64-row tiles 20.5,
// in tiles of the whole query 17.9, with the scalar loads a part ahead 15.2,
// and with all of a column's and the table's loads under way before the first
// is waited for 14.2 (4 B + 4 B written per cell: 4.8 ms at the rate of a
// large copy).  The context-vector products on the matrix cores
// (v_mfma_f32_16x16x1, the same fma chain bit for bit) take as many VALU
// instructions for 16 of a wavefront's ~24 rows as they save: 14.9.
// Rows of a tile: the whole query up to kPlainRowsMax, so that the column's
// setup (20 divisions, the loads) is paid once, unless the launch would have
// fewer than kPlainFill workgroups; then shorter tiles, at least 16 rows.
constexpr int kProdPitch = 40;  // of a column's product operands, in entries
constexpr int kPlainRowsMax = 256, kPlainRowsMin = 16, kPlainFill = 2048;

// a factor of a log-odds numerator the quotient correction below admits:
// +0 or [2^-32, 2], compared on the bit pattern
__device__ __forceinline__ bool in_quot_range(float v) {
  const uint32_t b = __builtin_bit_cast(uint32_t, v);
  return b == 0u || b - 0x2F800000u <= 0x10800000u;
}

// A query position's values as the plain kernel reads them
struct query_record {
  float trg[CTH_NAA];
  float cv[CTH_NCV];
  float normk;         // squared norm + 1 + kappa
  float prior;
  float ss[CTH_NSS];
  float ssh;           // last SS probability + 0.1
  int32_t ssrow[CTH_NSS];  // rows of the square SS table, as byte offsets
  int32_t quot;        // frequencies within in_quot_range
  float pad[64 - CTH_NAA - CTH_NCV - 10];
};
static_assert(sizeof(query_record) == 256, "query record");
// the two parts of a record as scalar loads fetch them
typedef float sv16 __attribute__((ext_vector_type(16), aligned(4)));
typedef float sv8 __attribute__((ext_vector_type(8), aligned(4)));
typedef float sv4 __attribute__((ext_vector_type(4), aligned(4)));
struct row_trg {
  sv16 a;
  sv4 b;
  __device__ __forceinline__ float at(int k) const { return k < 16 ? a[k] : b[k - 16]; }
};
struct row_tail {
  sv16 a;  // context vector 0..15
  sv8 b;   // 16..18, normk, prior, ss 0..2
  sv4 c;   // ssh, ssrow 0..2
  __device__ __forceinline__ float cv(int k) const { return k < 16 ? a[k] : b[k - 16]; }
  __device__ __forceinline__ float normk() const { return b[3]; }
  __device__ __forceinline__ float prior() const { return b[4]; }
  __device__ __forceinline__ float ss(int k) const { return b[5 + k]; }
  __device__ __forceinline__ float ssh() const { return c[0]; }
  __device__ __forceinline__ uint32_t ssrow(int k) const {
    const float v = c[1 + k];
    return __builtin_bit_cast(uint32_t, v);
  }
};
static_assert(offsetof(query_record, cv) == 80 && offsetof(query_record, normk) == 156 &&
                  offsetof(query_record, prior) == 160 && offsetof(query_record, ss) == 164 &&
                  offsetof(query_record, ssh) == 176 && offsetof(query_record, ssrow) == 180,
              "query record parts");

__global__ __launch_bounds__(256) void k_query_records(cth_dpset q, const cth_tables* __restrict__ tabs,
                                                       query_record* __restrict__ rec) {
  const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (i >= q.npos) return;
  query_record r;
  r.quot = 1;
  for (int a = 0; a < CTH_NAA; a++) {
    r.trg[a] = q.trg[a * q.ld + i];
    r.quot &= in_quot_range(r.trg[a]) ? 1 : 0;
  }
  for (int k = 0; k < CTH_NCV; k++) r.cv[k] = q.cv[k * q.ld + i];
  r.normk = q.cvnorm2[i] + 1.0f + tabs->cvkappa0inv;
  r.prior = q.cvprior[i];
  for (int k = 0; k < CTH_NSS; k++) {
    r.ss[k] = q.ss[k * q.ld + i];
    r.ssrow[k] = (k * 10 + (int)(r.ss[k] * 9.999f)) * 30 * (int)sizeof(float);
  }
  r.ssh = r.ss[CTH_NSS - 1] + 0.1f;
  for (float& v : r.pad) v = 0.0f;
  rec[i] = r;
}

// kBatch: as k_score_ddms's (ytab[blockIdx.y] a tile of `tile` rows, at most
// kPlainRowsMax).
// kPrec 1, 2: the log-odds sum from the BF16 / FP16 product on the matrix
// cores, 0: in FP32.
//
// The product's tile is 32 of the wavefront's rows x its 64 columns, two
// 32 x 32 blocks; it goes through the wavefront's own LDS block to one column
// per lane.  Against a product of its own kernel before, whose 64 x 64 tiles divide
// each column's frequencies again and whose logarithms are written and read
// back (4 B + 4 B a cell), the score stage of 142 Mcells takes 0.51 ms instead
// of 0.76.
template <int kPrec, bool kBatch>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_score_plain(
    cth_dpset q, const query_record* __restrict__ rec, int qp, cth_dpset db, int64_t col0, int ncols, int64_t ldsc,
    const cth_tables* __restrict__ tabs, float* __restrict__ scores, float* __restrict__ mods, int tile,
    const cth_bytile* __restrict__ ytab, const cth_bquery* __restrict__ bq) {
  // the SS table square (30 x 30, symmetric: entry r*30+c is ss_lookup(r, c)),
  // so that a lookup is one index add; a row's lookups fall into ten
  // neighbouring words, so the reads have no bank conflicts
  __shared__ float Lsq[30 * 30];
  __shared__ float Lcv[CTH_CVMAXCARD];
  // the product's column operands (rows of 80 bytes: aligned 16-byte reads,
  // spread over the banks), then each wavefront's 32 x 64 sums
  __shared__ __align__(16) float Lp[kPrec ? 4 * 32 * 64 : 1];
  const int tid = threadIdx.x;
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  int row0 = blockIdx.y * tile;
  if constexpr (kBatch) {
    const cth_bytile t = ytab[blockIdx.y];
    const cth_bquery Q = bq[t.b];
    qp = Q.qp;
    row0 = t.row0;
    scores += Q.off;
    mods += Q.off;
  }
  const int row1 = min(q.len[qp], row0 + tile);
  const int64_t q0 = q.dist[qp];
  const int col = blockIdx.x * kCols + lane;
  const bool colin = col < ncols;
  // the tables, stored after the column's loads are on their way
  float sqv[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int e = min(tid + 256 * k, 30 * 30 - 1);
    sqv[k] = ss_lookup(tabs->ss, e / 30, e % 30);
  }

  // this lane's template column (lanes past the last column read column 0
  // and leave after the staging): frequencies and the log-odds denominators
  // (CuBatchScoreMatrix_Init.cu:129-144,173-185: 0.5 (bq(a) + bt(a)), per
  // query and template profile), SS probabilities and their table columns,
  // context vector, its prior and squared norm.
  const int64_t tj = col0 + (colin ? col : 0);
  const int tp = db.pro[tj];
  const float kap = tabs->cvkappa0inv, cvpow = tabs->cvpowernu0, cvcterm = tabs->cvcterm;
  const int card = tabs->cvcard, cvshift = tabs->cvshift;
  const float key0 = tabs->cvkeys[0], key1 = tabs->cvkeys[card - 1];
  float ts[CTH_NSS];
  uint32_t tc[CTH_NSS];
#pragma unroll
  for (int j = 0; j < CTH_NSS; j++) {
    ts[j] = db.ss[j * db.ld + tj];
    tc[j] = 4u * (uint32_t)(j * 10 + (int)(ts[j] * 9.999f));
  }
  const float tsh = ts[CTH_NSS - 1] + 0.1f;
  const float tn = db.cvnorm2[tj] + 1.0f + kap;
  const float tprior = db.cvprior[tj];
  float tcv[CTH_NCV];
#pragma unroll
  for (int i = 0; i < CTH_NCV; i++) tcv[i] = db.cv[i * db.ld + tj];
#pragma unroll
  for (int k = 0; k < 4; k++)
    if (tid + 256 * k < 30 * 30) Lsq[tid + 256 * k] = sqv[k];
  for (int k = tid; k < tabs->cvcard; k += 256) Lcv[k] = tabs->cvvals[k];
  // The log-odds quotients num / den[a] by Markstein's correction: with
  // y = RN(1 / den) (an IEEE division, once per lane), q0 = RN(num y),
  // r = fma(-den, q0, num) (exact) and q = RN(q0 + r y) equal RN(num / den)
  // when no step underflows or overflows (P. Markstein, IBM J. Res. Dev.
  // 34:111-119, 1990): here when den lies in [2^-30, 2^30] and both factors
  // of num are 0 or in [2^-32, 2].  A wavefront whose columns or whose tile's
  // rows have an operand outside those ranges divides (quot).
  float tf[CTH_NAA], den[CTH_NAA], y[CTH_NAA];
  bool quot = true;
  // Whether every row of the tile is within the ranges: its rows' flags, one a
  // lane, under way with the column's loads and looked at by all 64 lanes before
  // those past the last column leave.  (Loaded when they are looked at, 1.9%
  // more of a launch of 32-row tiles.  The product does not ask, but the loads
  // bring the rows' records near: without them 0.51 ms instead of 0.48 for 142
  // Mcells.)
  int rowquot[kPlainRowsMax / 64];
#pragma unroll
  for (int k = 0; k < kPlainRowsMax / 64; k++)
    rowquot[k] = row0 + 64 * k < row1 ? rec[q0 + min(row0 + 64 * k + lane, row1 - 1)].quot : 1;
  auto rows_in_range = [&] {
#pragma unroll
    for (int k = 0; k < kPlainRowsMax / 64; k++) quot = quot && __builtin_amdgcn_ballot_w64(rowquot[k] == 0) == 0;
  };
  v8s pb[2][2];  // the product's column operands of this lane
  if constexpr (!kPrec) {
    // all loads first: left to itself the compiler loads an operand and waits
    // for it 20 times
    float bt[CTH_NAA], bqa[CTH_NAA];
#pragma unroll
    for (int a = 0; a < CTH_NAA; a++) {
      tf[a] = db.trg[a * db.ld + tj];
      bt[a] = db.bkg[tp * CTH_NAA + a];
      bqa[a] = q.bkg[qp * CTH_NAA + a];
    }
#pragma unroll
    for (int a = 0; a < CTH_NAA; a++) asm volatile("" : "+v"(tf[a]), "+v"(bt[a]), "+s"(bqa[a]));
    bool lane_ok = true;
#pragma unroll
    for (int a = 0; a < CTH_NAA; a++) {
      den[a] = 0.5f * (bqa[a] + bt[a]);
      y[a] = 1.0f / den[a];
      lane_ok &= in_quot_range(tf[a]) && __builtin_bit_cast(uint32_t, den[a]) - 0x30800000u <= 0x1E000000u;
    }
    quot = __builtin_amdgcn_ballot_w64(!lane_ok) == 0;
    __syncthreads();
    rows_in_range();
    if (!colin) return;
  } else {
    // each wavefront divides 5 of the 20 frequencies of the 64 columns and
    // clears 3 of the 12 entries that pad K to 32.  Lanes past the last
    // column stay: the product takes all 64.
    uint16_t* const B = reinterpret_cast<uint16_t*>(Lp) + lane * kProdPitch;
    for (int k = 5 * w; k < 5 * w + 5; k++)
      B[k] = mfma_operand<kPrec>(db.trg[k * db.ld + tj] /
                                 (0.5f * (q.bkg[qp * CTH_NAA + k] + db.bkg[tp * CTH_NAA + k])));
    for (int k = CTH_NAA + 3 * w; k < CTH_NAA + 3 * w + 3; k++) B[k] = 0;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
        pb[c][kb] = *reinterpret_cast<const v8s*>(reinterpret_cast<const uint16_t*>(Lp) +
                                                  (32 * c + (lane & 31)) * kProdPitch + 16 * kb + 8 * (lane >> 5));
    __syncthreads();
    rows_in_range();
  }
  const char* const sq = reinterpret_cast<const char*>(Lsq);

  // the sums of 32 of the wavefront's rows from `row` on (rows past the tile's
  // end repeat the last)
  float* const sums = &Lp[kPrec ? w * 32 * 64 : 0];
  auto product = [&](int row) {
    const float* const f = rec[q0 + min(row + 4 * (lane & 31), row1 - 1)].trg;
    const bool low = lane < 32;
    v8s a0, a1;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      a0[k] = (short)mfma_operand<kPrec>(f[(low ? 0 : 8) + k]);
      a1[k] = k < 4 && low ? (short)mfma_operand<kPrec>(f[16 + (k & 3)]) : 0;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int c = 0; c < 2; c++) {
      v16f acc = {};
      acc = mfma<kPrec>(a0, pb[c][0], acc);
      acc = mfma<kPrec>(a1, pb[c][1], acc);
#pragma unroll
      for (int r = 0; r < 16; r++) sums[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * 64 + 32 * c + (lane & 31)] = acc[r];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };

  // Rows in straight-line code, interleaved over the wavefronts so that
  // partial tiles stay balanced.  The row's values are scalar loads issued
  // well ahead of their use: the second part of its record while its log-odds
  // are summed, the frequencies of the next row while this one's SS and
  // context terms are.  The empty asm statements are where each part is
  // waited for; without them the compiler moves the loads to their uses and
  // waits four times per row.  The rare cells whose logarithms are not those
  // of positive normal numbers make the wavefront take them again with the
  // general function.  kQuot: log-odds by the quotient correction.
  auto rows = [&](auto kQuot) {
    int row = row0 + w;
    if (row >= row1) return;
    row_trg F{};
    auto load_trg = [&](int r) {
      if constexpr (!kPrec) {
        const query_record& Q = rec[q0 + r];
        F.a = *reinterpret_cast<const sv16*>(&Q.trg[0]);
        F.b = *reinterpret_cast<const sv4*>(&Q.trg[16]);
      }
    };
    load_trg(row);
    if constexpr (!kPrec) asm volatile("" : "+s"(F.a), "+s"(F.b));
    for (; row < row1; row += 4) {
      if constexpr (kPrec != 0) {
        if (((row - row0) & 127) < 4) product(row);
      }
      const query_record& Q = rec[q0 + row];
      float* const out = scores + row * ldsc + col;
      row_tail R;
      R.a = *reinterpret_cast<const sv16*>(&Q.cv[0]);
      R.b = *reinterpret_cast<const sv8*>(&Q.cv[16]);
      R.c = *reinterpret_cast<const sv4*>(&Q.ssh);
      __builtin_amdgcn_sched_barrier(0);
      float s = 0.0f;
      if constexpr (kPrec != 0) {
        s = sums[((row - row0) >> 2 & 31) * 64 + lane];
      } else {
#pragma unroll
        for (int a = 0; a < CTH_NAA; a++) {
          const float num = F.at(a) * tf[a];
          if constexpr (kQuot.value) {
            const float q0 = num * y[a];
            s = s + fmaf(fmaf(-den[a], q0, num), y[a], q0);
          } else {
            s = s + num / den[a];
          }
        }
      }
      asm volatile("" : "+s"(R.a), "+s"(R.b), "+s"(R.c));
      load_trg(min(row + 4, row1 - 1));
      __builtin_amdgcn_sched_barrier(0);
      // SS (CuBatchScoreMatrix_ssss.cuh:64-116)
      float sss = 0.0f;
#pragma unroll
      for (int i = 0; i < CTH_NSS; i++) {
#pragma unroll
        for (int j = 0; j < CTH_NSS; j++)
          sss = fmaf(R.ss(i) * ts[j], *reinterpret_cast<const float*>(sq + (R.ssrow(i) + tc[j])), sss);
      }
      {
        float v = fmaf(R.ssh() * tsh, 0.1111111f, sss);
        v -= CTH_SSSHIFT;
        v *= CTH_SSSWGT;
        sss = -99.f < sss ? v : sss;
      }
      // CVS (CuBatchScoreMatrix_cvs2s.cuh:80-113)
      float cvs = 0.0f;
#pragma unroll
      for (int i = 0; i < CTH_NCV; i++) cvs = fmaf(R.cv(i), tcv[i], cvs);
      cvs += kap;
      cvs = fmaf(-cvs, cvs, R.normk() * tn);
      const float prior = R.prior();
      if constexpr (!kPrec) asm volatile("" : "+s"(F.a), "+s"(F.b));
      const bool odd = !cth_logf_ordinary(cvs) || !cth_logf_ordinary(s);
      float lc = cth_logf_core(cvs);
      float ls = cth_logf_core(s);
      if (__builtin_amdgcn_ballot_w64(odd) != 0) {
        lc = cth_logf(cvs);
        ls = cth_logf(s);
      }
      s = ls - CTH_INITSHIFT;
      cvs = fmaf(cvpow, lc, cvcterm) - prior - tprior;
      int at = cvshift + (int)rintf(2.0f * cvs);
      at = key1 <= cvs ? card - 1 : at;
      at = cvs <= key0 ? 0 : at;
      cvs = Lcv[at] * CTH_CVSWGT;
      const float sc = sss + cvs;
      if (!kPrec || colin) {
        *out = s + sc;
        mods[row * ldsc + col] = fmaf(-CTH_CVSSHIFT, CTH_CVSWGT, sc);
      }
    }
  };
  if (quot) rows(std::true_type{});
  else rows(std::false_type{});
}

__global__ void k_selftest_logf(int* bad) {
  // every significand at a few exponents, with lanes of one exponent together
  const uint32_t m = blockIdx.x * 256 + threadIdx.x;
  const int exps[] = {1, 64, 126, 127, 128, 200, 254};
  for (int e : exps) {
    const float x = __builtin_bit_cast(float, (uint32_t)e << 23 | m);
    if (__builtin_bit_cast(uint32_t, cth_logf_dev(x)) != __builtin_bit_cast(uint32_t, cth_logf(x))) atomicAdd(bad, 1);
  }
  // arguments outside the fast path, alone and beside ordinary ones
  const uint32_t odd[] = {0u, 1u, 0x007fffffu, 0x7f800000u, 0x80000000u, 0xbf800000u, 0x3f800000u | m};
  const float x = __builtin_bit_cast(float, odd[m % 7]);
  if (__builtin_bit_cast(uint32_t, cth_logf_dev(x)) != __builtin_bit_cast(uint32_t, cth_logf(x))) atomicAdd(bad, 1);
}

}  // namespace

// Rows of one tile of k_score_plain over `rows` query rows (all queries of a
// batch) and ncols columns.  A batch with DDMS terms (ddms) runs both kernels
// over one table of tiles, so they are CTH_DDMS_TILE rows there, a multiple
// of kDRows; the plain kernel's share of its time is small.
extern "C" int cth_score_tile_rows(int ddms, int64_t rows, int64_t ncols) {
  if (ddms) return CTH_DDMS_TILE;
  const int64_t cols = (ncols + kCols - 1) / kCols;
  const int64_t fit = rows * cols / kPlainFill;  // rows per tile that leave kPlainFill workgroups
  return (int)std::max<int64_t>(kPlainRowsMin, std::min<int64_t>({(rows + 3) / 4 * 4, fit / 4 * 4, kPlainRowsMax}));
}
static_assert(CTH_DDMS_TILE <= kPlainRowsMax && kPlainRowsMax % 64 == 0, "rows whose flags a lane holds");
static_assert(CTH_DDMS_TILE % kDRows == 0 && kDRows >= CTH_SCORE_TILE_MIN && kPlainRowsMin >= CTH_SCORE_TILE_MIN,
              "row tiles");

// Columns of the distance-match launch that starts at column c: it takes 32
// work-items a column, and a grid dimension of 2^32 work-items or more is
// refused.  (A search's chunks have at most 6M columns, so they take one
// launch; a launch of 8M leaves its tail behind by far.)
static int ddms_slice(int ncols, int c) { return std::min(ncols - c, 1 << 23); }

template <bool kBatch>
static int launch_ddms(const cth_dpset* q, int qp, const cth_dpset* db, int64_t col0, int ncols, int64_t ldsc,
                       const cth_tables* dtabs, float* scores, float* mods, const int32_t* qoff, int ytiles,
                       const cth_bytile* ytab, int ysplit, const cth_bquery* bq, hipStream_t st) {
  for (int c = 0, n; c < ncols; c += n) {
    n = ddms_slice(ncols, c);
    hipLaunchKernelGGL(k_score_ddms<kBatch>, dim3((n + kDColsMin - 1) / kDColsMin, ytiles), dim3(kDThreads), 0, st, *q,
                       qp, *db, col0 + c, n, ldsc, dtabs, scores + c, mods + c, qoff, ytab, ysplit, bq);
    CTH_HIP_CHECK(hipGetLastError());
  }
  return 0;
}

// Host check of the launches over ncols columns: the largest grid's work-items,
// and the columns that all of them cover.
extern "C" void cth_selftest_ddms_launches(int ncols, uint64_t out[2]) {
  out[0] = out[1] = 0;
  for (int c = 0, n; c < ncols; c += n) {
    n = ddms_slice(ncols, c);
    out[0] = std::max<uint64_t>(out[0], (uint64_t)((n + kDColsMin - 1) / kDColsMin) * kDThreads);
    out[1] += (uint64_t)n;
  }
}

// Launch the score stage for query profile qp against template positions
// [col0, col0+ncols) of db; outputs are [Lq][ldsc].
// contraction 0: the FP32 log-odds term of the reference; 1 / 2: the term
// from the BF16 / FP16 matrix-core product.  ddms 0: no cell can have a DDMS
// term (the query's or every template's lists are shorter than DSTSEGM).
// qrec: the query set's records (cth_make_query_records).
extern "C" int cth_launch_score(const cth_dpset* q, const int32_t* qoff, const float* qrec, int qp, const cth_dpset* db, int64_t col0,
                                int ncols, int64_t ldsc, const cth_tables* dtabs, int lq, float* scores, float* mods,
                                int contraction, int ddms, hipStream_t st) {
  if (ncols <= 0 || lq <= 0) return 0;
  if (!qoff || !qrec) { cth_set_error("score: query distance offsets or records not built"); return -1; }
  if (ldsc < ncols) { cth_set_error("score: ldsc %lld < ncols %d", (long long)ldsc, ncols); return -1; }
  if (contraction < 0 || contraction > 2) {
    cth_set_error("score: contraction %d (0 FP32, 1 BF16, 2 FP16)", contraction);
    return -1;
  }
  const query_record* const rec = reinterpret_cast<const query_record*>(qrec);
  const int tile = cth_score_tile_rows(0, lq, ncols);
  const dim3 pgrid((ncols + kCols - 1) / kCols, (lq + tile - 1) / tile);
  if (contraction == 1) {
    hipLaunchKernelGGL((k_score_plain<1, false>), pgrid, dim3(256), 0, st, *q, rec, qp, *db, col0, ncols, ldsc,
                       dtabs, scores, mods, tile, nullptr, nullptr);
  } else if (contraction == 2) {
    hipLaunchKernelGGL((k_score_plain<2, false>), pgrid, dim3(256), 0, st, *q, rec, qp, *db, col0, ncols, ldsc,
                       dtabs, scores, mods, tile, nullptr, nullptr);
  } else {
    hipLaunchKernelGGL((k_score_plain<0, false>), pgrid, dim3(256), 0, st, *q, rec, qp, *db, col0, ncols, ldsc,
                       dtabs, scores, mods, tile, nullptr, nullptr);
  }
  CTH_HIP_CHECK(hipGetLastError());
  if (!ddms) return 0;
  return launch_ddms<false>(q, qp, db, col0, ncols, ldsc, dtabs, scores, mods, qoff, (lq + kDRows - 1) / kDRows,
                            nullptr, 1, nullptr, st);
}

// The score stage of a batch of queries: nytiles row tiles (ytab: query of
// the batch and first row, `tile` rows each, as cth_score_tile_rows gives
// them) against the whole resident database (ncols positions from column 0);
// each query's scores and modular scores at its offset (bq[].off, row stride
// ldsc); ddms 0 as in cth_launch_score.
extern "C" int cth_launch_score_batch(const cth_dpset* q, const int32_t* qoff, const float* qrec, const cth_dpset* db,
                                      int ncols,
                                      int64_t ldsc, const cth_tables* dtabs, const cth_bytile* ytab, int nytiles,
                                      const cth_bquery* bq, float* scores, float* mods, int ddms, int tile, hipStream_t st) {
  if (ncols <= 0 || nytiles <= 0) return 0;
  if (!qoff || !qrec) { cth_set_error("score batch: query distance offsets or records not built"); return -1; }
  if (ldsc < ncols) { cth_set_error("score batch: ldsc %lld < ncols %d", (long long)ldsc, ncols); return -1; }
  const int ysplit = ddms ? tile / kDRows : 1;
  if (tile < 1 || tile > kPlainRowsMax || (ddms && tile % kDRows)) {
    cth_set_error("score batch: row tiles of %d", tile);
    return -1;
  }
  if ((int64_t)nytiles * ysplit > 65535) { cth_set_error("score batch: %d row tiles", nytiles); return -1; }
  hipLaunchKernelGGL((k_score_plain<0, true>), dim3((ncols + kCols - 1) / kCols, nytiles), dim3(256), 0, st, *q,
                     reinterpret_cast<const query_record*>(qrec), 0, *db, (int64_t)0, ncols, ldsc, dtabs, scores,
                     mods, tile, ytab, bq);
  CTH_HIP_CHECK(hipGetLastError());
  if (!ddms) return 0;
  return launch_ddms<true>(q, 0, db, 0, ncols, ldsc, dtabs, scores, mods, qoff, nytiles * ysplit, ytab, ysplit, bq, st);
}

// The records of an uploaded query set that the plain kernel reads (256 bytes
// per position), allocated here.
extern "C" int cth_make_query_records(const cth_dpset* q, const cth_tables* dtabs, float** rec) {
  *rec = nullptr;
  const int64_t n = q->npos > 0 ? q->npos : 1;
  CTH_HIP_CHECK(hipMalloc((void**)rec, (size_t)n * sizeof(query_record)));
  hipLaunchKernelGGL(k_query_records, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, *q, dtabs,
                     reinterpret_cast<query_record*>(*rec));
  CTH_HIP_CHECK(hipGetLastError());
  CTH_HIP_CHECK(hipStreamSynchronize(0));
  return 0;
}

// Device check of cth_logf_dev against cth_logf over all significands:
// *bad = number of differing results (0 expected).
extern "C" int cth_selftest_logf(int* bad) {
  int* d = nullptr;
  CTH_HIP_CHECK(hipMalloc((void**)&d, sizeof(int)));
  CTH_HIP_CHECK(hipMemset(d, 0, sizeof(int)));
  hipLaunchKernelGGL(k_selftest_logf, dim3((1 << 23) / 256), dim3(256), 0, 0, d);
  const bool ok = hipGetLastError() == hipSuccess && hipMemcpy(bad, d, sizeof(int), hipMemcpyDeviceToHost) == hipSuccess;
  (void)hipFree(d);
  if (!ok) { cth_set_error("selftest_logf: launch or copy failed"); return -1; }
  return 0;
}
