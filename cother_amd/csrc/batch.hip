// batch.hip: the batched search -- many queries against the resident
// database in one pass of fused, persistent launches.
//
// cth_search runs the pipeline query by query and chunk by chunk.  For a batch
// of queries whose buffers fit the memory budget together, cth_search_batch
// instead runs every stage once over all (query, profile) pairs of the batch,
// and decides on the device which pairs go on to the next stage (as cth_search
// does for a chunk of the database, cth_chunk_finish below):
//   1. scores of every query of the batch (one launch, row tiles of all
//      queries);
//   2. phase-1 DP of every pair without traceback (persistent workgroups
//      taking pairs, longest first, from a device counter);
//   3. pairs over their query's score threshold -> list (device compaction);
//   4. DP with traceback and finalisation of the listed pairs (persistent);
//   5. passed pairs -> list; their statistics (histogram, then the parameters
//      and E-value; persistent);
//   6. pairs within their query's E-value threshold -> list; MAP forward,
//      backward, MAP DP and traceback of each in one persistent kernel;
//   7. the hit records of the listed pairs gathered into one array.
// The host uploads the batch's tables, launches the stages -- captured once
// as a HIP graph and replayed while the batch shape (sizes, buffers,
// options) stays the same; with stage timing requested they run eagerly
// between events -- and copies back the counts and the hit records: one
// synchronisation per batch.  Each pair's arithmetic is the per-query
// kernels' (the same device functions), so the hits equal cth_search's; the
// lists' order varies, the hit order is restored by the (log E-value,
// profile) sort.
//
// Covered: the FP32 contraction and databases of profiles of up to
// CTH_BATCH_LEN_MAX positions; other searches, and queries whose buffers alone
// exceed the budget, run through cth_search.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstring>
#include <numeric>
#include <vector>

#include "cth_batch.h"
#include "cth_ctx.h"
#include "cth_dp.h"
#include "cth_map.h"
#include "cth_search.h"
#include "cth_stats.h"

extern "C" int cth_launch_score_batch(const cth_dpset* q, const int32_t* qoff, const float* qrec, const cth_dpset* db,
                                      int ncols,
                                      int64_t ldsc, const cth_tables* dtabs, const cth_bytile* ytab, int nytiles,
                                      const cth_bquery* bq, float* scores, float* mods, int ddms, int tile, hipStream_t st);
extern "C" int cth_score_tile_rows(int ddms, int64_t rows, int64_t ncols);
extern "C" int cth_launch_dp_batch(const cth_dpset* q, const cth_dpset* db, const cth_bquery* bq,
                                   const cth_bpair* pairs, const int* list, const int* count, int n, int* next,
                                   int ltmax, int64_t ldsc, const float* scores, uint8_t* btck, cth_dpres* res,
                                   float* grow, int grid, int W, hipStream_t st);
extern "C" size_t cth_dp_batch_row_bytes(int grid, int ltmax);
extern "C" int cth_launch_stats_batch(const cth_dpset* q, const cth_dpset* db, const cth_bquery* bq,
                                      const cth_bpair* pairs, const int* list, const int* count, int64_t ldsc,
                                      const float* scores, const cth_dpres* dpres, int ssemodel, int lqmax, int* hist,
                                      int cap, double* out, int grid, hipStream_t st);
extern "C" int cth_launch_map_batch(const cth_dpset* q, const cth_dpset* db, const cth_bquery* bq,
                                    const cth_bpair* pairs, const int* list, const int* count, int ltmax, int lqmax,
                                    int64_t ldsc, const float* scores, const float* mods, float* post, uint8_t* btck,
                                    const double* stats, double* zrow, float minpp, char* alnout, int rowcap,
                                    cth_mapres* res, int grid, int W, int nsplit, float* back, hipStream_t st);
extern "C" int cth_map_split(int lq, int ltmax, int npairs);
extern "C" size_t cth_map_split_bytes(int lq, int ltmax, int n);

namespace {

enum { kCtrNext1 = 0, kCtrNext2, kCtrCand, kCtrPassed, kCtrHits, kNCtr = 8 };
// the device's clock where statistics begin and where the host takes over, as
// two 64-bit words behind a chunk's counters
enum { kMarkStats = 0, kMarkBack, kNMark };
static_assert(kNCtr % 2 == 0, "marks are aligned");

__global__ void k_batch_reset(int* ctr) {
  if (threadIdx.x < kNCtr) ctr[threadIdx.x] = 0;
}

// Pairs whose phase-1 maximum exceeds their query's score threshold go to
// the traceback pass (the only ones FinalizeDPPro traces back,
// cudp/CuBatchDP_final.cu:144); the others get an empty record.  On the way the
// statistics' histograms are cleared.
__global__ void k_select_cand(const cth_bquery* __restrict__ bq, const cth_bpair* __restrict__ pairs, int npairs,
                              cth_dpres* __restrict__ res, int* __restrict__ list, int* __restrict__ count,
                              int* __restrict__ hist, int nhist) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nhist; i += gridDim.x * blockDim.x) hist[i] = 0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < npairs; i += gridDim.x * blockDim.x) {
    cth_dpres r = res[i];
    if (bq[pairs[i].b].scorethld < r.maxsc) {
      list[atomicAdd(count, 1)] = i;
    } else {
      r.passed = 0; r.score = 0.0f; r.psts = 0; r.beg = 0;
      res[i] = r;
    }
  }
}

// passed pairs of the traceback pass -> list; that pass took the *ncand pairs of
// cand, or (null) all npairs.  mark: null, or where the clock goes
__global__ void k_select_passed(const cth_dpres* __restrict__ res, const int* __restrict__ cand,
                                const int* __restrict__ ncand, int npairs, int* __restrict__ list,
                                int* __restrict__ count, int64_t* __restrict__ mark) {
  if (mark && blockIdx.x == 0 && threadIdx.x == 0) mark[kMarkStats] = wall_clock64();
  const int n = cand ? *ncand : npairs;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
    const int i = cand ? cand[k] : k;
    if (res[i].passed) list[atomicAdd(count, 1)] = i;
  }
}

// passed pairs within their query's E-value threshold -> list (the profiles
// the MAP stage realigns, cumapdp/CuBatchMAPDP_fwd.cu:127-130); mark as above
__global__ void k_select_hits(const cth_bquery* __restrict__ bq, const cth_bpair* __restrict__ pairs,
                              const double* __restrict__ stats, const int* __restrict__ passed,
                              const int* __restrict__ npassed, int* __restrict__ list, int* __restrict__ count,
                              int64_t* __restrict__ mark) {
  if (mark && blockIdx.x == 0 && threadIdx.x == 0) mark[kMarkBack] = wall_clock64();
  const int n = *npassed;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
    const int i = passed[k];
    const float loge = (float)stats[(int64_t)i * CTH_STATS_NOUT + CTH_ST_LOGE];
    if (!(bq[pairs[i].b].logethld < loge)) list[atomicAdd(count, 1)] = i;
  }
}

// the hit records of the listed pairs, with the fields cth_search fills;
// alnoff holds the pair's slot in the list (its rows' place in alnout).  head:
// null, or where the counters and marks go in front of the records
__global__ void k_gather_hits(const cth_bquery* __restrict__ bq, const cth_bpair* __restrict__ pairs,
                              const cth_dpres* __restrict__ res, const double* __restrict__ stats,
                              const cth_mapres* __restrict__ mres, int do_map, const int* __restrict__ list,
                              const int* __restrict__ count, cth_hit* __restrict__ hits,
                              const int* __restrict__ ctr, int* __restrict__ head) {
  if (head && blockIdx.x == 0) {
    int64_t* const mark = reinterpret_cast<int64_t*>(head + kNCtr);
    if (threadIdx.x < kNCtr) head[threadIdx.x] = ctr[threadIdx.x];
    if (threadIdx.x == kMarkStats) mark[kMarkStats] = reinterpret_cast<const int64_t*>(ctr + kNCtr)[kMarkStats];
    if (threadIdx.x == kMarkBack) mark[kMarkBack] = wall_clock64();
  }
  const int n = *count;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
    const int i = list[k];
    const cth_bpair pr = pairs[i];
    const cth_dpres r = res[i];
    const double* s = stats + (int64_t)i * CTH_STATS_NOUT;
    cth_hit h;
    memset(&h, 0, sizeof h);
    h.query = bq[pr.b].qp;
    h.profile = pr.p;
    h.score = r.score;
    h.psts = r.psts;
    h.beg = r.beg;
    h.end = r.maxxy;
    h.logE = (float)s[CTH_ST_LOGE];
    h.logEpA = (float)s[CTH_ST_LOGEPA];
    h.lambda_est = (float)s[CTH_ST_LMBDEST];
    h.K_est = (float)s[CTH_ST_KEST];
    h.minsc = (float)s[CTH_ST_MIN];
    h.maxsc = (float)s[CTH_ST_MAX];
    h.expected = (float)s[CTH_ST_E];
    h.H = (float)s[CTH_ST_H];
    h.lambda = (float)s[CTH_ST_LMBD];
    h.K = (float)s[CTH_ST_K];
    if (do_map) {
      const cth_mapres m = mres[i];
      h.mapbeg = m.beg;
      h.mapend = m.end;
      h.idnts = m.idnts;
      h.ngaps = m.ngaps;
      h.alnlen = m.alnlen;
      h.pstvs_map = m.psts;
      h.mapscore = m.maxsc;
    }
    h.alnoff = (uint64_t)k;
    hits[k] = h;
  }
}

double now_ms() {
  return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }

// Pairs whose histograms k_hist_batch splits over workgroups: with more there
// is a workgroup for each anyway.
constexpr int kHistCap = 512;
int hist_ints(int npairs) { return std::min(npairs, kHistCap) * 641; }

// FNV-1a over the bytes of a plain struct
uint64_t fnv(const void* p, size_t n) {
  uint64_t h = 1469598103934665603ull;
  for (size_t k = 0; k < n; k++) h = (h ^ ((const uint8_t*)p)[k]) * 1099511628211ull;
  return h;
}

// The device layout of one batch: cell buffers (per query [Lq][ldsc], at the
// queries' offsets) and the small tables, records, lists and counters.
struct batch_layout {
  // cells
  float* scores; float* mods; float* post; uint8_t* btck;
  // small
  cth_bquery* bq; cth_bytile* ytab; cth_bpair* pairs; cth_dpres* res; double* stats; cth_mapres* mres;
  int* cand; int* passed; int* hitl; int* hist; int* ctr; double* zrow; cth_hit* hits; char* alnout; float* grow; float* back;
};

// The cell buffers in one piece: byte offsets of a batch of `cells` cells.  The
// sweeps read up to 8 floats to either side of their matrices: the traceback
// bytes come first, and a pad follows the last matrix.
struct cell_layout {
  size_t btck, scores, mods, post, bytes;
};
cell_layout lay_cells(size_t cells, bool map) {
  cell_layout C{};
  size_t o = 0;
  auto take = [&](size_t n) { const size_t at = o; o += up256(n); return at; };
  C.btck = take(cells);
  C.scores = take(4 * cells);
  C.mods = take(4 * cells);
  C.post = map ? take(4 * cells) : 0;
  C.bytes = o + CTH_SCORE_PAD * sizeof(float);
  return C;
}

// One batch's description on the host.
struct batch_plan {
  int q0, q1;                       // entries [q0,q1) of the query list
  std::vector<cth_bquery> bq;
  std::vector<cth_bytile> ytab;
  std::vector<cth_bpair> pairs;
  int64_t cells = 0;
  int lqmax = 0;
  int ddms = 1;                     // 0: no cell of the batch has a DDMS term
  int tile = 0;                     // rows of the score kernel's tiles
};

// Grids of the persistent launches (workgroups), wavefronts per pair of the two
// DP passes, and pairs that the MAP stage may take in its split form.
struct launch_shape {
  int dp_grid, dp_waves, trace_grid, small_grid, map_grid, trace_waves, map_split;
};

// One wavefront per pair where the pairs fill the chip (128,000 pairs of 99 x
// 231 positions: 6.8 ms, against 7.4 and 9.6 ms with two and three, whose
// wavefronts past a pair's last stripe wait), else one per stripe.  16
// workgroups per compute unit, more than are resident: those that start late
// take the pairs that are left (8 per unit: 7.2 ms, 10: 6.9, 12: 6.9, 16:
// 6.8).  Boundary rows in global memory are reserved per workgroup, so half
// as many then.  The traceback pass has few pairs: one wavefront per stripe.
//
// The boundary rows and the split form's backward values are not among the
// bytes that the budget counts: each takes an eighth of the batch's cell
// buffers at most (or the rows of one workgroup per compute unit, and 8 MB).
launch_shape choose_shape(int ncu, int npairs, int lqmax, int ltmax, size_t cellbytes, bool map) {
  launch_shape S;
  const int stripes = std::min(8, std::max(1, (lqmax + 63) / 64));
  S.dp_waves = npairs >= ncu * 8 ? 1 : stripes;
  S.trace_waves = stripes;
  S.dp_grid = ncu * (ltmax > CTH_DP_GLOBAL_FROM ? 8 : 16);
  S.small_grid = ncu * 4;
  S.trace_grid = S.small_grid;
  if (const size_t row = cth_dp_batch_row_bytes(1, ltmax)) {
    const int fit = (int)std::max<size_t>(ncu, std::min<size_t>(S.dp_grid, cellbytes / 8 / row));
    S.dp_grid = std::min(S.dp_grid, fit);
    S.trace_grid = std::min(S.trace_grid, fit);
  }
  S.map_grid = ncu * 16;  // (2000 pairs of 130 positions: 2.85 ms with four per unit, 2.1 with one per pair)
  S.map_split = map ? cth_map_split(lqmax, ltmax, npairs) : 0;
  if (S.map_split) {
    const size_t each = cth_map_split_bytes(lqmax, ltmax, 1);
    S.map_split = (int)std::min<size_t>(S.map_split, std::max((size_t)8 << 20, cellbytes / 8) / each);
  }
  return S;
}

int capture_or_launch(cth_ctx* c, const batch_plan& P, const batch_layout& L, const cth_search_opts* opt,
                      int64_t ldsc, int ltmax, int rowcap, const launch_shape& S, bool capture, bool timing) {
  const cth_devset& db = c->db;
  const int npairs = (int)P.pairs.size();
  const int ntiles = (int)P.ytab.size();
  hipStream_t st = c->st;
  hipGraph_t graph = nullptr;
  if (capture) CTH_HIP_CHECK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
  auto launches = [&]() -> int {
    if (timing) CTH_HIP_CHECK(hipEventRecord(c->ev[0], st));
    hipLaunchKernelGGL(k_batch_reset, dim3(1), dim3(64), 0, st, L.ctr);
    CTH_HIP_CHECK(hipGetLastError());
    if (cth_launch_score_batch(&c->q.d, c->q.ddoff, c->q.qrec, &db.d, (int)db.d.npos, ldsc, c->dtab, L.ytab, ntiles, L.bq,
                               L.scores, L.mods, P.ddms, P.tile, st))
      return -1;
    if (timing) CTH_HIP_CHECK(hipEventRecord(c->ev[1], st));
    if (cth_launch_dp_batch(&c->q.d, &db.d, L.bq, L.pairs, nullptr, nullptr, npairs, L.ctr + kCtrNext1, ltmax, ldsc,
                            L.scores, nullptr, L.res, L.grow, std::min(S.dp_grid, npairs),
                            S.dp_waves, st))
      return -1;
    const int sel_grid = std::max(1, std::min(1024, (npairs + 255) / 256));
    hipLaunchKernelGGL(k_select_cand, dim3(std::max(sel_grid, hist_ints(npairs) / 4096)), dim3(256), 0, st, L.bq, L.pairs, npairs, L.res, L.cand,
                       L.ctr + kCtrCand, L.hist, hist_ints(npairs));
    CTH_HIP_CHECK(hipGetLastError());
    if (cth_launch_dp_batch(&c->q.d, &db.d, L.bq, L.pairs, L.cand, L.ctr + kCtrCand, 0, L.ctr + kCtrNext2, ltmax,
                            ldsc, L.scores, L.btck, L.res, L.grow, std::min(S.trace_grid, npairs),
                            S.trace_waves, st))
      return -1;
    hipLaunchKernelGGL(k_select_passed, dim3(sel_grid), dim3(256), 0, st, L.res, L.cand, L.ctr + kCtrCand, npairs,
                       L.passed, L.ctr + kCtrPassed, nullptr);
    CTH_HIP_CHECK(hipGetLastError());
    if (timing) CTH_HIP_CHECK(hipEventRecord(c->ev[2], st));
    if (cth_launch_stats_batch(&c->q.d, &db.d, L.bq, L.pairs, L.passed, L.ctr + kCtrPassed, ldsc, L.scores, L.res,
                               opt->ssemodel, P.lqmax, L.hist, std::min(npairs, kHistCap), L.stats,
                               std::min(S.small_grid, npairs), st))
      return -1;
    hipLaunchKernelGGL(k_select_hits, dim3(sel_grid), dim3(256), 0, st, L.bq, L.pairs, L.stats, L.passed,
                       L.ctr + kCtrPassed, L.hitl, L.ctr + kCtrHits, nullptr);
    CTH_HIP_CHECK(hipGetLastError());
    if (timing) CTH_HIP_CHECK(hipEventRecord(c->ev[3], st));
    if (opt->do_map &&
        cth_launch_map_batch(&c->q.d, &db.d, L.bq, L.pairs, L.hitl, L.ctr + kCtrHits, ltmax, P.lqmax, ldsc, L.scores,
                             L.mods, L.post, L.btck, L.stats, L.zrow, opt->minpp > 0.0f ? opt->minpp : CTH_MINPP,
                             L.alnout, rowcap, L.mres, std::min(S.map_grid, npairs), S.trace_waves, S.map_split,
                             L.back, st))
      return -1;
    hipLaunchKernelGGL(k_gather_hits, dim3(sel_grid), dim3(256), 0, st, L.bq, L.pairs, L.res, L.stats, L.mres,
                       opt->do_map, L.hitl, L.ctr + kCtrHits, L.hits, nullptr, nullptr);
    CTH_HIP_CHECK(hipGetLastError());
    if (timing) CTH_HIP_CHECK(hipEventRecord(c->ev[4], st));
    return 0;
  };
  const int rc = launches();
  if (capture) {
    const hipError_t e = hipStreamEndCapture(st, &graph);
    if (rc) { if (graph) (void)hipGraphDestroy(graph); return -1; }
    if (e != hipSuccess) { cth_set_error("batch: graph capture: %s", hipGetErrorString(e)); return -1; }
    if (c->has_bgraph) { (void)hipGraphExecDestroy(c->bgraph); c->has_bgraph = 0; }
    const hipError_t ei = hipGraphInstantiate(&c->bgraph, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (ei != hipSuccess) { cth_set_error("batch: graph instantiation: %s", hipGetErrorString(ei)); return -1; }
    c->has_bgraph = 1;
    CTH_HIP_CHECK(hipGraphLaunch(c->bgraph, st));
  }
  return rc;
}

// A chunk's tables and counters, as the batched kernels read them: pair i is
// the chunk's profile i of query 0; and the statistics' histograms cleared.
__global__ void k_chunk_tables(cth_bquery Q, int p0, int np, cth_bquery* __restrict__ bq,
                               cth_bpair* __restrict__ pairs, int* __restrict__ ctr, int* __restrict__ hist,
                               int nhist) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  for (int k = i; k < nhist; k += gridDim.x * blockDim.x) hist[k] = 0;
  if (i < np) pairs[i] = cth_bpair{0, p0 + i};
  if (i < kNCtr) ctr[i] = 0;
  if (i == 0) *bq = Q;
}

// hit records that come back with the counters, and list entries
constexpr int kFirstHits = 128, kFirstList = 1024;
// what lies in front of either in device and in pinned memory
constexpr size_t kHead = 256;
// the MAP stage's workgroups per compute unit, as choose_shape's
constexpr int kChunkMapGrid = 16;

// A chunk's lists and records, by profile.
struct chunk_layout {
  cth_bquery* bq; cth_bpair* pairs; double* stats; cth_mapres* mres; int* cand; int* passed; int* hist;
  int* ctr; int* hitl;  // (the list follows the counters at kHead bytes)
  size_t bytes;
};
chunk_layout chunk_lay(int np, void* base) {
  chunk_layout L;
  size_t o = 0;
  auto take = [&](size_t n) { void* p = (uint8_t*)base + o; o += up256(n); return p; };
  L.bq = (cth_bquery*)take(sizeof(cth_bquery));
  L.pairs = (cth_bpair*)take(sizeof(cth_bpair) * np);
  L.stats = (double*)take(sizeof(double) * CTH_STATS_NOUT * np);
  L.mres = (cth_mapres*)take(sizeof(cth_mapres) * np);
  L.cand = (int*)take(sizeof(int) * np);
  L.passed = (int*)take(sizeof(int) * np);
  L.hist = (int*)take(sizeof(int) * hist_ints(np));
  L.ctr = (int*)take(kHead);
  L.hitl = (int*)take(sizeof(int) * np);
  L.bytes = o;
  return L;
}

// What the MAP stage and the hit records of n hits take, templates of up to
// ltmax positions: nsplit and grid as cth_launch_map_batch takes them.
struct hits_layout {
  int* head; cth_hit* hits;  // (the records follow the counters' copy at kHead bytes)
  double* zrow; float* back; char* alnout;
  size_t bytes;
};
hits_layout hits_lay(int lq, int ltmax, int n, bool rows, int nsplit, int grid, void* base) {
  hits_layout M;
  size_t o = 0;
  auto take = [&](size_t b) { void* p = (uint8_t*)base + o; o += up256(b); return p; };
  M.head = (int*)take(kHead);
  M.hits = (cth_hit*)take(sizeof(cth_hit) * n);
  M.zrow = (double*)take(sizeof(double) * std::max(grid, nsplit) * (size_t)lq);
  M.back = (float*)take(cth_map_split_bytes(lq, ltmax, nsplit));
  M.alnout = rows ? (char*)take((size_t)n * 5 * (size_t)(lq + ltmax)) : nullptr;
  M.bytes = o;
  return M;
}

}  // namespace

// The stages after a chunk's first DP pass, chosen and run on the device as
// the batched search does, where the host's choice of the next stage's profiles
// took four synchronisations with copies of all records between them (0.2-0.45
// ms of a search).
//
// The MAP stage's memory is sized for the hits, whose number and lengths come
// back first (kEarlyBytes: unless room for all profiles as hits is a few
// megabytes; then MAP follows at once, which saves the ~15 us between).  Known
// hits also need no grid for any number of them: of 4096 workgroups nearly all
// left at once, after 20 us.
int cth_chunk_finish(cth_ctx* c, const cth_chunk& k, const cth_search_opts* opt, int ncu, bool timing,
                     cth_chunk_hits& out) {
  constexpr size_t kEarlyBytes = (size_t)8 << 20;
  hipStream_t st = c->st;
  const cth_dpset *q = &c->q.d, *db = &c->db.d;
  out.hits.clear();
  out.rows.clear();
  out.rowcap = 0;
  out.npassed = 0;
  out.ms_stats = out.ms_map = 0.0f;
  out.ms_phase2 = 0.0;
  int clock_khz = 0;
  CTH_HIP_CHECK(hipDeviceGetAttribute(&clock_khz, hipDeviceAttributeWallClockRate, c->device));
  if (cth_ctx_reserve(c, &c->work, &c->cap_work, chunk_lay(k.np, nullptr).bytes)) return -1;
  const chunk_layout L = chunk_lay(k.np, c->work);
  constexpr size_t kPinned = kHead + std::max(sizeof(cth_hit) * kFirstHits, sizeof(int) * kFirstList);
  if (!c->h_pin) {
    CTH_HIP_CHECK(hipHostMalloc(&c->h_pin, kPinned));
    c->cap_pin = kPinned;
  }
  const int* const ctr = (const int*)c->h_pin;
  // The statistics begin where the host does not look: their time until it is
  // back is the device clock's.
  double back = 0.0;
  auto host_back = [&] {
    const int64_t* const mark = (const int64_t*)(ctr + kNCtr);
    back = now_ms();
    if (clock_khz > 0) back -= (double)(mark[kMarkBack] - mark[kMarkStats]) / clock_khz;
  };
  cth_bquery Q{};
  Q.qp = k.qi;
  Q.lq = k.lq;
  Q.off = -k.col0;
  Q.scorethld = k.scorethld;
  Q.logethld = k.logethld;
  Q.sspace = k.sspace;
  const int W = std::min(8, std::max(1, (k.lq + 63) / 64));
  const int grid = std::min(4 * ncu, k.np), sel = std::max(1, std::min(1024, (k.np + 255) / 256));
  const int nhist = hist_ints(k.np);
  hipLaunchKernelGGL(k_chunk_tables, dim3(std::max((k.np + 255) / 256, nhist / 4096)), dim3(256), 0, st, Q, k.p0, k.np,
                     L.bq, L.pairs, L.ctr, L.hist, nhist);
  CTH_HIP_CHECK(hipGetLastError());
  if (!k.traced) {
    hipLaunchKernelGGL(k_select_cand, dim3(sel), dim3(256), 0, st, L.bq, L.pairs, k.np, k.res, L.cand,
                       L.ctr + kCtrCand, nullptr, 0);
    CTH_HIP_CHECK(hipGetLastError());
    if (cth_launch_dp_batch(q, db, L.bq, L.pairs, L.cand, L.ctr + kCtrCand, 0, L.ctr + kCtrNext2, k.ltmax, k.ldsc,
                            k.scores, k.btck, k.res, nullptr, grid, W, st))
      return -1;
  }
  hipLaunchKernelGGL(k_select_passed, dim3(sel), dim3(256), 0, st, k.res, k.traced ? nullptr : L.cand,
                     L.ctr + kCtrCand, k.np, L.passed, L.ctr + kCtrPassed, (int64_t*)(L.ctr + kNCtr));
  CTH_HIP_CHECK(hipGetLastError());
  if (timing) CTH_HIP_CHECK(hipEventRecord(c->ev[2], st));
  if (cth_launch_stats_batch(q, db, L.bq, L.pairs, L.passed, L.ctr + kCtrPassed, k.ldsc, k.scores, k.res,
                             opt->ssemodel, k.lq, L.hist, std::min(k.np, kHistCap), L.stats, grid, st))
    return -1;
  hipLaunchKernelGGL(k_select_hits, dim3(sel), dim3(256), 0, st, L.bq, L.pairs, L.stats, L.passed,
                     L.ctr + kCtrPassed, L.hitl, L.ctr + kCtrHits, (int64_t*)(L.ctr + kNCtr));
  CTH_HIP_CHECK(hipGetLastError());
  if (timing) CTH_HIP_CHECK(hipEventRecord(c->ev[3], st));
  // the posteriors, which mem_budget counts, while the device is at work (0.3 ms
  // for 0.9 GB, on a context's first search)
  if (opt->do_map && cth_ctx_reserve(c, (void**)&c->mapbuf, &c->cap_mapbuf,
                                     sizeof(float) * ((size_t)k.lq * (size_t)k.ldsc + 2 * CTH_SCORE_PAD)))
    return -1;
  // the MAP stage's shape for any number of hits
  int nhit = k.np, ltmax = k.ltmax;
  int nsplit = opt->do_map ? cth_map_split(k.lq, ltmax, nhit) : 0;
  int mapgrid = opt->do_map ? std::min(kChunkMapGrid * ncu, nhit) : 0;
  const bool early = hits_lay(k.lq, ltmax, nhit, k.rows, nsplit, mapgrid, nullptr).bytes <= kEarlyBytes;
  if (!early) {
    // or, where that takes much memory, for those there are
    const int first = std::min(k.np, kFirstList);
    CTH_HIP_CHECK(hipMemcpyAsync(c->h_pin, L.ctr, kHead + sizeof(int) * first, hipMemcpyDeviceToHost, st));
    CTH_HIP_CHECK(hipStreamSynchronize(st));
    if (timing) CTH_HIP_CHECK(hipEventElapsedTime(&out.ms_stats, c->ev[2], c->ev[3]));
    host_back();
    nhit = ctr[kCtrHits];
    out.npassed = ctr[kCtrPassed];
    if (!nhit) {
      out.ms_phase2 = now_ms() - back;
      return 0;
    }
    std::vector<int> list((size_t)nhit);
    memcpy(list.data(), (const uint8_t*)c->h_pin + kHead, sizeof(int) * std::min(nhit, first));
    if (nhit > first) {
      CTH_HIP_CHECK(hipMemcpyAsync(list.data() + first, L.hitl + first, sizeof(int) * (nhit - first),
                                   hipMemcpyDeviceToHost, st));
      CTH_HIP_CHECK(hipStreamSynchronize(st));
    }
    ltmax = 0;
    for (int i : list) ltmax = std::max(ltmax, c->db.h_len[k.p0 + i]);
    if (opt->do_map) {
      nsplit = cth_map_split(k.lq, ltmax, nhit) >= nhit ? nhit : 0;
      mapgrid = nsplit ? 0 : std::min(kChunkMapGrid * ncu, nhit);
    }
  }
  out.rowcap = k.lq + ltmax;
  if (cth_ctx_reserve(c, &c->mapwork, &c->cap_mapwork,
                      hits_lay(k.lq, ltmax, nhit, k.rows, nsplit, mapgrid, nullptr).bytes))
    return -1;
  const hits_layout M = hits_lay(k.lq, ltmax, nhit, k.rows, nsplit, mapgrid, c->mapwork);
  if (timing && !early) CTH_HIP_CHECK(hipEventRecord(c->ev[3], st));
  if (opt->do_map &&
      cth_launch_map_batch(q, db, L.bq, L.pairs, L.hitl, L.ctr + kCtrHits, ltmax, k.lq, k.ldsc, k.scores, k.mods,
                           c->mapbuf + CTH_SCORE_PAD, k.btck, L.stats, M.zrow,
                           opt->minpp > 0.0f ? opt->minpp : CTH_MINPP, M.alnout, out.rowcap, L.mres, mapgrid, W,
                           nsplit, M.back, st))
    return -1;
  hipLaunchKernelGGL(k_gather_hits, dim3(std::max(1, std::min(1024, (nhit + 255) / 256))), dim3(256), 0, st, L.bq,
                     L.pairs, k.res, L.stats, L.mres, opt->do_map, L.hitl, L.ctr + kCtrHits, M.hits, L.ctr, M.head);
  CTH_HIP_CHECK(hipGetLastError());
  if (timing) CTH_HIP_CHECK(hipEventRecord(c->ev[4], st));
  const int first = std::min(nhit, kFirstHits);
  CTH_HIP_CHECK(hipMemcpyAsync(c->h_pin, M.head, kHead + sizeof(cth_hit) * first, hipMemcpyDeviceToHost, st));
  CTH_HIP_CHECK(hipStreamSynchronize(st));
  if (timing) {
    if (early) CTH_HIP_CHECK(hipEventElapsedTime(&out.ms_stats, c->ev[2], c->ev[3]));
    CTH_HIP_CHECK(hipEventElapsedTime(&out.ms_map, c->ev[3], c->ev[4]));
  }
  if (early) host_back();
  const int nb = ctr[kCtrHits];
  out.npassed = ctr[kCtrPassed];
  out.hits.resize(nb);
  if (nb) memcpy(out.hits.data(), (const uint8_t*)c->h_pin + kHead, sizeof(cth_hit) * std::min(nb, first));
  if (nb > first)
    CTH_HIP_CHECK(hipMemcpyAsync(out.hits.data() + first, M.hits + first, sizeof(cth_hit) * (nb - first),
                                 hipMemcpyDeviceToHost, st));
  if (nb && M.alnout) {
    out.rows.resize((size_t)nb * 5 * out.rowcap);
    CTH_HIP_CHECK(hipMemcpyAsync(out.rows.data(), M.alnout, out.rows.size(), hipMemcpyDeviceToHost, st));
  }
  if (nb > first || !out.rows.empty()) CTH_HIP_CHECK(hipStreamSynchronize(st));
  std::sort(out.hits.begin(), out.hits.end(), [](const cth_hit& a, const cth_hit& b) { return a.profile < b.profile; });
  out.ms_phase2 = now_ms() - back;
  return 0;
}

namespace {

// the batched search over the queries ql[0..nq) (distinct indices), hits per
// query in list order; nhits[k] for query ql[k]
int search_batch_list(cth_ctx* c, const int* ql, int nq, const cth_search_opts* opt, cth_hit* hits, int maxhits,
                      int* nhits, cth_search_stats* stats) {
  CTH_HIP_CHECK(hipSetDevice(c->device));
  const cth_devset& db = c->db;
  const int nprof = db.d.nprof;
  const int64_t npos = db.d.npos;
  const int ltmax = nprof ? *std::max_element(db.h_len, db.h_len + nprof) : 0;
  cth_search_stats st{};
  // the batched form covers the FP32 contraction and profiles within its
  // limit; otherwise the queries run through cth_search
  if (opt->contraction != 0 || ltmax > CTH_BATCH_LEN_MAX || nprof == 0) {
    int nh = 0;
    uint64_t used = 0;
    for (int k = 0; k < nq; k++) {
      cth_search_opts o1 = *opt;
      if (opt->alnbuf) {
        o1.alnbuf = opt->alnbuf + used;
        o1.alncap = opt->alncap - used;
      }
      int n1 = 0;
      cth_search_stats s1{};
      if (cth_search(c, ql[k], ql[k] + 1, &o1, hits + nh, maxhits - nh, &n1, &s1)) return -1;
      for (int j = 0; j < n1; j++) {
        if (opt->alnbuf) hits[nh + j].alnoff += used;
        if (opt->alnbuf && opt->do_map) used += 5 * (uint64_t)hits[nh + j].alnlen;
      }
      if (nhits) nhits[k] = n1;
      nh += n1;
      st.cells += s1.cells; st.npassed += s1.npassed; st.nchunks += s1.nchunks; st.map_cells += s1.map_cells;
      st.ms_phase1 += s1.ms_phase1; st.ms_phase2 += s1.ms_phase2; st.ms_k_score += s1.ms_k_score;
      st.ms_k_dp += s1.ms_k_dp; st.ms_k_stats += s1.ms_k_stats; st.ms_k_map += s1.ms_k_map;
    }
    if (stats) *stats = st;
    return 0;
  }
  const uint64_t dbsize = opt->dbsize ? opt->dbsize : (uint64_t)npos;
  const uint64_t ndbent = opt->ndb ? opt->ndb : (uint64_t)nprof;
  const size_t budget = opt->mem_budget ? opt->mem_budget : ((size_t)64 << 30);
  const int64_t ldsc = (npos + 63) / 64 * 64;
  const size_t bytes_per_cell = opt->do_map ? 13 : 9;
  const bool timing = opt->timing != 0;
  if (timing && !c->has_ev) {
    for (int k = 0; k < 4; k++) CTH_HIP_CHECK(hipEventCreate(&c->ev[k]));
    c->has_ev = 1;
  }
  if (timing && c->nbev < 5) {
    CTH_HIP_CHECK(hipEventCreate(&c->ev[4]));
    c->nbev = 5;
  }
  int ncu = 0;
  CTH_HIP_CHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device));
  // profiles in decreasing length: the longest DPs start first
  std::vector<int> porder(nprof);
  std::iota(porder.begin(), porder.end(), 0);
  std::stable_sort(porder.begin(), porder.end(), [&](int a, int b) { return db.h_len[a] > db.h_len[b]; });

  int nh = 0;
  uint64_t alnused = 0;
  // batch-local index of each query of the current batch (for its hits)
  std::vector<int> local(c->q.d.nprof, -1);
  for (int qa = 0; qa < nq;) {
    // the batch: consecutive entries of the list whose buffers fit the
    // budget together
    batch_plan P;
    P.q0 = qa;
    size_t bytes = 0;
    int qb = qa;
    int tiles = 0;
    while (qb < nq) {
      const int lq = c->q.h_len[ql[qb]];
      const size_t qbytes = (size_t)lq * (size_t)ldsc * bytes_per_cell;
      // row tiles of its score kernels, the most any choice of them has
      const int qt = (lq + CTH_DDMS_TILE - 1) / CTH_DDMS_TILE * (CTH_DDMS_TILE / CTH_SCORE_TILE_MIN);
      if (qb > qa && (bytes + qbytes > budget || tiles + qt > 65535)) break;
      bytes += qbytes;
      tiles += qt;
      qb++;
    }
    P.q1 = qb;
    // a query whose buffers alone exceed the budget runs in chunks through
    // cth_search (its alignment rows after those already written)
    if (qb == qa + 1 && bytes > budget) {
      cth_search_opts o1 = *opt;
      if (opt->alnbuf) {
        o1.alnbuf = opt->alnbuf + alnused;
        o1.alncap = opt->alncap - alnused;
      }
      int n1 = 0;
      cth_search_stats s1{};
      if (cth_search(c, ql[qa], ql[qa] + 1, &o1, hits + nh, maxhits - nh, &n1, &s1)) return -1;
      for (int k = 0; k < n1; k++) {
        if (opt->alnbuf) hits[nh + k].alnoff += alnused;
        if (opt->alnbuf && opt->do_map) alnused += 5 * (uint64_t)hits[nh + k].alnlen;
      }
      if (nhits) nhits[qa] = n1;
      nh += n1;
      st.cells += s1.cells; st.npassed += s1.npassed; st.nchunks += s1.nchunks; st.map_cells += s1.map_cells;
      st.ms_phase1 += s1.ms_phase1; st.ms_phase2 += s1.ms_phase2; st.ms_k_score += s1.ms_k_score;
      st.ms_k_dp += s1.ms_k_dp; st.ms_k_stats += s1.ms_k_stats; st.ms_k_map += s1.ms_k_map;
      qa++;
      continue;
    }
    // no DDMS term in the batch when the database's or every query's
    // distance lists are shorter than DSTSEGM: the plain score kernel alone
    // and row tiles by its own rule
    P.ddms = 0;
    if (cth_devset_has_ddms(&db, 0, nprof))
      for (int k = P.q0; k < P.q1 && !P.ddms; k++) P.ddms = cth_devset_has_ddms(&c->q, ql[k], ql[k] + 1);
    int64_t allrows = 0;
    for (int k = P.q0; k < P.q1; k++) allrows += c->q.h_len[ql[k]];
    const int rows = P.tile = cth_score_tile_rows(P.ddms, allrows, npos);
    for (int k = P.q0; k < P.q1; k++) {
      const int qi = ql[k];
      local[qi] = k - P.q0;
      cth_bquery Q{};
      Q.qp = qi;
      Q.lq = c->q.h_len[qi];
      Q.off = P.cells;
      cth_query_thresholds(opt->eval, (uint64_t)Q.lq, dbsize, ndbent, &Q.scorethld, &Q.logethld, &Q.sspace);
      const int b = (int)P.bq.size();
      P.bq.push_back(Q);
      for (int r0 = 0; r0 < Q.lq; r0 += rows) P.ytab.push_back(cth_bytile{b, r0});
      P.cells += (int64_t)Q.lq * ldsc;
      P.lqmax = std::max(P.lqmax, Q.lq);
    }
    // pairs: longest DPs (query length x profile length) first, equal
    // sizes in query-then-profile order (a stable sort; counting sort on the
    // size where the sizes are small enough for a table, ~4x faster on the
    // host per batch of 128,000 pairs)
    {
      std::vector<cth_bpair> src;
      src.reserve((size_t)P.bq.size() * porder.size());
      int64_t maxsz = 0;
      for (int b = 0; b < (int)P.bq.size(); b++) {
        for (int p : porder) src.push_back(cth_bpair{b, p});
        if (!porder.empty()) maxsz = std::max(maxsz, (int64_t)P.bq[b].lq * db.h_len[porder[0]]);
      }
      auto size_of = [&](const cth_bpair& x) { return (int64_t)P.bq[x.b].lq * db.h_len[x.p]; };
      if (maxsz < (int64_t)1 << 22) {
        std::vector<int> at((size_t)maxsz + 2, 0);
        for (const cth_bpair& x : src) at[(size_t)(maxsz - size_of(x)) + 1]++;
        for (size_t k = 1; k < at.size(); k++) at[k] += at[k - 1];
        P.pairs.resize(src.size());
        for (const cth_bpair& x : src) P.pairs[at[(size_t)(maxsz - size_of(x))]++] = x;
      } else {
        std::stable_sort(src.begin(), src.end(),
                         [&](const cth_bpair& x, const cth_bpair& y) { return size_of(x) > size_of(y); });
        P.pairs.swap(src);
      }
    }
    const int npairs = (int)P.pairs.size();
    const int rowcap = P.lqmax + ltmax;
    const size_t alnbytes = opt->alnbuf && opt->do_map ? (size_t)npairs * 5 * (size_t)rowcap : 0;
    // device buffers
    const size_t cells = (size_t)P.cells;
    const cell_layout cell = lay_cells(cells, opt->do_map != 0);
    const int small_max = std::max(1, std::min(npairs, ncu * 32));
    const launch_shape S = choose_shape(ncu, npairs, P.lqmax, ltmax, cell.bytes, opt->do_map != 0);
    const size_t backbytes = cth_map_split_bytes(P.lqmax, ltmax, S.map_split);
    const size_t growbytes = cth_dp_batch_row_bytes(std::min(npairs, std::max(S.dp_grid, S.trace_grid)), ltmax);
    const size_t sbytes = up256(sizeof(cth_bquery) * P.bq.size()) + up256(sizeof(cth_bytile) * P.ytab.size()) +
                          up256(sizeof(cth_bpair) * npairs) + up256(sizeof(cth_dpres) * npairs) +
                          up256(sizeof(double) * CTH_STATS_NOUT * npairs) + up256(sizeof(cth_mapres) * npairs) +
                          3 * up256(sizeof(int) * npairs) + up256(sizeof(int) * kNCtr) +
                          up256(sizeof(int) * hist_ints(npairs)) + up256(sizeof(double) * (size_t)small_max * P.lqmax) + up256(sizeof(cth_hit) * npairs) +
                          up256(alnbytes) + up256(growbytes) + up256(backbytes);
    if (cth_ctx_reserve(c, &c->bcells, &c->cap_bcells, cell.bytes)) return -1;
    if (cth_ctx_reserve(c, &c->bsmall, &c->cap_bsmall, sbytes)) return -1;
    batch_layout L{};
    {
      uint8_t* const o = (uint8_t*)c->bcells;
      L.btck = o + cell.btck;
      L.scores = (float*)(o + cell.scores);
      L.mods = (float*)(o + cell.mods);
      L.post = opt->do_map ? (float*)(o + cell.post) : nullptr;
      uint8_t* s = (uint8_t*)c->bsmall;
      auto takes = [&](size_t n) { uint8_t* p = s; s += up256(n); return p; };
      L.bq = (cth_bquery*)takes(sizeof(cth_bquery) * P.bq.size());
      L.ytab = (cth_bytile*)takes(sizeof(cth_bytile) * P.ytab.size());
      L.pairs = (cth_bpair*)takes(sizeof(cth_bpair) * npairs);
      L.res = (cth_dpres*)takes(sizeof(cth_dpres) * npairs);
      L.stats = (double*)takes(sizeof(double) * CTH_STATS_NOUT * npairs);
      L.mres = (cth_mapres*)takes(sizeof(cth_mapres) * npairs);
      L.cand = (int*)takes(sizeof(int) * npairs);
      L.passed = (int*)takes(sizeof(int) * npairs);
      L.hitl = (int*)takes(sizeof(int) * npairs);
      L.ctr = (int*)takes(sizeof(int) * kNCtr);
      L.hist = (int*)takes(sizeof(int) * hist_ints(npairs));
      L.zrow = (double*)takes(sizeof(double) * (size_t)small_max * P.lqmax);
      L.hits = (cth_hit*)takes(sizeof(cth_hit) * npairs);
      L.alnout = alnbytes ? (char*)takes(alnbytes) : nullptr;
      L.grow = growbytes ? (float*)takes(growbytes) : nullptr;
      L.back = backbytes ? (float*)takes(backbytes) : nullptr;
    }
    // the batch's tables (outside the graph: a replayed graph reads the current ones)
    CTH_HIP_CHECK(hipMemcpyAsync(L.bq, P.bq.data(), sizeof(cth_bquery) * P.bq.size(), hipMemcpyHostToDevice, c->st));
    CTH_HIP_CHECK(hipMemcpyAsync(L.ytab, P.ytab.data(), sizeof(cth_bytile) * P.ytab.size(), hipMemcpyHostToDevice,
                                 c->st));
    CTH_HIP_CHECK(hipMemcpyAsync(L.pairs, P.pairs.data(), sizeof(cth_bpair) * npairs, hipMemcpyHostToDevice, c->st));
    const double t0 = now_ms();
    // the graph: replayed when everything its launches captured is the same
    // (buffers and their layout, sizes, options, the uploaded sets)
    uint32_t mp;
    memcpy(&mp, &opt->minpp, sizeof mp);
    uint64_t key[15] = {(uint64_t)(uintptr_t)c->bcells, (uint64_t)(uintptr_t)c->bsmall, (uint64_t)npairs,
                        (uint64_t)P.ytab.size() | ((uint64_t)P.bq.size() << 32), (uint64_t)P.tile,
                        (uint64_t)P.cells, (uint64_t)P.lqmax | ((uint64_t)rowcap << 32),
                        (uint64_t)S.dp_grid | ((uint64_t)S.small_grid << 32),
                        (uint64_t)S.trace_grid | ((uint64_t)S.map_split << 32),
                        (uint64_t)opt->do_map | ((uint64_t)opt->ssemodel << 8) | ((uint64_t)(alnbytes != 0) << 17) |
                            ((uint64_t)P.ddms << 18) | ((uint64_t)S.dp_waves << 20) |
                            ((uint64_t)S.trace_waves << 24) | ((uint64_t)mp << 32),
                        fnv(&db.d, sizeof db.d), fnv(&c->q.d, sizeof c->q.d),
                        (uint64_t)(uintptr_t)c->q.ddoff, (uint64_t)(uintptr_t)c->q.qrec, (uint64_t)(uintptr_t)c->dtab};
    if (timing) {
      // stage events: the launches run eagerly
      if (capture_or_launch(c, P, L, opt, ldsc, ltmax, rowcap, S, false, true)) return -1;
    } else if (c->has_bgraph && memcmp(key, c->bkey, sizeof key) == 0) {
      CTH_HIP_CHECK(hipGraphLaunch(c->bgraph, c->st));
      c->nbgraph_replays++;
    } else {
      if (capture_or_launch(c, P, L, opt, ldsc, ltmax, rowcap, S, true, false)) return -1;
      memcpy(c->bkey, key, sizeof key);
      c->nbgraph_captures++;
    }
    // results: counts, then the hit records (and their alignment rows)
    int ctr[kNCtr];
    CTH_HIP_CHECK(hipMemcpyAsync(ctr, L.ctr, sizeof ctr, hipMemcpyDeviceToHost, c->st));
    CTH_HIP_CHECK(hipStreamSynchronize(c->st));
    const int nb = ctr[kCtrHits];
    std::vector<cth_hit> bh(nb);
    std::vector<char> rows_h;
    if (nb) CTH_HIP_CHECK(hipMemcpyAsync(bh.data(), L.hits, sizeof(cth_hit) * nb, hipMemcpyDeviceToHost, c->st));
    if (nb && alnbytes) {
      rows_h.resize((size_t)nb * 5 * rowcap);
      CTH_HIP_CHECK(hipMemcpyAsync(rows_h.data(), L.alnout, rows_h.size(), hipMemcpyDeviceToHost, c->st));
    }
    CTH_HIP_CHECK(hipStreamSynchronize(c->st));
    const double t1 = now_ms();
    if (timing) {
      float a = 0, b = 0, s2 = 0, m = 0;
      CTH_HIP_CHECK(hipEventElapsedTime(&a, c->ev[0], c->ev[1]));
      CTH_HIP_CHECK(hipEventElapsedTime(&b, c->ev[1], c->ev[2]));
      CTH_HIP_CHECK(hipEventElapsedTime(&s2, c->ev[2], c->ev[3]));
      CTH_HIP_CHECK(hipEventElapsedTime(&m, c->ev[3], c->ev[4]));
      st.ms_k_score += a;
      st.ms_k_dp += b;
      st.ms_k_stats += s2;
      st.ms_k_map += m;
    }
    // hits per query: those with an alignment (with MAP), sorted by (log E, profile)
    std::vector<std::vector<cth_hit>> per(P.q1 - P.q0);
    for (const cth_hit& h : bh) {
      if (opt->do_map) st.map_cells += (double)c->q.h_len[h.query] * (double)db.h_len[h.profile];
      if (opt->do_map && h.alnlen < 1) continue;
      per[local[h.query]].push_back(h);
    }
    for (int b = 0; b < P.q1 - P.q0; b++) {
      auto& v = per[b];
      std::sort(v.begin(), v.end(), [](const cth_hit& x, const cth_hit& y) {
        return x.logE < y.logE || (x.logE == y.logE && x.profile < y.profile);
      });
      if (nh + (int)v.size() > maxhits) { cth_set_error("search_batch: hit buffer full (%d)", maxhits); return -1; }
      for (cth_hit h : v) {
        if (alnbytes) {
          const size_t n = (size_t)h.alnlen;
          if (alnused + 5 * n > opt->alncap) {
            cth_set_error("search_batch: alignment buffer full (%llu bytes)", (unsigned long long)opt->alncap);
            return -1;
          }
          const char* src = rows_h.data() + h.alnoff * 5 * (size_t)rowcap;
          for (int r = 0; r < 5; r++)
            for (size_t m = 0; m < n; m++) opt->alnbuf[alnused + r * n + m] = src[r * (size_t)rowcap + n - 1 - m];
          h.alnoff = alnused;
          alnused += 5 * n;
        } else {
          h.alnoff = 0;
        }
        hits[nh++] = h;
      }
      if (nhits) nhits[P.q0 + b] = (int)v.size();
    }
    st.cells += (double)P.cells;
    st.npassed += ctr[kCtrPassed];
    st.nchunks += 1;
    st.ms_phase1 += t1 - t0;
    qa = P.q1;
  }
  if (stats) *stats = st;
  return 0;
}

}  // namespace

extern "C" int cth_search_batch(cth_ctx* c, int q0, int q1, const cth_search_opts* opt, cth_hit* hits, int maxhits,
                                int* nhits, cth_search_stats* stats) {
  if (!c->has_q || !c->has_db) { cth_set_error("search_batch: queries or database not uploaded"); return -1; }
  if (q0 < 0 || q1 > c->q.d.nprof || q0 >= q1) { cth_set_error("search_batch: bad query range [%d,%d)", q0, q1); return -1; }
  if (cth_search_opts_check(opt, "search_batch")) return -1;
  std::vector<int> ql(q1 - q0);
  std::iota(ql.begin(), ql.end(), q0);
  return search_batch_list(c, ql.data(), q1 - q0, opt, hits, maxhits, nhits, stats);
}

extern "C" int cth_search_batch_list(cth_ctx* c, const int32_t* qidx, int nq, const cth_search_opts* opt,
                                     cth_hit* hits, int maxhits, int* nhits, cth_search_stats* stats) {
  if (!c->has_q || !c->has_db) { cth_set_error("search_batch_list: queries or database not uploaded"); return -1; }
  if (!qidx || nq < 1) { cth_set_error("search_batch_list: empty query list"); return -1; }
  if (cth_search_opts_check(opt, "search_batch_list")) return -1;
  std::vector<char> seen(c->q.d.nprof, 0);
  std::vector<int> ql(nq);
  for (int k = 0; k < nq; k++) {
    const int q = qidx[k];
    if (q < 0 || q >= c->q.d.nprof) { cth_set_error("search_batch_list: query %d out of range", q); return -1; }
    if (seen[q]) { cth_set_error("search_batch_list: query %d listed twice", q); return -1; }
    seen[q] = 1;
    ql[k] = q;
  }
  return search_batch_list(c, ql.data(), nq, opt, hits, maxhits, nhits, stats);
}

// Host check of the cell buffers' layout: byte offsets of the traceback bytes,
// scores, modular scores and posteriors, and the size of the whole.
extern "C" void cth_selftest_batch_cells(uint64_t cells, int do_map, uint64_t out[5]) {
  const cell_layout C = lay_cells((size_t)cells, do_map != 0);
  out[0] = C.btck; out[1] = C.scores; out[2] = C.mods; out[3] = C.post; out[4] = C.bytes;
}

// Counts of graph captures and replays of the batched search on a context
// (measurement aid).
extern "C" int cth_batch_graph_counts(const cth_ctx* c, int64_t* captures, int64_t* replays) {
  if (captures) *captures = c->nbgraph_captures;
  if (replays) *replays = c->nbgraph_replays;
  return 0;
}
