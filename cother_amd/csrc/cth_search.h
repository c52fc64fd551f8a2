// cth_search.h: the public search types (defined in include/cother_hip.h).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "cother_hip.h"
#include "cth_dp.h"

// checks of the option fields every search entry point shares (0 or -1 with the error set)
extern "C" int cth_search_opts_check(const cth_search_opts* opt, const char* who);
// a query's score threshold, log E-value threshold and length-adjusted search space
extern "C" void cth_query_thresholds(float eval, uint64_t lq, uint64_t dbsize, uint64_t ndb, float* scorethld,
                                     float* logethld, double* sspace);

// One query against the resident profiles [p0, p0+np), whose scores, modular
// scores and first-pass records (res) are on their way on the context's stream.
// Buffers as cth_launch_dp_list takes them, column 0 at col0.
struct cth_chunk {
  int qi, lq, p0, np, ltmax;
  int64_t col0, ldsc;
  float scorethld, logethld;
  double sspace;
  const float* scores;
  const float* mods;
  uint8_t* btck;
  cth_dpres* res;
  int rows;    // alignment rows wanted
  int traced;  // the first pass left traceback bytes and finalised records
};
// What the rest of its pipeline leaves: the hit records in profile order (their
// alnoff a slot of rows, 5 x rowcap letters each), before those without an
// alignment are dropped, and the number of passed profiles.
struct cth_chunk_hits {
  std::vector<cth_hit> hits;
  std::vector<char> rows;
  int rowcap;
  int npassed;
  double ms_phase2;        // wall time from the end of phase 1 on
  float ms_stats, ms_map;  // with stage timing
};
// The call itself.  The context's work area holds its lists and records (about
// 250 bytes a profile), its mapbuf and mapwork the MAP stage's; timing: the
// context's events 2 to 4 are recorded after phase 1, the statistics and MAP.
int cth_chunk_finish(struct cth_ctx* c, const cth_chunk& k, const cth_search_opts* opt, int ncu, bool timing,
                     cth_chunk_hits& out);
