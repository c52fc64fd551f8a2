// stats.hip: alignment statistics and E-values for profiles passed to phase 2.
//
// k_hist  : the 641-bin histogram of rint(32*clamp(S,-10,10)) over each passed
//           profile's Lq x Lt scores (integer counts; masked 'X' positions
//           skipped), the work of CalcScoreProbsXuninfDynPlmProfile
//           (cuss/CuBatchSS_dynplm.cu:134-182), rows over several workgroups
//           where profiles are few.
// k_stats : one workgroup per passed profile computes in double precision the
//           parameters of CalcStatParamsDynPlmProfile (cuss/CuBatchSS_dynplm.cu:
//           193-430): expected score, min/max, lambda by Newton-Raphson with
//           bisection, relative entropy, K by the sigma series on the
//           reference's 21x32 score grid (the 672 grid cells spread over the
//           threads, each sum a workgroup reduction in a fixed order), then
//           the SS18 E-value of CalcSignificanceSS18DynPlmProfile
//           (cuss/CuBatchSS_dynplm.cu:447-580, cuss/CuBatchSS_SS18.cuh:119-453)
//           with the two small networks of cuss/CuBatchSS_NN.cuh:37-202.
//           Special functions: log regularized incomplete beta and upper
//           incomplete gamma by Lentz continued fractions and the lower-gamma
//           series (Numerical Recipes 3rd ed., 6.2, 6.4), in double precision.
// Both are latency: a search has a handful of passed profiles.  10 profiles of
// a 250-position query: 1.24 -> 0.12 ms (sums by one lane and one workgroup
// per histogram before); 3 of a 2000-position query 11.6 -> 0.14 ms.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cth_batch.h"
#include "cth_dev.h"
#include "cth_dp.h"
#include "cth_stats.h"

namespace {

constexpr int kNSC = 21, kScale = 32, kSscMin = -320, kNssc = 641;
constexpr double kLogSpMin = -8.7336545e+01, kLogSpMax = 8.8722839e+01;

// NN weights and SS18 adjustment parameters (cupro/CuDeviceMemory.cu:43-77)
__constant__ float c_nnw[93] = {
    3.1179029f, 0.2732032f, -1.7865388f, -2.7370650f, -2.4113938f,
    2.8802990f, -0.0845794f, 0.7335855f, -0.4155596f, -3.5943765f,
    -2.3533863f, -0.1646748f, 2.6470928f, 1.6489798f, -0.7481717f,
    -0.1763256f, 0.3270687f, 0.5918245f, 0.4900585f, 0.0253580f,
    2.0547640f, 1.4051396f, -1.7874640f, 2.0048461f, 0.6947985f,
    -0.0605839f, 0.0533123f, -1.0046299f, 0.9682557f, 0.0f,
    -0.0173019f, -0.0051053f, 0.6215832f, -0.5038284f, 0.0f,
    0.0600411f, -0.0527767f, 1.0036328f, -0.9667071f, 0.0f,
    -5.9555713f, -3.1437676f, 1.8754493f, 3.4776044f, 0.0f,
    2.8086869f, -0.5250554f, 0.3085814f, 0.5244239f, 2.4166220f,
    -4.4935289f, -11.5416831f, 0.4601384f, 4.1707612f, 0.0f,
    1.4710020f, 0.7746900f, 0.5248285f, -2.2621661f, 0.0f,
    -1.4710009f, -0.7746948f, -0.5248293f, 2.2621667f, 0.0f,
    4.8137710f, 1.0000337f, 2.0837171f, -5.3104535f, 0.0f,
    2.5137293f, 4.2316344f, -0.8620832f, 0.8620837f, 3.1901578f,
    0.1f, 12.0f, 1.0f, 4.0f, 0.05f, 1.0f, 0.1f, 0.35f, 0.65f,
    0.6f, 16.0f, 1.0f, 12.0f, 0.3f, -1.7f, 0.1f, 0.45f, 0.65f};

constexpr int kThreads = 256, kWaves = kThreads / 64;
// copies of the histogram, by lane: the scores of neighbouring cells fall
// into few bins, and atomics of a wavefront on one LDS word serialise
constexpr int kCopies = 4;
// rows of a wavefront whose scores are loaded together: with one at a time it
// waited for every row's (1500 profiles of 372 x 235 cells 243 us instead of
// 316; two or eight rows, and more copies, are alike)
constexpr int kHistRows = 4;

// Adds the scores of query rows [y0, y1) of query qp against profile p
// (scores from scores[colp], row stride ldsc) to the workgroup's histogram
// copies h (kCopies x 641, zeroed), a row per wavefront at a time.
__device__ __forceinline__ void hist_fill(const cth_dpset& q, int qp, const cth_dpset& db, int p, int64_t colp,
                                          int64_t ldsc, const float* __restrict__ scores, int y0, int y1, int* h) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lt = db.len[p];
  const char* qaa = q.aa + q.dist[qp];
  const char* taa = db.aa + db.dist[p];
  int* const hl = h + (lane & (kCopies - 1));
  for (int x0 = 0; x0 < lt; x0 += 256) {
    // four columns per lane, their masked positions once per column block
    bool use[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int x = x0 + 64 * i + lane;
      use[i] = x < lt && taa[x] != 'X';
    }
    for (int y = y0 + w; y < y1; y += kHistRows * kWaves) {
      float v[kHistRows][4];
      bool in[kHistRows];
#pragma unroll
      for (int r = 0; r < kHistRows; r++) {
        const int yr = min(y + r * kWaves, y1 - 1);
        in[r] = y + r * kWaves < y1 && qaa[yr] != 'X';
        const float* const row = scores + (int64_t)yr * ldsc + colp + x0 + lane;
#pragma unroll
        for (int i = 0; i < 4; i++) v[r][i] = use[i] ? row[64 * i] : 0.0f;
      }
#pragma unroll
      for (int r = 0; r < kHistRows; r++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float s = v[r][i];
          if (s < -10.0f) s = -10.0f;
          else if (s > 10.0f) s = 10.0f;
          if (in[r] && use[i]) atomicAdd(&hl[((int)rintf(s * 32.0f) - kSscMin) * kCopies], 1);
        }
      }
    }
  }
}

// workgroup (k, split) adds its share of profile k's rows to hist (zeroed)
__global__ __launch_bounds__(kThreads) void k_hist(const cth_dpset q, int qp, const cth_dpset db, int64_t col0,
                                                   int64_t ldsc, const float* __restrict__ scores,
                                                   const int* __restrict__ plist, int* __restrict__ hist) {
  __shared__ int h[kNssc * kCopies];
  const int k = blockIdx.x;
  const int p = plist[k];
  const int lq = q.len[qp], ny = (lq + (int)gridDim.y - 1) / (int)gridDim.y;
  const int y0 = (int)blockIdx.y * ny, y1 = min(lq, y0 + ny);
  if (y0 >= y1) return;
  for (int b = threadIdx.x; b < kNssc * kCopies; b += kThreads) h[b] = 0;
  __syncthreads();
  hist_fill(q, qp, db, p, db.dist[p] - col0, ldsc, scores, y0, y1, h);
  __syncthreads();
  for (int b = threadIdx.x; b < kNssc; b += kThreads) {
    int n = 0;
    for (int i = 0; i < kCopies; i++) n += h[b * kCopies + i];
    if (n) atomicAdd(&hist[(int64_t)k * kNssc + b], n);
  }
}

__global__ void k_hist_zero(int* hist, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += gridDim.x * (int64_t)blockDim.x)
    hist[i] = 0;
}

__device__ void grid_bounds(int y, int* left, int* right) {
  const int u = y - 10;
  int l = u * kScale - (kScale >> 1) - kSscMin;
  int r = u * kScale + (kScale >> 1) - kSscMin;
  if (u <= 0) { l++; if (l < 0) l = 0; }
  if (0 <= u) { r--; if (kNssc - 1 < r) r = kNssc - 1; }
  *left = l; *right = r;
}

// v with the lanes moved by a DPP control (lanes without a source: 0)
template <int kCtrl, int kRowMask>
__device__ __forceinline__ double dpp_add(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, kCtrl, kRowMask, 0xf, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), kCtrl, kRowMask, 0xf, false);
  return v + __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
// The wavefront's sum of v, in every lane: within rows of 16 lanes, then over
// the rows, in the DPP moves' fixed order (a shuffle waits for the LDS).
__device__ __forceinline__ double wave_sum(double v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);  // row_bcast:15, :31
  v = dpp_add<0x143, 0xc>(v);
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)b, 63);
  const uint32_t hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// The workgroup's sums (and extremes) of two doubles per thread, to every
// thread: a sum in each wavefront, then the wavefronts in order.  red:
// 2 kWaves doubles of LDS.
__device__ __forceinline__ void block_sum2(double& a, double& b, double* red) {
  a = wave_sum(a);
  b = wave_sum(b);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { red[2 * w] = a; red[2 * w + 1] = b; }
  __syncthreads();
  a = red[0]; b = red[1];
  for (int k = 1; k < kWaves; k++) { a += red[2 * k]; b += red[2 * k + 1]; }
  __syncthreads();
}
__device__ __forceinline__ void block_minmax(double& mn, double& mxs, double* red) {
  for (int off = 32; off >= 1; off >>= 1) {
    const double a = __shfl_xor(mn, off), b = __shfl_xor(mxs, off);
    if (a < mn) mn = a;
    if (b > mxs) mxs = b;
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { red[2 * w] = mn; red[2 * w + 1] = mxs; }
  __syncthreads();
  for (int k = 0; k < kWaves; k++) {
    if (red[2 * k] < mn) mn = red[2 * k];
    if (red[2 * k + 1] > mxs) mxs = red[2 * k + 1];
  }
  __syncthreads();
}

// a thread's cells of the 21 x 32 grid: cell threadIdx.x + 256 i, its score
// and probability
constexpr int kCells = (kNSC * kScale + kThreads - 1) / kThreads;
struct grid_cells {
  double g[kCells];
  double sc[kCells];
};

// the lambda equation and its derivative at x, to every thread
__device__ void lambda_eq(const grid_cells& C, double x, double mn, double mxs, double* red, double* f, double* df) {
  double lf = 0.0, ldf = 0.0;
  for (int i = 0; i < kCells; i++) {
    double sc = C.sc[i];
    if (C.g[i] != 0.0 && mn <= sc && sc <= mxs) {
      sc -= mxs;
      const double e = x * sc;
      if (kLogSpMin < e) {
        const double t = exp(e) * C.g[i];
        lf += t;
        ldf += t * sc;
      }
    }
  }
  block_sum2(lf, ldf, red);
  const double e = x * -mxs;
  if (kLogSpMin < e) {
    const double t = exp(e);
    lf -= t;
    ldf += t * mxs;
  }
  *f = lf;
  *df = ldf;
}

// uniform over the workgroup: every thread follows the same sums
__device__ double find_lambda(const grid_cells& C, double mn, double mxs, double* red) {
  const double x1 = 1.0e-5, x2 = 10.0, acc = 1.0e-4;
  double f, df, fl, dx, dxold, xh, xl, rts;
  lambda_eq(C, x1, mn, mxs, red, &fl, &df);
  lambda_eq(C, x2, mn, mxs, red, &f, &df);
  if ((fl > 0.0 && f > 0.0) || (fl < 0.0 && f < 0.0)) return -1.0;
  if (fl < 0.0) { xl = x1; xh = x2; } else { xh = x1; xl = x2; }
  rts = 0.5 * (x1 + x2);
  dxold = fabs(x2 - x1);
  dx = dxold;
  lambda_eq(C, rts, mn, mxs, red, &f, &df);
  int n;
  for (n = 0; n < 32; n++) {
    bool stop = false;
    if ((((rts - xh) * df - f) * ((rts - xl) * df - f) > 0.0) || (fabs(2.0 * f) > fabs(dxold * df))) {
      dxold = dx;
      dx = 0.5 * (xh - xl);
      rts = xl + dx;
      if (xl == rts) stop = true;
    } else {
      dxold = dx;
      dx = f / df;
      const double t = rts;
      rts -= dx;
      if (t == rts) stop = true;
    }
    if (fabs(dx) < acc) stop = true;
    if (stop) break;
    lambda_eq(C, rts, mn, mxs, red, &f, &df);
    if (f < 0.0) xl = rts; else xh = rts;
  }
  return n == 32 ? -1.0 : rts;
}

__device__ double betacf(double a, double b, double x) {
  const double FPMIN = 1e-300, EPS = 1e-15;
  const double qab = a + b, qap = a + 1.0, qam = a - 1.0;
  double c = 1.0, d = 1.0 - qab * x / qap;
  if (fabs(d) < FPMIN) d = FPMIN;
  d = 1.0 / d;
  double h = d;
  for (int m = 1; m < 10000; m++) {
    const int m2 = 2 * m;
    double aa = m * (b - m) * x / ((qam + m2) * (a + m2));
    d = 1.0 + aa * d; if (fabs(d) < FPMIN) d = FPMIN;
    c = 1.0 + aa / c; if (fabs(c) < FPMIN) c = FPMIN;
    d = 1.0 / d;
    h *= d * c;
    aa = -(a + m) * (qab + m) * x / ((a + m2) * (qap + m2));
    d = 1.0 + aa * d; if (fabs(d) < FPMIN) d = FPMIN;
    c = 1.0 + aa / c; if (fabs(c) < FPMIN) c = FPMIN;
    d = 1.0 / d;
    const double del = d * c;
    h *= del;
    if (fabs(del - 1.0) < EPS) break;
  }
  return h;
}

__device__ double lbetainc(double a, double b, double x) {
  if (x <= 0.0) return -999.0;
  if (x >= 1.0) return 0.0;
  const double lbt = lgamma(a + b) - lgamma(a) - lgamma(b) + a * log(x) + b * log1p(-x);
  if (x < (a + 1.0) / (a + b + 2.0)) return lbt + log(betacf(a, b, x)) - log(a);
  const double c = exp(lbt + log(betacf(b, a, 1.0 - x)) - log(b));
  return log1p(-c);
}

__device__ double lgammaincq(double a, double x) {
  if (x <= 0.0) return 0.0;
  const double gln = lgamma(a);
  if (x < a + 1.0) {
    double ap = a, del = 1.0 / a, sum = del;
    for (int n = 0; n < 100000; n++) {
      ap += 1.0;
      del *= x / ap;
      sum += del;
      if (fabs(del) < fabs(sum) * 1e-16) break;
    }
    return log1p(-(sum * exp(-x + a * log(x) - gln)));
  }
  const double FPMIN = 1e-300;
  double b = x + 1.0 - a, c = 1.0 / FPMIN, d = 1.0 / b, h = d;
  for (int i = 1; i < 100000; i++) {
    const double an = -i * (i - a);
    b += 2.0;
    d = an * d + b; if (fabs(d) < FPMIN) d = FPMIN;
    c = b + an / c; if (fabs(c) < FPMIN) c = FPMIN;
    d = 1.0 / d;
    const double del = d * c;
    h *= del;
    if (fabs(del - 1.0) < 1e-16) break;
  }
  return -x + a * log(x) - gln + log(h);
}

__device__ double sig2(double v) { return 2.0 / (1.0 + exp(-v)) - 1.0; }

// one network (cuss/CuBatchSS_NN.cuh:37-148): hidden unit h has bias w[5h]
// and input weights w[5h+1..5h+4], the output bias w[20] and unit weights
// w[21..24]; activation 2/(1+e^-x) - 1
__device__ double nn_out(const double in[4], const float* w, double factor) {
  double acc = w[20];
  for (int h = 0; h < 4; h++) {
    double pre = w[5 * h];
    for (int i = 0; i < 4; i++) pre += in[i] * w[5 * h + 1 + i];
    acc += sig2(pre) * w[21 + h];
  }
  return sig2(acc) * factor;
}

// constants of cuss/CuBatchSS_SS18.cuh:17-41 at the values of the reference's
// single-precision literals
constexpr double kSS18MinScale = (double)0.1f, kSS18Log001 = (double)-4.605170186f,
                 kSS18LogInvNPairs = (double)-9.210340372f, kSS18NbdShape = (double)0.1f,
                 kSS18NbdProb = (double)0.757213f, kSS18EbmDfo2 = (double)1.346206f,
                 kSS18EbmC = (double)1.485656f;

// The significance of one alignment in parts that do not wait for each other:
// what follows from the profiles and the positives alone, what follows from
// lambda, and the rest.
struct sig_parts {
  double emu, logpp;  // network of the effective lengths; positives' log p-value
  double lmu, lsc;    // networks of lambda
};

// emu and logpp (SS18; PredictEVDParametersSS18, cuss/CuBatchSS_SS18.cuh:119-233)
__device__ void sig_profiles(int lq, int lt, double qeno, double teno, double psts, sig_parts& S) {
  const double ln1k = 6.90775527898213681510242167860;
  double in[4];
  double e1 = qeno, e2 = teno;
  int n1 = lq, n2 = lt;
  if (e1 < e2) { double t = e1; e1 = e2; e2 = t; int u = n1; n1 = n2; n2 = u; }
  else if (e1 == e2 && n1 < n2) { int u = n1; n1 = n2; n2 = u; }
  in[0] = (double)0.05f * e1; in[1] = log((double)n1) / ln1k;
  in[2] = (double)0.05f * e2; in[3] = log((double)n2) / ln1k;
  S.emu = nn_out(in, c_nnw, 30.0);
  const double l1l2 = (double)(float)((uint32_t)lq * (uint32_t)lt);
  const double lp = l1l2 < 625.0 ? 625.0 : l1l2;
  const double pn = rint(100000.0 * psts / pow(lp, 1.5));
  S.logpp = lbetainc(pn + 1.0, kSS18NbdShape, kSS18NbdProb);
}

// lmu and lsc
__device__ void sig_lambda(int lq, int lt, double lambda, sig_parts& S) {
  const double ln1k = 6.90775527898213681510242167860;
  double in[4];
  double lm = rint(lambda * 10.0) / 10.0;
  if (lm <= 0.0) lm = 0.1;
  if (10.0 < lm) lm = 10.0;
  int n1 = lq, n2 = lt;
  if (n1 < n2) { int u = n1; n1 = n2; n2 = u; }
  in[0] = (double)0.2f * lm; in[1] = log((double)n1) / ln1k; in[2] = log((double)n2) / ln1k; in[3] = 0.0;
  S.lmu = nn_out(in, c_nnw + 25, 30.0);
  S.lsc = nn_out(in, c_nnw + 50, 5.0);
}

// out = [lmbdest, kest, logE, logEpA]: SSEMODEL 0 observed statistics (S not
// used), 1 and 2 the SS18 model and its variant
__device__ void significance(int ssemodel, int lq, int lt, double searchspace, double score, double lambda, double K,
                             const sig_parts& S, double* out) {
  const double lref = CTH_UNGAP_LAMBDA, kref = CTH_UNGAP_K, lg = CTH_GAPPED_LAMBDA, kg = CTH_GAPPED_K;
  out[0] = 0.0; out[1] = 0.0;
  if (0.0 < lambda) out[0] = lambda * (lg / lref);
  if (0.0 < K) out[1] = K * (kg / kref);
  const double l1l2 = (double)(float)((uint32_t)lq * (uint32_t)lt);
  if (lambda <= 0.0 || K <= 0.0) out[3] = log(kref * l1l2) - lref * score;
  else out[3] = log(K * l1l2) - lambda * score;
  if (ssemodel == 0) {
    // observed statistics: the gapped reference parameters alone
    // (CalcSignificanceObsDynPlmProfile -> CalculateEvalueObs,
    // cuss/CuBatchSS_dynplm.cu:594-660, cuss/CuBatchSS_SS18.cuh:355-381)
    out[2] = log(kg * searchspace) - lg * score;
    return;
  }
  double emu = S.emu, lmu = S.lmu, lsc = S.lsc;
  const float* adj = ssemodel == 2 ? c_nnw + 84 : c_nnw + 75;
  if (emu < 3.0) emu = 3.0;
  if (lmu < 3.0) lmu = 3.0;
  if (lsc < kSS18MinScale) lsc = kSS18MinScale;
  lsc = adj[6] * (exp(lsc) - 1.0);
  if (lsc < kSS18MinScale) lsc = kSS18MinScale;
  if (5.0 < lsc) lsc = 5.0;
  double scaleE = adj[4] * emu + adj[5];
  if (scaleE < kSS18MinScale) scaleE = kSS18MinScale;
  if (5.0 < scaleE) scaleE = 5.0;
  emu = adj[0] * emu + adj[1];
  lmu = adj[2] * lmu + adj[3];
  double alpha = adj[7], ibeta = adj[8];
  if (0.0 < lambda) {
    const double r = 1.0 / lambda;
    alpha -= alpha * (double)0.1f * (r < 10.0 ? r : 10.0);
    ibeta += (1.0 - ibeta) * (double)0.1f * (r < 10.0 ? r : 10.0);
  }
  const double mu = alpha * emu + (1.0 - alpha) * lmu;
  const double scale = (1.0 - ibeta) * scaleE + ibeta * lsc;
  // CalculateEvalueSS18 (cuss/CuBatchSS_SS18.cuh:255-351)
  if (mu <= 0.0 || scale <= 0.0) {
    out[2] = log(kg * searchspace) - lg * score;
    return;
  }
  double logK = mu / scale;
  if (K > kref && 0.0 < K && K < 1.0 && 0.0 < kref && kref < 1.0) logK += log(K / kref);
  double logexp = logK - score / scale;
  if (ssemodel == 2) logexp += kSS18LogInvNPairs;
  double logp = logexp;
  if (kSS18Log001 <= logexp) {
    if (kLogSpMax - 3.0 < logexp) logp = 0.0;
    else {
      const double t = exp(logexp);
      if (kLogSpMax - 3.0 < t) logp = 0.0;
      else logp = log(1.0 - exp(-t));
    }
  }
  logp = lgammaincq(kSS18EbmDfo2, (-logp - S.logpp) / kSS18EbmC);
  logexp = logp;
  if (kSS18Log001 <= logp) {
    const double p = exp(logp);
    logexp = 77.0;
    if (p < 1.0) logexp = log(-log(1.0 - p));
  }
  logexp += log(searchspace / l1l2);
  out[2] = logexp;
}

// The sigma series of K (cuss/CuBatchSS_K.cuh) by one wavefront: the sum over j
// of P_j / j for unscaled scores minu..maxu of probabilities pu, lambda.  A
// cell's next value is the sum over i of G[c - i] pu[i], the grid's rows being
// 32 scores apart and its cells consecutive.  Only cells of scores within +-32
// get values, 66 consecutive ones: a lane's two are in registers with their
// weights exp(lambda min(score, 0)), and the values in LDS need no barriers.
// G: the grid at the start, which this overwrites around those cells.
//
// 32 turns over all 672 cells on the workgroup, its barriers and shuffles, took
// 61 us of a profile's 92.
__device__ double sigma_series(int minu, int maxu, double lambda, double* G, const double* pu) {
  constexpr int kFirst = 10 * kScale - 17, kActive = 66;  // scores -32..16 and 16..32
  const int lane = threadIdx.x & 63, range = maxu - minu + 1;
  int cell[2], sc[2];
  double weight[2];
  bool on[2];
#pragma unroll
  for (int s = 0; s < 2; s++) {
    const int k = min(lane + 64 * s, kActive - 1);
    cell[s] = kFirst + k;
    sc[s] = k < 49 ? k - 32 : k - 33;
    const double e = sc[s] < 0 ? lambda * (double)sc[s] : 0.0;
    on[s] = lane + 64 * s < kActive && kLogSpMin < e;
    weight[s] = exp(e);
  }
  double sigma = 0.0, Pj = 1.0;
  int minscore = minu, maxscore = maxu;
  for (int j = 1; j <= 32 && 1.0e-4 < Pj; j++) {
    int lo[2], hi[2];
    double v[2] = {0.0, 0.0};
#pragma unroll
    for (int s = 0; s < 2; s++) {
      lo[s] = maxscore - sc[s] < range ? maxu - (maxscore - sc[s]) : minu;
      hi[s] = sc[s] - minscore < range ? minu + (sc[s] - minscore) : maxu;
      if (!(on[s] && minscore <= sc[s] && sc[s] <= maxscore)) hi[s] = lo[s] - 1;
    }
    for (int i = minu; i <= maxu; i += 4) {
      double g[2][4], p[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        p[u] = pu[min(i + u + 10, kNSC - 1)];
        g[0][u] = G[cell[0] - i - u];
        g[1][u] = G[cell[1] - i - u];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
#pragma unroll
        for (int s = 0; s < 2; s++)
          if (lo[s] <= i + u && i + u <= hi[s]) v[s] += g[s][u] * p[u];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (j == 1 && lane < 13) G[kFirst - 1 - lane] = G[kFirst + kActive + lane] = 0.0;
    G[cell[0]] = v[0];
    if (lane + 64 < kActive) G[cell[1]] = v[1];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    Pj = wave_sum(v[0] * weight[0] + v[1] * weight[1]);
    sigma += Pj / j;
    minscore += minu;
    maxscore += maxu;
  }
  return sigma;
}

// The statistics of one passed profile p (one workgroup): parameters from
// its histogram (bin b the sum of hc[b * copies .. +copies)), then the
// significance of its phase-1 record r, into the CTH_STATS_NOUT doubles at o.
// The grid's cells are spread over the threads, each sum a workgroup
// reduction in a fixed order: a serial chain in one lane (672 exponentials per
// evaluation of the lambda equation, ~12 evaluations) took ~0.8 ms.
template <int kHistCopies>
__device__ __forceinline__ void stats_one(const cth_dpset& q, int qp, const cth_dpset& db, int p, const int* hc,
                                          double searchspace, int ssemodel, const cth_dpres& r, double* o) {
  __shared__ double G[kNSC * kScale];
  __shared__ double pu[kNSC];
  __shared__ double red[2 * kWaves];
  __shared__ sig_parts S;
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = q.len[qp], lt = db.len[p];
  auto bin = [&](int b) {
    int n = 0;
    for (int i = 0; i < kHistCopies; i++) n += hc[b * kHistCopies + i];
    return (double)n;
  };
  // counts (whole numbers: their sums are exact in any order)
  grid_cells C;
  for (int i = 0; i < kCells; i++) {
    const int c = tid + kThreads * i, y = c / kScale, x = c - y * kScale;
    C.g[i] = 0.0;
    C.sc[i] = 0.0;
    if (c < kNSC * kScale) {
      int l, rr;
      grid_bounds(y, &l, &rr);
      C.sc[i] = l + x + kSscMin;
      if (l + x <= rr) C.g[i] = bin(l + x);
    }
    double n = C.g[i];
    for (int off = 16; off >= 1; off >>= 1) n += __shfl_xor(n, off);
    if (c < kNSC * kScale && x == 0) pu[y] = n;
  }
  double total = 0.0, E = 0.0;
  for (int b = tid; b < kNssc; b += kThreads) total += bin(b);
  block_sum2(total, E, red);
  for (int i = 0; i < kCells; i++) C.g[i] = C.g[i] / total;
  if (tid < kNSC) pu[tid] = pu[tid] / total;
  double mn = 0.0, mxs = 0.0, zero = 0.0;
  E = 0.0;
  for (int i = 0; i < kCells; i++) {
    E += C.sc[i] * C.g[i];
    const double v = C.g[i] ? C.sc[i] : 0.0;
    if (v < mn) mn = v;
    if (v > mxs) mxs = v;
  }
  block_sum2(E, zero, red);
  block_minmax(mn, mxs, red);
  double lambda = -1.0;
  if (!(0.0 <= E || mxs <= 0.0)) lambda = find_lambda(C, mn, mxs, red);
  double H = -1.0;
  if (lambda > 0.0) {
    H = 0.0;
    for (int i = 0; i < kCells; i++) {
      const double sc = C.sc[i];
      if (C.g[i] != 0.0 && mn <= sc && sc <= mxs) {
        const double yy = lambda * sc;
        if (kLogSpMin < yy && yy < kLogSpMax - 3.0) H += exp(yy) * yy * C.g[i];
      }
    }
    zero = 0.0;
    block_sum2(H, zero, red);
  }
  lambda *= kScale;
  E /= kScale;
  for (int i = 0; i < kCells; i++) {
    const int c = tid + kThreads * i;
    if (c < kNSC * kScale) G[c] = c / kScale == 10 ? 1.0 : C.g[i];
  }
  __syncthreads();
  double umn = 0.0, umx = 0.0;
  for (int y = 0; y < kNSC; y++) {
    const double v = pu[y] ? (double)(y - 10) : 0.0;
    if (v < umn) umn = v;
    if (v > umx) umx = v;
  }
  // K on wavefront 0, meanwhile the significance's independent parts on two others
  double K = -1.0;
  if (w == 0 && !(0.0 <= E || lambda <= 0.0 || H <= 0.0)) {
    if (umn == -1.0 && umx == 1.0) {
      const double a = pu[9], b = pu[11];
      K = (a - b) * (a - b) / a;
    } else if (umn == -1.0 || umx == 1.0) {
      if (umx != 1.0) K = lambda / H * (1.0 - exp(-lambda)) * (E * E);
      else K = H / lambda * (1.0 - exp(-lambda));
    } else {
      const double sigma = sigma_series((int)umn, (int)umx, lambda, G, pu);
      K = lambda * exp(-2.0 * sigma) / (H * (1.0 - exp(-lambda)));
    }
  }
  if (ssemodel != 0 && (tid & 63) == 0) {
    if (w == 1) sig_profiles(lq, lt, (double)q.eno[qp], (double)db.eno[p], (double)r.psts, S);
    if (w == 2) sig_lambda(lq, lt, lambda, S);
  }
  __syncthreads();
  if (tid == 0) {
    double sig[4];
    significance(ssemodel, lq, lt, searchspace, (double)r.score, lambda, K, S, sig);
    o[CTH_ST_LMBDEST] = sig[0]; o[CTH_ST_KEST] = sig[1]; o[CTH_ST_LOGE] = sig[2]; o[CTH_ST_LOGEPA] = sig[3];
    o[CTH_ST_MIN] = umn; o[CTH_ST_MAX] = umx; o[CTH_ST_E] = E; o[CTH_ST_H] = H;
    o[CTH_ST_LMBD] = lambda; o[CTH_ST_K] = K;
  }
}

__global__ __launch_bounds__(kThreads) void k_stats(const cth_dpset q, int qp, const cth_dpset db,
                                                    const int* __restrict__ plist, const int* __restrict__ prel,
                                                    const cth_dpres* __restrict__ dpres,
                                                    const int* __restrict__ hist, double searchspace, int ssemodel,
                                                    double* __restrict__ out) {
  const int k = blockIdx.x;
  stats_one<1>(q, qp, db, plist[k], hist + (int64_t)k * kNssc, searchspace, ssemodel, dpres[prel[k]],
               out + (int64_t)k * CTH_STATS_NOUT);
}

// Histograms of the *count passed pairs listed in list into hist (zeroed, one
// per list slot), where they are at most cap: rows over workgroups as in
// cth_launch_stats.  More pairs leave theirs to k_stats_batch.
__global__ __launch_bounds__(kThreads) void k_hist_batch(const cth_dpset q, const cth_dpset db,
                                                         const cth_bquery* __restrict__ bq,
                                                         const cth_bpair* __restrict__ pairs,
                                                         const int* __restrict__ list, const int* __restrict__ count,
                                                         int64_t ldsc, const float* __restrict__ scores, int lqmax,
                                                         int* __restrict__ hist, int cap) {
  __shared__ int h[kNssc * kCopies];
  const int nj = *count;
  if (nj < 1 || nj > cap) return;
  const int split = max(1, min(1024 / nj, (lqmax + 15) / 16));
  for (int u = blockIdx.x; u < nj * split; u += gridDim.x) {
    const int k = u / split;
    const cth_bpair pr = pairs[list[k]];
    const cth_bquery Q = bq[pr.b];
    const int ny = (Q.lq + split - 1) / split;
    const int y0 = (u - k * split) * ny, y1 = min(Q.lq, y0 + ny);
    if (y0 >= y1) continue;
    for (int b = threadIdx.x; b < kNssc * kCopies; b += kThreads) h[b] = 0;
    __syncthreads();
    hist_fill(q, Q.qp, db, pr.p, db.dist[pr.p], ldsc, scores + Q.off, y0, y1, h);
    __syncthreads();
    for (int b = threadIdx.x; b < kNssc; b += kThreads) {
      int n = 0;
      for (int i = 0; i < kCopies; i++) n += h[b * kCopies + i];
      if (n) atomicAdd(&hist[(int64_t)k * kNssc + b], n);
    }
    __syncthreads();
  }
}

// Batched statistics over the *count passed pairs listed in list
// (persistent, one workgroup per pair at a time): its histogram from
// k_hist_batch, or in LDS where those are more than cap, then the parameters
// and significance against the pair's query's search space; out and dpres are
// per pair.
__global__ __launch_bounds__(kThreads) void k_stats_batch(const cth_dpset q, const cth_dpset db,
                                                          const cth_bquery* __restrict__ bq,
                                                          const cth_bpair* __restrict__ pairs,
                                                          const int* __restrict__ list, const int* __restrict__ count,
                                                          int64_t ldsc, const float* __restrict__ scores,
                                                          const cth_dpres* __restrict__ dpres, int ssemodel,
                                                          const int* __restrict__ hist, int cap,
                                                          double* __restrict__ out) {
  __shared__ int h[kNssc * kCopies];
  const int nj = *count;
  for (int k = blockIdx.x; k < nj; k += gridDim.x) {
    const int i = list[k];
    const cth_bpair pr = pairs[i];
    const cth_bquery Q = bq[pr.b];
    for (int b = threadIdx.x; b < kNssc * kCopies; b += kThreads)
      h[b] = nj <= cap && b % kCopies == 0 ? hist[(int64_t)k * kNssc + b / kCopies] : 0;
    __syncthreads();
    if (nj > cap) {
      hist_fill(q, Q.qp, db, pr.p, db.dist[pr.p], ldsc, scores + Q.off, 0, Q.lq, h);
      __syncthreads();
    }
    stats_one<kCopies>(q, Q.qp, db, pr.p, h, Q.sspace, ssemodel, dpres[i], out + (int64_t)i * CTH_STATS_NOUT);
    __syncthreads();
  }
}

}  // namespace

// Statistics for the np2 passed profiles listed in plist (indices into the
// launch's profile range, relative to p0 as the DP results are); hist is
// scratch of np2*641 ints, out receives np2 x CTH_STATS_NOUT doubles.
extern "C" int cth_launch_stats(const cth_dpset* q, int qp, int lq, const cth_dpset* db, int p0, int64_t col0,
                                int64_t ldsc, const float* scores, const int* plist_abs, const int* plist_rel,
                                const cth_dpres* dpres, int np2, double searchspace, int ssemodel, int* hist,
                                double* out, hipStream_t st) {
  if (np2 <= 0) return 0;
  (void)p0;
  // few profiles: their rows over several workgroups each, at least 16 rows
  // apiece, about four workgroups per compute unit
  const int split = std::max(1, std::min(1024 / np2, (lq + 15) / 16));
  const int64_t n = (int64_t)np2 * kNssc;
  hipLaunchKernelGGL(k_hist_zero, dim3((unsigned)std::min<int64_t>((n + 255) / 256, 1024)), dim3(256), 0, st, hist, n);
  hipLaunchKernelGGL(k_hist, dim3(np2, split), dim3(kThreads), 0, st, *q, qp, *db, col0, ldsc, scores, plist_abs, hist);
  CTH_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(k_stats, dim3(np2), dim3(kThreads), 0, st, *q, qp, *db, plist_abs, plist_rel, dpres, hist,
                     searchspace, ssemodel, out);
  CTH_HIP_CHECK(hipGetLastError());
  return 0;
}

// Batched statistics (k_hist_batch, k_stats_batch) on a persistent grid of
// `grid` workgroups over the *count pairs of list; hist: cap x 641 zeroed ints;
// lqmax: the longest query; out: CTH_STATS_NOUT doubles per pair.
extern "C" int cth_launch_stats_batch(const cth_dpset* q, const cth_dpset* db, const cth_bquery* bq,
                                      const cth_bpair* pairs, const int* list, const int* count, int64_t ldsc,
                                      const float* scores, const cth_dpres* dpres, int ssemodel, int lqmax, int* hist,
                                      int cap, double* out, int grid, hipStream_t st) {
  if (grid < 1) return 0;
  hipLaunchKernelGGL(k_hist_batch, dim3(1024), dim3(kThreads), 0, st, *q, *db, bq, pairs, list, count, ldsc, scores,
                     lqmax, hist, cap);
  CTH_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(k_stats_batch, dim3(grid), dim3(kThreads), 0, st, *q, *db, bq, pairs, list, count, ldsc, scores,
                     dpres, ssemodel, hist, cap, out);
  CTH_HIP_CHECK(hipGetLastError());
  return 0;
}
