// selftest_mfma.hip: device check of the matrix instructions' lane layout
// (cth_mfma.h), on which the reduced-precision log-odds product of
// k_score_plain (score.hip) relies.
#include <hip/hip_runtime.h>

#include "cth_dev.h"
#include "cth_math.h"
#include "cth_mfma.h"

namespace {

// Lane layout check of the 32x32x16 instructions: A = I (32 x 16 block of
// the identity), B[k][c] = 32 (k - 8 h) + c for k in [8 h, 8 h + 8) and 0
// elsewhere (h = 0, 1; every value below 256, exact in BF16), so
// D[r][c] = B[r][c] for r < 16; out[lane*16 + r] receives accumulator r of
// each lane.
template <int kPrec>
__global__ void k_selftest_mfma(float* out, int h) {
  const int lane = threadIdx.x;
  const int l32 = lane & 31, ko = (lane >> 5) * 8;
  v8s a, b;
  for (int k = 0; k < 8; k++) {
    const int kk = ko + k;
    const float av = (l32 == kk) ? 1.0f : 0.0f;
    const float bv = (kk >> 3) == h ? (float)(32 * (kk - 8 * h) + l32) : 0.0f;
    a[k] = (short)mfma_operand<kPrec>(av);
    b[k] = (short)mfma_operand<kPrec>(bv);
  }
  v16f acc = {};
  acc = mfma<kPrec>(a, b, acc);
  for (int r = 0; r < 16; r++) out[lane * 16 + r] = acc[r];
}

}  // namespace

// Device check of the MFMA lane layout assumed above: 0 when every
// accumulator holds the expected element (for both precisions).
extern "C" int cth_selftest_mfma(int* bad) {
  float* d = nullptr;
  CTH_HIP_CHECK(hipMalloc((void**)&d, 64 * 16 * sizeof(float)));
  float h[64 * 16];
  *bad = 0;
  for (int prec = 1; prec <= 2; prec++)
    for (int half = 0; half < 2; half++) {
      if (prec == 1) hipLaunchKernelGGL(k_selftest_mfma<1>, dim3(1), dim3(64), 0, 0, d, half);
      else hipLaunchKernelGGL(k_selftest_mfma<2>, dim3(1), dim3(64), 0, 0, d, half);
      if (hipMemcpy(h, d, sizeof h, hipMemcpyDeviceToHost) != hipSuccess) {
        (void)hipFree(d);
        cth_set_error("selftest_mfma: copy failed");
        return -1;
      }
      for (int lane = 0; lane < 64; lane++)
        for (int r = 0; r < 16; r++) {
          const int row = 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), col = lane & 31;
          const float want = (row >> 3) == half ? (float)(32 * (row - 8 * half) + col) : 0.0f;
          if (h[lane * 16 + r] != want) (*bad)++;
        }
    }
  (void)hipFree(d);
  return 0;
}
