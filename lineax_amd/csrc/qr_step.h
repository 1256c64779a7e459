// What the QR panel step kernels (qr_step_*.hip) and the
// factorisation around them (qr.hip) share.
#pragma once
#include "lxa_common.h"

namespace lxa {

// What a launch does with the panel at column k.
enum : int {
  kStepPanel = 0,      // factor it (one workgroup per system)
  kStepUpdate = 1,     // apply it to the columns on its right
  kStepLookahead = 2,  // apply it, and factor the panel after it
};

constexpr int kStepMaxRows = 4096;  // tallest panel the step kernel factors

// One launch of qr_step_kernel over `count` systems, the panel at column k
// (kcol == nullptr) or kcol[s] + k of system s.  rows bounds their rows from
// that column on and right the columns right of the panel.
int qr_step(hipStream_t st, int64_t count, const lxa_qr_desc* desc, int mode, int k, const int32_t* kcol, int rows,
            int right, float* a, float* tau, float* tblk);
int qr_step(hipStream_t st, int64_t count, const lxa_qr_desc* desc, int mode, int k, const int32_t* kcol, int rows,
            int right, double* a, double* tau, double* tblk);
// Panels (and their updates, kStepLookahead) of 2049 to kStepMaxRows rows.
int qr_step_tall(hipStream_t st, int64_t count, const lxa_qr_desc* desc, int mode, int k, const int32_t* kcol, int rows,
                 int right, double* a, double* tau, double* tblk);

namespace {

template <typename T>
struct QrCfg {
  static constexpr int NB = 16;
};

constexpr int kPanelThreads = 512;   // 2 waves per SIMD: 256 VGPRs each
constexpr int kPanelWaves = kPanelThreads / kWave;

// Householder vector entry j of panel-relative row (row - k): 1 on the
// diagonal, the stored value below it, 0 above.
template <typename T>
__device__ __forceinline__ T vpick(int row, int diag, T stored) {
  return row > diag ? stored : (row == diag ? T(1) : T(0));
}

}  // namespace
}  // namespace lxa
