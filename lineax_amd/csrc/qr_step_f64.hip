#include "qr_step_kernel.h"

namespace lxa {

int qr_step(hipStream_t st, int64_t count, const lxa_qr_desc* desc, int mode, int k, const int32_t* kcol, int rows,
            int right, double* a, double* tau, double* tblk) {
  if (mode == kStepUpdate) return launch_step<double, 0, 0>(st, count, desc, mode, k, kcol, right, a, tau, tblk);
  // as few register slots as hold the rows: more cost workgroups a CU
  if (rows <= 512) return launch_step<double, 4, 0>(st, count, desc, mode, k, kcol, right, a, tau, tblk);
  if (rows <= 1024) return launch_step<double, 8, 0>(st, count, desc, mode, k, kcol, right, a, tau, tblk);
  if (rows <= 2048) return launch_step<double, 16, 0>(st, count, desc, mode, k, kcol, right, a, tau, tblk);
  return qr_step_tall(st, count, desc, mode, k, kcol, rows, right, a, tau, tblk);
}

}  // namespace lxa
