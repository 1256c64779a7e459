#include "qr_step_kernel.h"

namespace lxa {

int qr_step(hipStream_t st, int64_t count, const lxa_qr_desc* desc, int mode, int k, const int32_t* kcol, int rows,
            int right, float* a, float* tau, float* tblk) {
  if (mode == kStepUpdate) return launch_step<float, 0, 0>(st, count, desc, mode, k, kcol, right, a, tau, tblk);
  // as few register slots as hold the rows: more cost workgroups a CU
  if (rows <= 512) return launch_step<float, 4, 0>(st, count, desc, mode, k, kcol, right, a, tau, tblk);
  if (rows <= 1024) return launch_step<float, 8, 0>(st, count, desc, mode, k, kcol, right, a, tau, tblk);
  if (rows <= 2048) return launch_step<float, 16, 0>(st, count, desc, mode, k, kcol, right, a, tau, tblk);
  if (rows <= kStepMaxRows) return launch_step<float, 28, 4>(st, count, desc, mode, k, kcol, right, a, tau, tblk);
  return set_error(LXA_EINVAL, "qr step: panel of %d rows", rows);  // panel_only and qr_steps see to that
}

}  // namespace lxa
