#include "qr_step_kernel.h"

namespace lxa {

int qr_step_tall(hipStream_t st, int64_t count, const lxa_qr_desc* desc, int mode, int k, const int32_t* kcol, int rows,
                 int right, double* a, double* tau, double* tblk) {
  if (rows <= 3072) return launch_step<double, 20, 4>(st, count, desc, mode, k, kcol, right, a, tau, tblk);
  if (rows <= kStepMaxRows) return launch_step<double, 24, 8>(st, count, desc, mode, k, kcol, right, a, tau, tblk);
  return set_error(LXA_EINVAL, "qr step: panel of %d rows", rows);  // panel_only and qr_steps see to that
}

}  // namespace lxa
