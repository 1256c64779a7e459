// Entry points of the uneven-batch Cholesky solve (whose kernels are in
// chol_mfma.hip): the workspace and no-allocation variants, the autotuner's
// hook and the autotune table's query.
#include <mutex>

#include "lxa_common.h"
#include "uneven_tune.h"

namespace lxa {
namespace {

constexpr int kMaxN = 256;
constexpr int64_t kMaxGrid = 2147483647;

}  // namespace
}  // namespace lxa

namespace lxa {

int chol_mfma_launch(hipStream_t s, int64_t count, int max_n, const int32_t* n, const int64_t* a_offset,
                     const float* a, const int64_t* b_offset, const float* b, void* x, int x_dtype,
                     const int32_t* order, bool persistent, bool sorted, int max_refine, double tol, int32_t* info,
                     int32_t* iters, double* eta, unsigned int* queue, int max4, int max8);

namespace {

// Work-queue counters of the persistent launches: one per tile class, and the
// flag of the sortedness check.
constexpr int kQueueCounters = 4;
constexpr size_t kUnevenWorkspaceBytes = 16;  // kQueueCounters 4-byte counters, rounded up
static_assert(kQueueCounters * sizeof(unsigned int) <= kUnevenWorkspaceBytes, "workspace holds the queue counters");

// Device scratch of lxa_chol_uneven_solve_noalloc: the queue counters live in
// this file-scope array instead of a caller's workspace.  Each GPU the
// library runs on holds its own copy until the process ends.  Host code uses
// the address hipGetSymbolAddress returns for the current device, never the
// array's name (a host-side stand-in, not a device address).
constexpr size_t kNoAllocScratchBytes = 256;
static_assert(kUnevenWorkspaceBytes <= kNoAllocScratchBytes, "queue counters exceed the no-alloc scratch");
__device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;

// Device address of `scratch` on the current device, looked up once per
// device (with that device current) and kept; 0 on success.
int noalloc_scratch(unsigned int** out) {
  static std::mutex mu;
  static void* ptr[kMaxDevices] = {};
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_error(e, "lxa_chol_uneven_solve_noalloc: hipGetDevice");
  if (dev < 0 || dev >= kMaxDevices)
    return set_error(LXA_EUNSUPPORTED, "lxa_chol_uneven_solve_noalloc: device %d beyond %d", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_error(e, "lxa_chol_uneven_solve_noalloc: hipGetSymbolAddress(scratch)");
    if (!p) return set_error(LXA_EHIP, "lxa_chol_uneven_solve_noalloc: null scratch address");
    ptr[dev] = p;
  }
  *out = static_cast<unsigned int*>(ptr[dev]);
  return LXA_OK;
}

int uneven_check(int64_t count, int max_n, const int32_t* n, const int64_t* a_offset, const float* a,
                 const int64_t* b_offset, const float* b, void* x, int x_dtype, const int32_t* order,
                 int max_refine, int32_t* info) {
  LXA_REQUIRE(count >= 0 && count <= kMaxGrid, "lxa_chol_uneven_solve: bad count");
  LXA_REQUIRE(max_n >= 1 && max_n <= kMaxN, "lxa_chol_uneven_solve: max_n must be in [1, %d]", kMaxN);
  LXA_REQUIRE(n && a_offset && a && b_offset && b && x && order && info, "lxa_chol_uneven_solve: null pointer");
  LXA_REQUIRE(x_dtype == LXA_F32 || x_dtype == LXA_F64, "lxa_chol_uneven_solve: bad x_dtype");
  LXA_REQUIRE(max_refine >= 0 && max_refine <= 64, "lxa_chol_uneven_solve: max_refine in [0, 64]");
  LXA_REQUIRE(max_refine == 0 || x_dtype == LXA_F64, "lxa_chol_uneven_solve: refinement needs x_dtype F64");
  return LXA_OK;
}

// The launches of one uneven solve (chol_mfma.hip); `queue` holds
// kQueueCounters counters (persistent launches clear them with a fill kernel).
int uneven_launch(hipStream_t s, int64_t count, int max_n, const int32_t* n, const int64_t* a_offset,
                  const float* a, const int64_t* b_offset, const float* b, void* x, int x_dtype,
                  const int32_t* order, int flags, int max_refine, double tol, int32_t* info, int32_t* iters,
                  double* eta, unsigned int* queue, int max4 = kTunedMax4, int max8 = kTunedMax8) {
  return chol_mfma_launch(s, count, max_n, n, a_offset, a, b_offset, b, x, x_dtype, order,
                          (flags & LXA_UNEVEN_PERSISTENT) != 0, (flags & LXA_UNEVEN_SORTED) != 0, max_refine, tol,
                          info, iters, eta, queue, max4, max8);
}

}  // namespace
}  // namespace lxa

extern "C" int lxa_chol_uneven_workspace_size(int64_t count, size_t* bytes) {
  LXA_REQUIRE(count >= 0 && bytes, "lxa_chol_uneven_workspace_size: bad argument");
  *bytes = lxa::kUnevenWorkspaceBytes;  // work-queue counters
  return LXA_OK;
}

extern "C" int lxa_chol_uneven_solve(void* stream, int64_t count, int max_n, const int32_t* n,
                                     const int64_t* a_offset, const float* a, const int64_t* b_offset,
                                     const float* b, void* x, int x_dtype, const int32_t* order, int flags,
                                     int max_refine, double tol, int32_t* info, int32_t* iters, double* eta,
                                     void* workspace, size_t workspace_bytes) {
  if (int rc = lxa::uneven_check(count, max_n, n, a_offset, a, b_offset, b, x, x_dtype, order, max_refine, info))
    return rc;
  const bool persistent = (flags & LXA_UNEVEN_PERSISTENT) != 0;
  LXA_REQUIRE(!persistent || (workspace && workspace_bytes >= lxa::kUnevenWorkspaceBytes),
              "lxa_chol_uneven_solve: the persistent launch needs a workspace of %zu bytes (got %zu)",
              lxa::kUnevenWorkspaceBytes, workspace ? workspace_bytes : static_cast<size_t>(0));
  if (count == 0) return LXA_OK;
  return lxa::uneven_launch(static_cast<hipStream_t>(stream), count, max_n, n, a_offset, a, b_offset, b, x, x_dtype,
                            order, flags, max_refine, tol, info, iters, eta, static_cast<unsigned int*>(workspace));
}

extern "C" int lxa_chol_uneven_solve_noalloc(void* stream, int64_t count, int max_n, const int32_t* n,
                                             const int64_t* a_offset, const float* a, const int64_t* b_offset,
                                             const float* b, void* x, int x_dtype, const int32_t* order, int flags,
                                             int max_refine, double tol, int32_t* info, int32_t* iters,
                                             double* eta) {
  if (int rc = lxa::uneven_check(count, max_n, n, a_offset, a, b_offset, b, x, x_dtype, order, max_refine, info))
    return rc;
  size_t need = 0;
  if (int rc = lxa_chol_uneven_workspace_size(count, &need)) return rc;
  LXA_REQUIRE(need <= lxa::kNoAllocScratchBytes,
              "lxa_chol_uneven_solve_noalloc: needs %zu bytes of scratch, more than its %zu", need,
              lxa::kNoAllocScratchBytes);
  unsigned int* queue = nullptr;
  if (int rc = lxa::noalloc_scratch(&queue)) return rc;
  if (count == 0) return LXA_OK;
  return lxa::uneven_launch(static_cast<hipStream_t>(stream), count, max_n, n, a_offset, a, b_offset, b, x, x_dtype,
                            order, flags, max_refine, tol, info, iters, eta, queue);
}

extern "C" int lxa_chol_uneven_tune_solve(void* stream, int64_t count, int max_n, const int32_t* n,
                                          const int64_t* a_offset, const float* a, const int64_t* b_offset,
                                          const float* b, void* x, int x_dtype, const int32_t* order, int flags,
                                          int max_refine, double tol, int32_t* info, int32_t* iters, double* eta,
                                          void* workspace, size_t workspace_bytes, int max4, int max8) {
  if (int rc = lxa::uneven_check(count, max_n, n, a_offset, a, b_offset, b, x, x_dtype, order, max_refine, info))
    return rc;
  const bool persistent = (flags & LXA_UNEVEN_PERSISTENT) != 0;
  LXA_REQUIRE(!persistent || (workspace && workspace_bytes >= lxa::kUnevenWorkspaceBytes),
              "lxa_chol_uneven_tune_solve: the persistent launch needs a workspace of %zu bytes (got %zu)",
              lxa::kUnevenWorkspaceBytes, workspace ? workspace_bytes : static_cast<size_t>(0));
  if (count == 0) return LXA_OK;
  return lxa::uneven_launch(static_cast<hipStream_t>(stream), count, max_n, n, a_offset, a, b_offset, b, x, x_dtype,
                            order, flags, max_refine, tol, info, iters, eta, static_cast<unsigned int*>(workspace),
                            max4, max8);
}

extern "C" int lxa_chol_uneven_tuned_classes(int* max4, int* max8) {
  LXA_REQUIRE(max4 && max8, "lxa_chol_uneven_tuned_classes: null pointer");
  *max4 = lxa::kTunedMax4;
  *max8 = lxa::kTunedMax8;
  return LXA_OK;
}
