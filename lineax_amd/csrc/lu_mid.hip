// Batched LU (getrf, partial pivoting) and solve (getrs) of orders 65..256,
// one 512-thread workgroup per system.
//
// Factor: right-looking, 16 columns at a time.
//   panel    one wave: lane l holds rows l, l + 64, ... of the panel in
//            registers.  Pivot search by register moves between lanes, pivot
//            row by readlane, no barrier inside the panel.  Interchanges are
//            implicit (every row tracks its LAPACK position); rows are written
//            back at their final positions.
//   columns  one thread per column outside the panel: the panel's net row
//            permutation (pivot rows in, displaced rows out) and, right of it,
//            the product with the inverse of the unit lower 16 x 16 block.
//   update   A22 -= L21 U12 in 16 x 16 tiles on the matrix cores, the type's
//            own products and sums.
// The matrix stays in LDS where it fits (order 199 in float, 141 in double);
// above that it stays in global memory (L2) with L21 and U12 staged in LDS.
// The result is getrf's: factors in place, 0-based interchange sequence, info
// the first exactly zero pivot.
//
// What bounds it: the chain of n pivot searches and broadcasts, about 0.3 us
// each.  One column per global pass of 256 threads, which this replaces, took
// 5 us a column (200 float systems of order 100: 518 us).
#include <climits>
#include <type_traits>

#include "lxa_common.h"

namespace lxa {
namespace {

constexpr int kP = 16;         // panel width
constexpr int kThreads = 512;
constexpr int kWaves = kThreads / kWave;
constexpr int kLpLd = kP + 1;  // row stride of the staged L21

// Order of |v| with NaN largest, in 32-bit words: high, then low.
__device__ __forceinline__ unsigned key_hi(float v) { return __float_as_uint(v) & 0x7fffffffu; }
__device__ __forceinline__ unsigned key_hi(double v) {
  return static_cast<unsigned>(static_cast<unsigned long long>(__double_as_longlong(v)) >> 32) & 0x7fffffffu;
}
__device__ __forceinline__ unsigned key_lo(float) { return 0u; }
__device__ __forceinline__ unsigned key_lo(double v) {
  return static_cast<unsigned>(static_cast<unsigned long long>(__double_as_longlong(v)) & 0xffffffffull);
}

__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
  v = max(v, lane_xor_u32<32>(v));
  v = max(v, lane_xor_u32<16>(v));
  v = max(v, lane_xor_u32<8>(v));
  v = max(v, lane_xor_u32<4>(v));
  v = max(v, lane_xor_u32<2>(v));
  v = max(v, lane_xor_u32<1>(v));
  return v;
}

// S row slots per lane of the panel wave; InLds: the matrix is in LDS.
template <typename T, int S, bool InLds>
__global__ __launch_bounds__(kThreads) void lu_mid_factor_kernel(int n, T* __restrict__ a, int64_t a_stride,
                                                                 int32_t* __restrict__ piv,
                                                                 int32_t* __restrict__ info) {
  using M4 = typename Mma<T>::acc;
  extern __shared__ __align__(16) unsigned char lxa_smem[];
  T* sm = reinterpret_cast<T*>(lxa_smem);
  __shared__ int s_prow[kP];   // original row of the panel's pivot t
  __shared__ int s_disp[kP];   // where row k0 + t goes if it is no pivot, else -1
  __shared__ T s_l11[kP][kP + 1];
  const int64_t sys = blockIdx.x;
  T* A = a + sys * a_stride;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int q = lane & 15, g = lane >> 4;
  const int ld = InLds ? (n | 1) : n;  // odd: rows start in different banks
  T* W = InLds ? sm : A;
  T* Lp = sm;                  // !InLds: [n][kLpLd]
  T* Up = sm + n * kLpLd;      // !InLds: [kP][n + 1]
  if constexpr (InLds) {
    for (int i = wv; i < n; i += kWaves)
      for (int j = lane; j < n; j += kWave) W[i * ld + j] = A[(int64_t)i * n + j];
    __syncthreads();
  }
  int zero_at = 0;
  for (int k0 = 0; k0 < n; k0 += kP) {
    const int w = min(kP, n - k0);
    if (wv == 0) {
      T row[S][kP];
      int pos[S];
      bool done[S];
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int r = lane + kWave * s;
        pos[s] = r;
        done[s] = r < k0 || r >= n;
        const int rc = min(max(r, k0), n - 1);
#pragma unroll
        for (int c = 0; c < kP; ++c) row[s][c] = W[rc * ld + min(k0 + c, n - 1)];
#pragma unroll
        for (int c = 0; c < kP; ++c)
          if (done[s] || c >= w) row[s][c] = T(0);
      }
      static_for<0, kP>([&](auto T_) __attribute__((always_inline)) {
        constexpr int t = decltype(T_)::value;
        if (t >= w) return;  // uniform
        // largest |a_ik| over the remaining rows, ties to the smallest position
        unsigned kh = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) kh = max(kh, done[s] ? 0u : key_hi(row[s][t]));
        const unsigned mh = __builtin_amdgcn_readfirstlane(wave_max_u32(kh));
        bool cand[S];
        int hits = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
          cand[s] = !done[s] && key_hi(row[s][t]) == mh;
          hits += __popcll(__ballot(cand[s]));
        }
        if (hits > 1) {  // uniform
          if constexpr (sizeof(T) == 8) {
            unsigned kl = 0;
#pragma unroll
            for (int s = 0; s < S; ++s) kl = max(kl, cand[s] ? key_lo(row[s][t]) : 0u);
            const unsigned ml = __builtin_amdgcn_readfirstlane(wave_max_u32(kl));
#pragma unroll
            for (int s = 0; s < S; ++s) cand[s] = cand[s] && key_lo(row[s][t]) == ml;
          }
          unsigned near = 0;  // positions below 2^15, so the largest complement is the smallest position
#pragma unroll
          for (int s = 0; s < S; ++s) near = max(near, cand[s] ? 0x7fffu - (unsigned)pos[s] : 0u);
          const unsigned best = __builtin_amdgcn_readfirstlane(wave_max_u32(near));
#pragma unroll
          for (int s = 0; s < S; ++s) cand[s] = cand[s] && 0x7fffu - (unsigned)pos[s] == best;
        }
        int cp = 0;
        T pv[kP];
#pragma unroll
        for (int c = 0; c < kP; ++c) pv[c] = T(0);
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const unsigned long long b = __ballot(cand[s]);
          if (b) {  // uniform: exactly one slot of one lane
            const int L = __ffsll(b) - 1;
            cp = __builtin_amdgcn_readlane(pos[s], L);
#pragma unroll
            for (int c = t; c < kP; ++c) pv[c] = from_lane(row[s][c], L);
          }
        }
        const T pval = pv[t];
        if (pval == T(0) && zero_at == 0) zero_at = k0 + t + 1;
        if (lane == 0) piv[sys * n + k0 + t] = cp;
        const bool fast = plain_range(pval);
        const T rp = T(1) / pval;
#pragma unroll
        for (int s = 0; s < S; ++s) {
          if (cand[s]) {
            pos[s] = k0 + t;
            done[s] = true;
          } else if (!done[s] && pos[s] == k0 + t) {
            pos[s] = cp;
          }
          T l = row[s][t];
          if (fast) {
            l = divide(l, pval, rp);
          } else if (pval != T(0)) {
            l = l / pval;
          }
          if (!done[s]) {
            row[s][t] = l;
#pragma unroll
            for (int c = t + 1; c < kP; ++c) row[s][c] -= l * pv[c];
          }
        }
      });
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int r = lane + kWave * s;
        if (r >= k0 && r < n) {
#pragma unroll
          for (int c = 0; c < kP; ++c) {
            if (c < w) W[pos[s] * ld + k0 + c] = row[s][c];
            if constexpr (!InLds) Lp[pos[s] * kLpLd + c] = row[s][c];
          }
          if (pos[s] < k0 + w) {
            s_prow[pos[s] - k0] = r;
#pragma unroll
            for (int c = 0; c < kP; ++c) s_l11[pos[s] - k0][c] = row[s][c];
          }
          if (r < k0 + w) s_disp[r - k0] = pos[s] < k0 + w ? -1 : pos[s];
        }
      }
    }
    __syncthreads();
    // ---- columns outside the panel (w < kP only in the last panel, which
    // has none on its right)
    for (int c = tid; c < n; c += kThreads) {
      if (c >= k0 && c < k0 + w) continue;
      T v[kP], d[kP];
#pragma unroll
      for (int t = 0; t < kP; ++t) {
        const int tt = min(t, w - 1);
        v[t] = W[s_prow[tt] * ld + c];
        d[t] = W[(k0 + tt) * ld + c];
      }
      if (c >= k0 + w) {
        static_for<0, kP>([&](auto T_) __attribute__((always_inline)) {
          constexpr int t = decltype(T_)::value;
#pragma unroll
          for (int i = t + 1; i < kP; ++i) v[i] -= s_l11[i][t] * v[t];
          // one column of the block in flight at a time (all 120 entries
          // loaded ahead would not fit the registers)
          __builtin_amdgcn_sched_barrier(0);
        });
      }
#pragma unroll
      for (int t = 0; t < kP; ++t) {
        if (t < w) {
          const int to = s_disp[t];
          if (to >= 0) W[to * ld + c] = d[t];
          W[(k0 + t) * ld + c] = v[t];
          if constexpr (!InLds) Up[t * (n + 1) + c] = v[t];
        }
      }
    }
    __syncthreads();
    // ---- A22 -= L21 U12: waves take 16-row strips and up to four 16-column
    // tiles of them at a time
    const int base = k0 + kP, rest = n - base;
    if (rest > 0) {
      const int T16 = (rest + 15) / 16, C4 = (T16 + 3) / 4;
      for (int item = wv; item < T16 * C4; item += kWaves) {
        const int rt = item / C4, ct = 4 * (item % C4);
        M4 acc[4];
        const int r0 = base + 16 * rt;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int col = min(base + 16 * (ct + u) + q, n - 1);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[u][e] = W[min(r0 + Mma<T>::row(g, e), n - 1) * ld + col];
        }
        const int lr = min(r0 + q, n - 1);
#pragma unroll
        for (int h = 0; h < kP; h += 4) {
          const T av = -(InLds ? W[lr * ld + k0 + h + g] : Lp[lr * kLpLd + h + g]);
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int col = min(base + 16 * (ct + u) + q, n - 1);
            const T bv = InLds ? W[(k0 + h + g) * ld + col] : Up[(h + g) * (n + 1) + col];
            acc[u] = Mma<T>::mul(av, bv, acc[u]);
          }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int col = base + 16 * (ct + u) + q;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = r0 + Mma<T>::row(g, e);
            if (r < n && col < n) W[r * ld + col] = acc[u][e];
          }
        }
      }
    }
    __syncthreads();
  }
  if constexpr (InLds) {
    for (int i = wv; i < n; i += kWaves)
      for (int j = lane; j < n; j += kWave) A[(int64_t)i * n + j] = W[i * ld + j];
  }
  if (tid == 0) info[sys] = zero_at;
}

// ---------------------------------------------------------------------------
// Solve: one 256-thread workgroup per system, thread i owns unknown i.  Both
// triangles go block by block (16 unknowns): the wave that owns the block
// runs its chain with the multipliers in registers (they are that wave's
// own entries of the block's columns), the other waves then subtract the
// block's products; the next block's entries are loaded meanwhile.
// ---------------------------------------------------------------------------
constexpr int kSolveThreads = 256;

template <typename T>
__global__ __launch_bounds__(kSolveThreads) void lu_mid_solve_kernel(int n, const T* __restrict__ lu,
                                                                     int64_t lu_stride,
                                                                     const int32_t* __restrict__ piv,
                                                                     int64_t piv_stride, T* __restrict__ b,
                                                                     int64_t b_stride, int trans) {
  __shared__ T ys[kSolveThreads];
  __shared__ int pv[kSolveThreads];
  const int64_t sys = blockIdx.x;
  const T* A = lu + sys * lu_stride;
  T* B = b + sys * b_stride;
  const int i = threadIdx.x, wv = i >> 6;
  const bool in = i < n;
  const int ic = min(i, n - 1);
  const int blocks = (n + kP - 1) / kP;
  const T diag = A[(int64_t)ic * n + ic];
  T y = in ? B[i] : T(0);
  int q = i;
  if (in) {
    q = piv[sys * piv_stride + i];
    q = q < 0 ? 0 : (q >= n ? n - 1 : q);
  }
  pv[i] = q;
  __syncthreads();
  if (!trans) {
    // where the interchanges take entry i
    int p = i;
    for (int k = 0; k < n; ++k) {
      const int o = pv[k];
      p = (p == k) ? o : ((p == o) ? k : p);
    }
    if (in) ys[p] = y;
    __syncthreads();
    y = in ? ys[i] : T(0);
    __syncthreads();
  }
  const T rdiag = T(1) / diag;
  bool fast = __all(plain_range(diag));

  // entries that couple unknown i to the 16 unknowns of block p
  auto fetch = [&](int p, T (&v)[kP]) {
#pragma unroll
    for (int j = 0; j < kP; ++j) {
      const int c = p * kP + j, cc = min(c, n - 1);
      const T e = trans ? A[(int64_t)cc * n + ic] : A[(int64_t)ic * n + cc];
      v[j] = c < n ? e : T(0);
    }
  };
  // one triangle; Up: ascending blocks, unknowns after the block are updated
  auto sweep = [&](auto Up_, auto Div_) __attribute__((always_inline)) {
    constexpr bool Up = decltype(Up_)::value, Div = decltype(Div_)::value;
    T v[kP], nx[kP];
    fetch(Up ? 0 : blocks - 1, nx);
    for (int s = 0; s < blocks; ++s) {
      const int p = Up ? s : blocks - 1 - s;
      const int r0 = p * kP;
#pragma unroll
      for (int j = 0; j < kP; ++j) v[j] = nx[j];
      if (s + 1 < blocks) fetch(Up ? p + 1 : p - 1, nx);
      if (wv == r0 >> 6) {
        const int l0 = r0 & 63;
#pragma unroll
        for (int u = 0; u < kP; ++u) {
          const int j = Up ? u : kP - 1 - u;
          if (Div && i == r0 + j) y = in ? (fast ? divide(y, diag, rdiag) : y / diag) : T(0);
          const T yj = from_lane(y, l0 + j);
          if (Up ? i > r0 + j : i < r0 + j) y -= v[j] * yj;
        }
        if (i >= r0 && i < r0 + kP) ys[i] = y;
      }
      lds_barrier();
      if (Up ? wv > (r0 >> 6) : wv < (r0 >> 6)) {
#pragma unroll
        for (int j = 0; j < kP; ++j) y -= v[j] * ys[r0 + j];
      }
    }
    __syncthreads();
  };
  using Yes = std::true_type;
  using No = std::false_type;
  const T rhs = y;
  while (true) {
    if (!trans) {
      sweep(Yes{}, No{});   // L y = P b
      sweep(No{}, Yes{});   // U x = y
    } else {
      sweep(Yes{}, Yes{});  // U^T z = b
      sweep(No{}, No{});    // L^T w = z
    }
    // NaN may be an infinite quotient: once more with divisions
    if (!__syncthreads_or(fast && in && y != y)) break;
    fast = false;
    y = rhs;
  }
  int p = i;
  if (trans) {
    for (int k = n - 1; k >= 0; --k) {
      const int o = pv[k];
      p = (p == k) ? o : ((p == o) ? k : p);
    }
  }
  if (in) B[p] = y;  // every read of B is behind the barriers above
}

template <typename T, int S, bool InLds>
int factor_launch(hipStream_t st, int64_t batch, int n, T* a, int64_t stride, int32_t* piv, int32_t* info,
                  size_t smem) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&lu_mid_factor_kernel<T, S, InLds>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  if (e != hipSuccess) return hip_error(e, "hipFuncSetAttribute(lu_mid_factor_kernel)");
  lu_mid_factor_kernel<T, S, InLds><<<dim3((unsigned)batch), kThreads, smem, st>>>(n, a, stride, piv, info);
  LXA_LAUNCH_CHECK("lu_mid_factor_kernel");
  return LXA_OK;
}

template <typename T>
int factor_t(hipStream_t st, int64_t batch, int n, T* a, int64_t stride, int32_t* piv, int32_t* info) {
  const size_t whole = sizeof(T) * (size_t)n * (n | 1);
  const size_t staged = sizeof(T) * ((size_t)n * kLpLd + (size_t)kP * (n + 1));
  // the rest of the 160 KiB holds the 16 x 16 block and the row lists
  if (whole <= 160 * 1024 - 3 * 1024) {
    if (n <= 128) return factor_launch<T, 2, true>(st, batch, n, a, stride, piv, info, whole);
    if (n <= 192) return factor_launch<T, 3, true>(st, batch, n, a, stride, piv, info, whole);
    return factor_launch<T, 4, true>(st, batch, n, a, stride, piv, info, whole);
  }
  if (n <= 192) return factor_launch<T, 3, false>(st, batch, n, a, stride, piv, info, staged);
  return factor_launch<T, 4, false>(st, batch, n, a, stride, piv, info, staged);
}

template <typename T>
int solve_t(hipStream_t st, int64_t batch, int n, const T* lu, int64_t lus, const int32_t* piv, int64_t ps, T* b,
            int64_t bs, int trans) {
  lu_mid_solve_kernel<T><<<dim3((unsigned)batch), kSolveThreads, 0, st>>>(n, lu, lus, piv, ps, b, bs, trans);
  LXA_LAUNCH_CHECK("lu_mid_solve_kernel");
  return LXA_OK;
}

}  // namespace

int lu_mid_factor(hipStream_t s, int64_t batch, int n, float* a, int64_t stride, int32_t* piv, int32_t* info) {
  return factor_t<float>(s, batch, n, a, stride, piv, info);
}
int lu_mid_factor(hipStream_t s, int64_t batch, int n, double* a, int64_t stride, int32_t* piv, int32_t* info) {
  return factor_t<double>(s, batch, n, a, stride, piv, info);
}
int lu_mid_solve(hipStream_t s, int64_t batch, int n, const float* lu, int64_t lus, const int32_t* piv, int64_t ps,
                 float* b, int64_t bs, int trans) {
  return solve_t<float>(s, batch, n, lu, lus, piv, ps, b, bs, trans);
}
int lu_mid_solve(hipStream_t s, int64_t batch, int n, const double* lu, int64_t lus, const int32_t* piv, int64_t ps,
                 double* b, int64_t bs, int trans) {
  return solve_t<double>(s, batch, n, lu, lus, piv, ps, b, bs, trans);
}

}  // namespace lxa
