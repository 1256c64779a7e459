// Householder QR over uneven batches (geqrf / ormqr) and triangular solves
// for gfx950.
//
// Factorisation (lxa_qr_factor) is blocked, right-looking, compact WY, 16
// columns at a time, one launch per panel (qr_step_kernel).  A 512-thread
// workgroup owns 16 columns of one system and all their rows, in registers in
// the layout of the matrix cores' results:
//   update  C <- (I - V T V^T)^T C: W = V^T C, T^T W and C - V (T^T W) are
//           matrix-core products whose inner index is permuted so that a
//           result register is an operand register of the next product; C is
//           read and written once per panel.
//   panel   the workgroup that updated the columns next to the panel factors
//           them at once, while the others are still updating theirs.  Lane
//           q of each 16-lane row holds column q, so the products of column j
//           with all others are one multiply-add per element (column j by a
//           DPP row broadcast), the sum over a wave is two exchanges, and one
//           barrier per column carries products, norm and diagonal row.
// Panels taller than 4096 rows are factored from global memory by
// qr_panel_kernel and updated in two sweeps over C.
//
// The panel's chain of columns bounds single and small batches (29 us a panel
// at up to 512 rows, 64 us at 3001 double rows, 76 us at 4000 float rows, one
// barrier and two passes over the registers a column), HBM the large ones.  With a
// launch each for panel, partial products, their sum and the update, 256
// float systems of 512 x 256 took 1490 us; they take 940 us here.
//
// Reference: lineax/_solver/qr.py:55-92 calls jnp.linalg.qr(mode="raw")
// (geqrf), jax.lax.linalg.ormqr and jax.scipy.linalg.solve_triangular; the
// reflector convention here is LAPACK's (larfg: beta = -sign(alpha) ||x||,
// tau = (beta - alpha) / beta, v = x / (alpha - beta), tau = 0 when x = 0).

#include "qr_step.h"

namespace lxa {
namespace {

constexpr int kBigThreads = 1024;    // apply / triangular solve workgroups
constexpr int kBigWaves = kBigThreads / kWave;

// Block sum of K values per thread over a workgroup of WAVES waves.
// stage: LDS [WAVES][K]; out: LDS [K].  Every thread gets the sums.
template <int K, int WAVES, typename R>
__device__ __forceinline__ void block_sum(R (&v)[K], R* stage, R* out, int tid) {
  const int lane = tid & (kWave - 1);
  const int wv = tid >> 6;
  const R x = wave_reduce_scatter<K>(v, lane);
  constexpr int kShift = 6 - Log2<K>::value;
  if ((lane & ((1 << kShift) - 1)) == 0) stage[wv * K + (lane >> kShift)] = x;
  __syncthreads();
  if (tid < K) {
    R s = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) s += stage[w * K + tid];
    out[tid] = s;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < K; ++i) v[i] = out[i];
}

// Two block sums (K1 values of type R1, K2 of type R2 per thread) behind one
// pair of barriers: the second array's cross-wave pass runs on another wave.
template <int K1, int K2, int WAVES, typename R1, typename R2>
__device__ __forceinline__ void block_sum2(R1 (&u)[K1], R1* stage1, R1* out1, R2 (&v)[K2], R2* stage2, R2* out2,
                                           int tid) {
  static_assert(WAVES >= 2, "the two cross-wave passes run on waves 0 and 1");
  const int lane = tid & (kWave - 1);
  const int wv = tid >> 6;
  const R1 x1 = wave_reduce_scatter<K1>(u, lane);
  const R2 x2 = wave_reduce_scatter<K2>(v, lane);
  constexpr int kShift1 = 6 - Log2<K1>::value, kShift2 = 6 - Log2<K2>::value;
  if ((lane & ((1 << kShift1) - 1)) == 0) stage1[wv * K1 + (lane >> kShift1)] = x1;
  if ((lane & ((1 << kShift2) - 1)) == 0) stage2[wv * K2 + (lane >> kShift2)] = x2;
  __syncthreads();
  if (tid < K1) {
    R1 t = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) t += stage1[w * K1 + tid];
    out1[tid] = t;
  } else if (tid >= kWave && tid < kWave + K2) {
    R2 t = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) t += stage2[w * K2 + tid - kWave];
    out2[tid - kWave] = t;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < K1; ++i) u[i] = out1[i];
#pragma unroll
  for (int i = 0; i < K2; ++i) v[i] = out2[i];
}

// ---------------------------------------------------------------------------
// Panel factorisation with the rows in global memory (any height).  One pass a
// column: a row is updated by the column's reflector and its products for the
// next column are taken while it is in registers.  What a column reads and
// writes through the caches bounds it: a double system of 10000 x 60 takes 4618
// us a call, 5455 with a pass for the products and one for the update.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kPanelThreads) void qr_panel_kernel(const lxa_qr_desc* __restrict__ descs, int k_all,
                                                                 const int32_t* __restrict__ kcol,
                                                                 T* __restrict__ a, T* __restrict__ tau,
                                                                 T* __restrict__ tblk) {
  constexpr int NB = QrCfg<T>::NB;
  constexpr int KW = NB;  // width of the per-column dot reduction (>= NB - 1)
  __shared__ double s_stage2[kPanelWaves];
  __shared__ double s_out2[1];
  __shared__ T s_stage[kPanelWaves * KW];
  __shared__ T s_out[KW];
  __shared__ T s_diag[2][NB];  // the diagonal row of the current column
  __shared__ T s_g[NB][NB];    // s_g[a][j] = v_a^T v_j, a < j

  const lxa_qr_desc d = descs[blockIdx.x];
  const int m = d.m, n = d.n, lda = d.lda;
  const int kmax = min(m, n);
  const int kc = kcol ? kcol[blockIdx.x] : 0;
  if (kc >= kmax - k_all) return;  // no sum here: a system that is done may say so by any large column
  const int k = kc + k_all;
  const int nb = min(NB, kmax - k);
  const int tid = threadIdx.x;
  T* A = a + d.a_offset;
  const int nr = (m - k + kPanelThreads - 1) / kPanelThreads;
  // a row's panel entries, all loads unconditional where the panel is whole
  // (a test per column had made each wait for the one before)
  auto load_row = [&](int row, T (&v)[NB]) {
    const T* p = A + (int64_t)row * lda + k;
    if (nb == NB) {
#pragma unroll
      for (int c = 0; c < NB; ++c) v[c] = p[c];
    } else {
#pragma unroll
      for (int c = 0; c < NB; ++c) v[c] = c < nb ? p[c] : T(0);
    }
  };

  // sums over the rows below column c's diagonal: with x = column c there,
  // ||x||^2 and the raw products x^T A(:, i) with the panel's other columns
  double nv[1] = {0.0};
  T dots[KW];
#pragma unroll
  for (int c = 0; c < KW; ++c) dots[c] = T(0);
  auto add_row = [&](auto C_, int row, const T (&v)[NB]) __attribute__((always_inline)) {
    constexpr int c = decltype(C_)::value;
    const T x = row < m && row > k + c ? v[c] : T(0);
    nv[0] += (double)x * (double)x;
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if (i != c) dots[i] += x * v[i];
  };
  // f(row, entries) for this thread's rows, two rows' loads ahead of either's use
  auto each_row = [&](auto&& f) __attribute__((always_inline)) {
    for (int r = 0; r < nr; r += 2) {
      const int row0 = k + tid + r * kPanelThreads, row1 = row0 + kPanelThreads;
      T v0[NB], v1[NB];
      load_row(min(row0, m - 1), v0);
      load_row(min(row1, m - 1), v1);
      f(row0, v0);
      f(row1, v1);
    }
  };
  each_row([&](int row, T (&v)[NB]) __attribute__((always_inline)) {
    add_row(std::integral_constant<int, 0>{}, row, v);
  });

  T taus[NB];
  // the column loop at compile time (every register index a constant)
  static_for<0, NB>([&](auto J_) __attribute__((always_inline)) {
    constexpr int j = decltype(J_)::value;
    taus[j] = T(0);
    if (j >= nb) return;  // uniform
    const int diag = k + j;
    // ---- one block reduction per column; the diagonal row goes to LDS (thread
    // j holds it).  v = [1; x / (alpha - beta)] then gives
    //   v^T A(:, c)  = A(diag, c) + scale * x^T A(:, c)    (c > j, larf)
    //   v_c^T v      = v_c(diag)  + scale * v_c^T x        (c < j, larft)
    // so the norm and the products share one pair of barriers.
    T* sd = s_diag[j & 1];  // double-buffered: readers of column j - 1 may lag
    if (tid == j) {
#pragma unroll
      for (int c = 0; c < NB; ++c) sd[c] = c < nb ? A[(int64_t)diag * lda + k + c] : T(0);
    }
    block_sum2<1, KW, kPanelWaves>(nv, s_stage2, s_out2, dots, s_stage, s_out, tid);
    const double ss = nv[0], alpha = (double)sd[j];
    T tj = T(0), beta = (T)alpha, scale = T(1);
    if (ss != 0.0) {
      const double bd = -copysign(sqrt(alpha * alpha + ss), alpha);
      beta = (T)bd;
      tj = (T)((bd - alpha) / bd);
      scale = (T)(1.0 / (alpha - bd));
    }
    taus[j] = tj;
    T acc[KW];
#pragma unroll
    for (int c = 0; c < KW; ++c) acc[c] = (c != j && c < nb) ? sd[c] + scale * dots[c] : T(0);
    if (tid == 0) {
#pragma unroll
      for (int c = 0; c < NB; ++c)
        if (c < j) s_g[c][j] = acc[c];
    }
    nv[0] = 0.0;
#pragma unroll
    for (int c = 0; c < KW; ++c) dots[c] = T(0);
    // ---- scale x into v, put beta on the diagonal, apply (I - tau v v^T) to
    // the panel columns right of j, and take the next column's sums
    each_row([&](int row, T (&v)[NB]) __attribute__((always_inline)) {
      if (row < m && row >= diag) {
        T* p = A + (int64_t)row * lda + k;
        const T vj = row > diag ? v[j] * scale : T(1);
        if (row == diag) {
          p[j] = beta;
        } else if (ss != 0.0) {
          p[j] = vj;
        }
        v[j] = vj;
        if (tj != T(0)) {
          const T tv = tj * vj;
#pragma unroll
          for (int c = j + 1; c < NB; ++c) v[c] -= tv * acc[c];
          if (nb == NB) {
#pragma unroll
            for (int c = j + 1; c < NB; ++c) p[c] = v[c];
          } else {
#pragma unroll
            for (int c = j + 1; c < NB; ++c)
              if (c < nb) p[c] = v[c];
          }
        }
      }
      if constexpr (j + 1 < NB) add_row(std::integral_constant<int, j + 1>{}, row, v);
    });
  });
  __syncthreads();  // s_g complete

  // ---- T (larft, forward, columnwise): lane a owns row a of T.
  if (tid < NB) {
    const int ra = tid;
    T trow[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      T v = T(0);
      if (i < nb) {
        if (ra == i) {
          v = taus[i];
        } else if (ra < i) {
          T s = T(0);
#pragma unroll
          for (int b = 0; b < NB; ++b)
            if (b >= ra && b < i) s += trow[b] * s_g[b][i];
          v = -taus[i] * s;
        }
      }
      trow[i] = v;
    }
    T* Tp = tblk + d.t_offset + (int64_t)(k / NB) * NB * NB + ra * NB;
#pragma unroll
    for (int i = 0; i < NB; ++i) Tp[i] = trow[i];
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if (i == ra && i < nb) tau[d.tau_offset + k + i] = taus[i];
  }
}

// ---------------------------------------------------------------------------
// b <- Q^T b (trans) or Q b: one workgroup per (system, right-hand side),
// panel by panel: w = V^T b; w = T^T w (or T w); b -= V w.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kBigThreads) void qr_apply_kernel(const lxa_qr_desc* __restrict__ descs,
                                                                 const T* __restrict__ a,
                                                                 const T* __restrict__ tblk, T* __restrict__ b,
                                                                 int trans) {
  constexpr int NB = QrCfg<T>::NB;
  __shared__ T s_stage[kBigWaves * NB];
  __shared__ T s_out[NB];
  __shared__ T s_w[NB];
  const lxa_qr_desc d = descs[blockIdx.x];
  const int m = d.m, n = d.n, lda = d.lda;
  const int kmax = min(m, n);
  if (kmax <= 0) return;
  const int tid = threadIdx.x;
  const T* A = a + d.a_offset;
  T* x = b + d.b_offset + (int64_t)blockIdx.y * d.ldb;
  const int panels = (kmax + NB - 1) / NB;
  for (int q = 0; q < panels; ++q) {
    const int p = trans ? q : panels - 1 - q;
    const int k = p * NB;
    const int nb = min(NB, kmax - k);
    T acc[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[j] = T(0);
    for (int row = k + tid; row < m; row += kBigThreads) {
      const T xv = x[row];
      const T* Ar = A + (int64_t)row * lda + k;
#pragma unroll
      for (int j = 0; j < NB; ++j)
        if (j < nb) acc[j] += vpick(row, k + j, Ar[j]) * xv;
    }
    block_sum<NB, kBigWaves>(acc, s_stage, s_out, tid);
    if (tid < NB) {
      const T* Tp = tblk + d.t_offset + (int64_t)p * NB * NB;
      T s = T(0);
      if (trans) {  // (T^T w)_tid = sum_{i <= tid} T[i][tid] w_i
#pragma unroll
        for (int i = 0; i < NB; ++i)
          if (i <= tid) s += Tp[i * NB + tid] * acc[i];
      } else {  // (T w)_tid = sum_{i >= tid} T[tid][i] w_i
#pragma unroll
        for (int i = 0; i < NB; ++i)
          if (i >= tid) s += Tp[tid * NB + i] * acc[i];
      }
      s_w[tid] = s;
    }
    __syncthreads();
    T w[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) w[j] = s_w[j];
    for (int row = k + tid; row < m; row += kBigThreads) {
      const T* Ar = A + (int64_t)row * lda + k;
      T s = T(0);
#pragma unroll
      for (int j = 0; j < NB; ++j)
        if (j < nb) s += vpick(row, k + j, Ar[j]) * w[j];
      x[row] -= s;
    }
    __syncthreads();  // x rows are re-read by other threads in the next panel
  }
}

// ---------------------------------------------------------------------------
// The same product for systems of up to kApplyMaxRows rows, one vector per
// workgroup: the vector lives in LDS and NB lanes share a row (lane j reads
// column j of the panel, so a wave load covers 64 / NB contiguous row
// segments instead of 64 scattered ones).  Each lane keeps its entries of the
// first RPT passes' rows in registers between the reduction and the update;
// REST: there may be further rows, which are read twice.  Per panel:
//   w = V^T x (lanes of a column, then waves, summed in a fixed order);
//   w = T^T w or T w (wave 0, shuffles);  x -= V w (row sums of 8 or 16 rows
//   at a time by a reduce-scatter over their 16 lanes).
// One compute unit reading V bounds it.  A double system of 3001 x 391: 429 us;
// all rows read twice with a four-step butterfly per row 764 us.
// ---------------------------------------------------------------------------
constexpr int kApplyMaxRows = 16384;

// Sums K values (K a power of two <= 16) over the 16 lanes of a row; lane j
// of the row holds the sum of value j / (16 / K).  v is destroyed.
template <int K, int L = 0, typename T>
__device__ __forceinline__ T row_reduce_scatter(T (&v)[K], int j) {
  constexpr int off = 8 >> L, half = K >> (L + 1);
  if constexpr (off == 0) {
    return v[0];
  } else if constexpr (half >= 1) {
    const bool upper = (j & off) != 0;
#pragma unroll
    for (int i = 0; i < half; ++i) {
      const T keep = upper ? v[i + half] : v[i];
      const T send = upper ? v[i] : v[i + half];
      v[i] = keep + lane_xor<off>(send);
    }
    return row_reduce_scatter<K, L + 1>(v, j);
  } else {
    v[0] += lane_xor<off>(v[0]);
    return row_reduce_scatter<K, L + 1>(v, j);
  }
}

template <typename T, int RPT, bool REST>
__global__ __launch_bounds__(kBigThreads) void qr_apply_rows_kernel(const lxa_qr_desc* __restrict__ descs,
                                                                    const T* __restrict__ a,
                                                                    const T* __restrict__ tblk,
                                                                    T* __restrict__ b, int trans) {
  constexpr int NB = QrCfg<T>::NB;
  constexpr int G = kWave / NB;       // rows per wave load
  constexpr int RP = kBigWaves * G;   // rows per pass of the workgroup
  extern __shared__ __align__(16) unsigned char apply_smem[];
  T* xs = reinterpret_cast<T*>(apply_smem);
  __shared__ T s_part[kBigWaves][NB];
  __shared__ T s_w[NB];
  const lxa_qr_desc d = descs[blockIdx.x];
  const int m = d.m, lda = d.lda;
  const int kmax = min(m, d.n);
  if (kmax <= 0) return;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid >> 6;
  const int j = lane % NB, rg = wv * G + lane / NB;
  const T* A = a + d.a_offset;
  T* x = b + d.b_offset + (int64_t)blockIdx.y * d.ldb;
  for (int i = tid; i < m; i += kBigThreads) xs[i] = x[i];
  __syncthreads();
  const int panels = (kmax + NB - 1) / NB;
  T v[RPT > 0 ? RPT : 1];
  for (int q = 0; q < panels; ++q) {
    const int p = trans ? q : panels - 1 - q;
    const int k = p * NB;
    const int nb = min(NB, kmax - k);
    const int jc = min(j, nb - 1);  // clamped column: loads stay inside the panel
    const T* Ak = A + k + jc;
    // wave 0's row (trans) or column of the panel's T block, loaded now so
    // the loads overlap the reduction below instead of one wait per term
    T tv[NB];
    if (wv == 0) {
      const T* Tp = tblk + d.t_offset + (int64_t)p * NB * NB;
      const int lt = min(lane, NB - 1);
#pragma unroll
      for (int i = 0; i < NB; ++i) tv[i] = trans ? Tp[i * NB + lt] : Tp[lt * NB + i];
    }
    T acc = T(0);
    if constexpr (RPT > 0) {
#pragma unroll
      for (int t = 0; t < RPT; ++t) {
        const int row = k + rg + t * RP;
        const T st = Ak[(int64_t)min(row, m - 1) * lda];
        v[t] = (row < m && j < nb) ? vpick(row, k + j, st) : T(0);
        if (t % 16 == 15) __builtin_amdgcn_sched_barrier(0);  // addresses of 16 rows at a time
      }
#pragma unroll
      for (int t = 0; t < RPT; ++t) {
        const int row = k + rg + t * RP;
        if (row < m) acc += v[t] * xs[row];
      }
    }
    if constexpr (REST) {
      // eight rows per round, loads issued together (clamped rows, masked)
      for (int row0 = k + rg + RPT * RP; row0 < m; row0 += 8 * RP) {
        T st[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) st[u] = Ak[(int64_t)min(row0 + u * RP, m - 1) * lda];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int row = row0 + u * RP;
          if (row < m && j < nb) acc += vpick(row, k + j, st[u]) * xs[row];
        }
      }
    }
#pragma unroll
    for (int off = NB; off < kWave; off <<= 1) acc += __shfl_xor(acc, off, kWave);
    if (lane < NB) s_part[wv][lane] = acc;
    __syncthreads();
    if (wv == 0) {
      T wsum = T(0);
      if (lane < NB) {
#pragma unroll
        for (int w = 0; w < kBigWaves; ++w) wsum += s_part[w][lane];
      }
      T s = T(0);
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const T wi = __shfl(wsum, i, kWave);
        if (lane < NB && i < nb && lane < nb) {
          if (trans) {  // (T^T w)_lane = sum_{i <= lane} T[i][lane] w_i
            if (i <= lane) s += tv[i] * wi;
          } else {  // (T w)_lane = sum_{i >= lane} T[lane][i] w_i
            if (i >= lane) s += tv[i] * wi;
          }
        }
      }
      if (lane < NB) s_w[lane] = s;
    }
    __syncthreads();
    const T wj = s_w[j];
    if constexpr (RPT > 0) {
      constexpr int K = RPT < NB ? RPT : NB;
#pragma unroll
      for (int t0 = 0; t0 < RPT; t0 += K) {
        T s[K];
#pragma unroll
        for (int t = 0; t < K; ++t) s[t] = v[t0 + t] * wj;
        const T sum = row_reduce_scatter<K>(s, j);
        const int row = k + rg + (t0 + j / (NB / K)) * RP;
        if (j % (NB / K) == 0 && row < m) xs[row] -= sum;
      }
    }
    if constexpr (REST) {
      for (int row0 = k + rg + RPT * RP; row0 < m; row0 += 8 * RP) {
        T st[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) st[u] = Ak[(int64_t)min(row0 + u * RP, m - 1) * lda];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int row = row0 + u * RP;
          st[u] = (row < m && j < nb) ? vpick(row, k + j, st[u]) * wj : T(0);
        }
        const T sum = row_reduce_scatter<8>(st, j);
        const int row = row0 + j / 2 * RP;
        if (j % 2 == 0 && row < m) xs[row] -= sum;
      }
    }
    __syncthreads();
  }
  for (int i = tid; i < m; i += kBigThreads) x[i] = xs[i];
}

template <typename T, int RPT, bool REST>
int launch_apply_rows(hipStream_t st, dim3 grid, int max_m, const lxa_qr_desc* desc, const void* a, const void* tblk,
                      void* b, int trans) {
  const size_t smem = sizeof(T) * (size_t)max_m;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&qr_apply_rows_kernel<T, RPT, REST>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  if (e != hipSuccess) return hip_error(e, "hipFuncSetAttribute(qr_apply_rows)");
  qr_apply_rows_kernel<T, RPT, REST><<<grid, kBigThreads, smem, st>>>(
      desc, static_cast<const T*>(a), static_cast<const T*>(tblk), static_cast<T*>(b), trans);
  LXA_LAUNCH_CHECK("qr_apply_rows_kernel");
  return LXA_OK;
}

template <typename T>
int apply_rows(hipStream_t st, dim3 grid, int max_m, const lxa_qr_desc* desc, const void* a, const void* tblk,
               void* b, int trans) {
  // 16 waves of 128 registers hold 16 panel entries a lane, 1024 rows; a system
  // of 1500 x 391 takes 131 us (float) / 223 us (double) so, 167 / 290 us with
  // 64 entries in eight waves, of 3001 rows 288 / 429 us and, with the 128 / 96
  // entries that eight waves cannot hold, 574 / 674 us.  Above 4096 rows the
  // 1024 are too few to matter: 8000 x 100 185 / 290 us with them, 171 / 288 us
  // without.
  constexpr int kPass = 16 * (kWave / QrCfg<T>::NB);  // rows per pass of 16 waves
  if (max_m <= 4 * kPass) return launch_apply_rows<T, 4, false>(st, grid, max_m, desc, a, tblk, b, trans);
  if (max_m <= 8 * kPass) return launch_apply_rows<T, 8, false>(st, grid, max_m, desc, a, tblk, b, trans);
  if (max_m <= 16 * kPass) return launch_apply_rows<T, 16, false>(st, grid, max_m, desc, a, tblk, b, trans);
  if (max_m <= 4096) return launch_apply_rows<T, 16, true>(st, grid, max_m, desc, a, tblk, b, trans);
  return launch_apply_rows<T, 0, true>(st, grid, max_m, desc, a, tblk, b, trans);
}

// ---------------------------------------------------------------------------
// Triangular solve with an upper triangular R, R[i][j] = a[i*rs + j*cs]:
// back substitution for R x = y (tr = 0), forward for R^T x = y (tr = 1).
// One workgroup per (system, right-hand side); x lives in LDS; 64-row
// blocks: a parallel product with the solved part, then one wave solves the
// diagonal block from an LDS copy of it.
// ---------------------------------------------------------------------------
constexpr int kTrsvBlock = 64;
constexpr int kTrsvMaxK = 8192;

template <typename T>
__global__ __launch_bounds__(kBigThreads) void trsv_kernel(const lxa_qr_desc* __restrict__ descs,
                                                             const T* __restrict__ a, T* __restrict__ b, int lower,
                                                             int trans, int unit_diag) {
  extern __shared__ __align__(16) unsigned char trsv_smem[];
  T* xs = reinterpret_cast<T*>(trsv_smem);                      // [kTrsvMaxK] (only k used)
  T* tile = xs + ((kTrsvMaxK + 1) & ~1);                        // [64][65]
  T* red = tile + kTrsvBlock * (kTrsvBlock + 1);                // [16][64]
  T* rinv = red + kBigWaves * kWave;                            // [64] reciprocal diagonal
  const lxa_qr_desc d = descs[blockIdx.x];
  const int kk = min(d.m, d.n);
  if (kk <= 0) return;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid >> 6;
  const T* A = a + d.a_offset;
  const int64_t rs = lower ? 1 : d.lda, cs = lower ? d.lda : 1;
  const int tr = trans ^ lower;
  T* y = b + d.b_offset + (int64_t)blockIdx.y * d.ldb;
  for (int i = tid; i < kk; i += kBigThreads) xs[i] = y[i];
  __syncthreads();
  const int blocks = (kk + kTrsvBlock - 1) / kTrsvBlock;
  for (int q = 0; q < blocks; ++q) {
    const int bi = tr ? q : blocks - 1 - q;
    const int r0 = bi * kTrsvBlock;
    const int r1 = min(kk, r0 + kTrsvBlock);
    const int bs = r1 - r0;
    // diagonal block tile[i][j] = R[r0 + i][r0 + j]: loads issued here (clamped
    // indices, masked values), stored to LDS after the product pass
    constexpr int kTileVals = kTrsvBlock * kTrsvBlock / kBigThreads;
    T tv[kTileVals];
#pragma unroll
    for (int u = 0; u < kTileVals; ++u) {
      const int idx = tid + u * kBigThreads;
      const int i = idx >> 6, j = idx & 63;
      const T v = A[(int64_t)(r0 + min(i, bs - 1)) * rs + (int64_t)(r0 + min(j, bs - 1)) * cs];
      tv[u] = (i < bs && j < bs && j >= i) ? v : T(0);
    }
    if (!tr) {
      // z_i = y_i - sum_{c >= r1} R[i][c] x_c: wave wv takes rows r0 + wv + 16 t
      // (eight independent partial sums keep eight loads in flight per lane)
      for (int i = wv; i < bs; i += kBigWaves) {
        T s8[8] = {};
        const T* Ri = A + (int64_t)(r0 + i) * rs;
        int c = r1 + lane;
        for (; c + 7 * kWave < kk; c += 8 * kWave) {
#pragma unroll
          for (int u = 0; u < 8; ++u) s8[u] += Ri[(int64_t)(c + u * kWave) * cs] * xs[c + u * kWave];
        }
        for (; c < kk; c += kWave) s8[0] += Ri[(int64_t)c * cs] * xs[c];
        T s = ((s8[0] + s8[1]) + (s8[2] + s8[3])) + ((s8[4] + s8[5]) + (s8[6] + s8[7]));
        s = wave_sum(s);
        if (lane == 0) red[i] = s;
      }
    } else {
      // z_i = y_i - sum_{c < r0} R[c][i] x_c: thread (column i, group g)
      const int i = lane, g = wv;
      T s8[8] = {};
      if (i < bs) {
        const T* Ai = A + (int64_t)(r0 + i) * cs;
        int c = g;
        for (; c + 7 * kBigWaves < r0; c += 8 * kBigWaves) {
#pragma unroll
          for (int u = 0; u < 8; ++u) s8[u] += Ai[(int64_t)(c + u * kBigWaves) * rs] * xs[c + u * kBigWaves];
        }
        for (; c < r0; c += kBigWaves) s8[0] += Ai[(int64_t)c * rs] * xs[c];
      }
      red[g * kWave + i] = ((s8[0] + s8[1]) + (s8[2] + s8[3])) + ((s8[4] + s8[5]) + (s8[6] + s8[7]));
    }
#pragma unroll
    for (int u = 0; u < kTileVals; ++u) {
      const int idx = tid + u * kBigThreads;
      const int i = idx >> 6, j = idx & 63;
      tile[i * (kTrsvBlock + 1) + j] = tv[u];
      if (i == j) rinv[i] = (unit_diag || i >= bs) ? T(1) : T(1) / tv[u];
    }
    __syncthreads();
    if (wv == 0) {
      T z = T(0);
      if (lane < bs) {
        if (!tr) {
          z = xs[r0 + lane] - red[lane];
        } else {
          T s = T(0);
#pragma unroll
          for (int g = 0; g < kBigWaves; ++g) s += red[g * kWave + lane];
          z = xs[r0 + lane] - s;
        }
      }
      // Substitution through the block, one unknown per step: lane j scales
      // by the reciprocal pivot and readlane broadcasts it (a register read,
      // not an LDS round trip).  Fully unrolled, so the LDS reads of the
      // multipliers do not wait on the chain.  Steps j >= bs are no-ops
      // (zero padding, x_j = 0).
      const T rl = rinv[lane];
      if (!tr) {
#pragma unroll
        for (int j = kTrsvBlock - 1; j >= 0; --j) {
          const T mult = tile[lane * (kTrsvBlock + 1) + j];
          if (lane == j) z *= rl;
          const T xj = j < bs ? from_lane(z, j) : T(0);
          if (lane < j) z -= mult * xj;
        }
      } else {
#pragma unroll
        for (int j = 0; j < kTrsvBlock; ++j) {
          const T mult = tile[j * (kTrsvBlock + 1) + lane];
          if (lane == j) z *= rl;
          const T xj = j < bs ? from_lane(z, j) : T(0);
          if (lane > j) z -= mult * xj;
        }
      }
      if (lane < bs) xs[r0 + lane] = z;
    }
    __syncthreads();
  }
  for (int i = tid; i < kk; i += kBigThreads) y[i] = xs[i];
}

size_t trsv_smem_bytes(int dtype) {
  const size_t e = dtype == LXA_F64 ? 8 : 4;
  return e * (((kTrsvMaxK + 1) & ~1) + kTrsvBlock * (kTrsvBlock + 1) + kBigWaves * kWave + kTrsvBlock);
}

// Panels at column k (kcol == nullptr) or kcol[s] + k of system s.  max_rows
// bounds the panels' rows over the systems that still have columns.
template <typename T>
int panel_only(hipStream_t st, int64_t count, const lxa_qr_desc* desc, int k, const int32_t* kcol, int max_rows, T* a,
               T* tau, T* tblk) {
  if (max_rows <= kStepMaxRows) return qr_step(st, count, desc, kStepPanel, k, kcol, max_rows, 0, a, tau, tblk);
  qr_panel_kernel<T><<<dim3((unsigned)count), kPanelThreads, 0, st>>>(desc, k, kcol, a, tau, tblk);
  LXA_LAUNCH_CHECK("qr_panel_kernel");
  return LXA_OK;
}

// `steps` panel steps of every system from column 0 (kcol == nullptr) or
// kcol[s] on: each factors a panel and updates the columns right of it.
// max_rows bounds m - kcol and max_right the columns right of the first panel
// (n - kcol - 1, as a last panel may have a single column).  The update of a
// step factors the panel of the next one, so only the first panel has a
// launch of its own.
template <typename T>
int qr_steps(hipStream_t st, int64_t count, const lxa_qr_desc* desc, const int32_t* kcol, int steps, int max_rows,
             int max_right, T* a, T* tau, T* tblk) {
  constexpr int NB = QrCfg<T>::NB;
  if (int rc = panel_only<T>(st, count, desc, 0, kcol, max_rows, a, tau, tblk)) return rc;
  for (int j = 0; j < steps; ++j) {
    const int k = NB * j, rows = max_rows - k, right = max_right - k;
    if (rows <= 0 || right <= 0) break;
    const bool more = j + 1 < steps && rows > NB, ahead = more && rows <= kStepMaxRows;
    if (int rc = qr_step(st, count, desc, ahead ? kStepLookahead : kStepUpdate, k, kcol, rows, right, a, tau, tblk))
      return rc;
    if (more && !ahead) {
      if (int rc = panel_only<T>(st, count, desc, k + NB, kcol, rows - NB, a, tau, tblk)) return rc;
    }
  }
  return LXA_OK;
}

int check_batch(int dtype, int64_t count, const void* desc) {
  LXA_REQUIRE(dtype == LXA_F32 || dtype == LXA_F64, "dtype must be LXA_F32 or LXA_F64 (got %d)", dtype);
  LXA_REQUIRE(count >= 0 && count <= 0x7fffffff, "count out of range (%lld)", (long long)count);
  LXA_REQUIRE(count == 0 || desc != nullptr, "desc is NULL");
  return LXA_OK;
}

}  // namespace
}  // namespace lxa

using namespace lxa;

extern "C" int lxa_qr_block(int dtype) { return dtype == LXA_F64 ? QrCfg<double>::NB : QrCfg<float>::NB; }

extern "C" int lxa_qr_work_elems(int dtype, int64_t m, int64_t n, int64_t* elems) {
  LXA_REQUIRE(dtype == LXA_F32 || dtype == LXA_F64, "dtype must be LXA_F32 or LXA_F64 (got %d)", dtype);
  LXA_REQUIRE(m >= 0 && n >= 0 && elems != nullptr, "invalid arguments");
  *elems = 1;  // nothing is used: the smallest buffer that is one
  return LXA_OK;
}

extern "C" int lxa_qr_factor(void* stream, int dtype, int64_t count, const lxa_qr_desc* desc, int max_m, int max_n,
                             int max_k, void* a, void* tau, void* tblk, void* work) {
  if (int rc = check_batch(dtype, count, desc)) return rc;
  LXA_REQUIRE(max_m >= 0 && max_n >= 0 && max_k >= 0 && max_k <= max_m && max_k <= max_n,
              "inconsistent bounds max_m=%d max_n=%d max_k=%d", max_m, max_n, max_k);
  if (count == 0 || max_k == 0) return LXA_OK;
  LXA_REQUIRE(a && tau && tblk && work, "a, tau, tblk and work must be non-NULL");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == LXA_F32)
    return qr_steps<float>(st, count, desc, nullptr, (max_k + 15) / 16, max_m, max_n - 1, static_cast<float*>(a),
                           static_cast<float*>(tau), static_cast<float*>(tblk));
  return qr_steps<double>(st, count, desc, nullptr, (max_k + 15) / 16, max_m, max_n - 1, static_cast<double*>(a),
                          static_cast<double*>(tau), static_cast<double*>(tblk));
}

extern "C" int lxa_qr_factor_step(void* stream, int dtype, int64_t count, const lxa_qr_desc* desc,
                                  const int32_t* kcol, int max_rows, int max_trail_cols, void* a, void* tau,
                                  void* tblk, void* work) {
  return lxa_qr_factor_steps(stream, dtype, count, desc, kcol, 1, max_rows, max_trail_cols, a, tau, tblk, work);
}

extern "C" int lxa_qr_factor_steps(void* stream, int dtype, int64_t count, const lxa_qr_desc* desc,
                                   const int32_t* kcol, int steps, int max_rows, int max_trail_cols, void* a,
                                   void* tau, void* tblk, void* work) {
  LXA_REQUIRE(steps >= 0, "steps must be >= 0");
  if (int rc = check_batch(dtype, count, desc)) return rc;
  LXA_REQUIRE(kcol != nullptr, "kcol must be non-NULL");
  LXA_REQUIRE(max_rows >= 0, "max_rows must be >= 0");
  if (count == 0 || max_rows == 0 || steps == 0) return LXA_OK;
  LXA_REQUIRE(a && tau && tblk && work, "a, tau, tblk and work must be non-NULL");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == LXA_F32)
    return qr_steps<float>(st, count, desc, kcol, steps, max_rows, max_trail_cols, static_cast<float*>(a),
                           static_cast<float*>(tau), static_cast<float*>(tblk));
  return qr_steps<double>(st, count, desc, kcol, steps, max_rows, max_trail_cols, static_cast<double*>(a),
                          static_cast<double*>(tau), static_cast<double*>(tblk));
}

extern "C" int lxa_qr_apply(void* stream, int dtype, int64_t count, const lxa_qr_desc* desc, int max_m, int max_k,
                            const void* a, const void* tblk, int nrhs, void* b, int trans) {
  if (int rc = check_batch(dtype, count, desc)) return rc;
  LXA_REQUIRE(nrhs >= 0 && nrhs <= 65535, "nrhs out of range (%d)", nrhs);
  LXA_REQUIRE(max_k >= 0 && max_m >= max_k, "inconsistent bounds max_m=%d max_k=%d", max_m, max_k);
  if (count == 0 || nrhs == 0 || max_k == 0) return LXA_OK;
  LXA_REQUIRE(a && tblk && b, "a, tblk and b must be non-NULL");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)count, (unsigned)nrhs);
  if (max_m <= kApplyMaxRows) {
    if (dtype == LXA_F32) return apply_rows<float>(st, grid, max_m, desc, a, tblk, b, trans ? 1 : 0);
    return apply_rows<double>(st, grid, max_m, desc, a, tblk, b, trans ? 1 : 0);
  }
  if (dtype == LXA_F32)
    qr_apply_kernel<float><<<grid, kBigThreads, 0, st>>>(desc, static_cast<const float*>(a),
                                                          static_cast<const float*>(tblk), static_cast<float*>(b),
                                                          trans ? 1 : 0);
  else
    qr_apply_kernel<double><<<grid, kBigThreads, 0, st>>>(desc, static_cast<const double*>(a),
                                                           static_cast<const double*>(tblk), static_cast<double*>(b),
                                                           trans ? 1 : 0);
  LXA_LAUNCH_CHECK("qr_apply_kernel");
  return LXA_OK;
}

extern "C" int lxa_trsv(void* stream, int dtype, int64_t count, const lxa_qr_desc* desc, int max_k, const void* a,
                        int nrhs, void* b, int lower, int trans, int unit_diag) {
  if (int rc = check_batch(dtype, count, desc)) return rc;
  LXA_REQUIRE(nrhs >= 0 && nrhs <= 65535, "nrhs out of range (%d)", nrhs);
  if (max_k > kTrsvMaxK)
    return set_error(LXA_EUNSUPPORTED, "triangular solves support order <= %d (got %d)", kTrsvMaxK, max_k);
  if (count == 0 || nrhs == 0 || max_k <= 0) return LXA_OK;
  LXA_REQUIRE(a && b, "a and b must be non-NULL");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)count, (unsigned)nrhs);
  const size_t smem = trsv_smem_bytes(dtype);
  if (dtype == LXA_F32) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&trsv_kernel<float>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return hip_error(e, "hipFuncSetAttribute(trsv)");
    trsv_kernel<float><<<grid, kBigThreads, smem, st>>>(desc, static_cast<const float*>(a), static_cast<float*>(b),
                                                          lower ? 1 : 0, trans ? 1 : 0, unit_diag ? 1 : 0);
  } else {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&trsv_kernel<double>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return hip_error(e, "hipFuncSetAttribute(trsv)");
    trsv_kernel<double><<<grid, kBigThreads, smem, st>>>(desc, static_cast<const double*>(a),
                                                           static_cast<double*>(b), lower ? 1 : 0, trans ? 1 : 0,
                                                           unit_diag ? 1 : 0);
  }
  LXA_LAUNCH_CHECK("trsv_kernel");
  return LXA_OK;
}
