// The QR panel step kernel (qr.hip says what it is for).  Its unrolled
// instances are most of the library's compile time, so float, double and the
// double ones with the most registers are in files of their own.
#pragma once
#include <algorithm>

#include "qr_step.h"

namespace lxa {
namespace {

// ---------------------------------------------------------------------------
// One panel step for 16 columns of one system per workgroup.
// ---------------------------------------------------------------------------

// Where the inner index of a product (Mma) is the row index of an earlier
// result, step e takes inner indices row(0..3, e), so that register e of that
// result is the B operand as it stands.

// The 64-bit move (one instruction instead of two); the builtin takes 64-bit
// values only with literal controls, hence the switch (j is a constant).
__device__ __forceinline__ long long row_bcast64(long long v, int j) {
#define LXA_ROW_BCAST(J) \
  case J:                \
    return __builtin_amdgcn_update_dpp(v, v, 0x150 + J, 0xF, 0xF, true);
  switch (j) {
    LXA_ROW_BCAST(0)
    LXA_ROW_BCAST(1)
    LXA_ROW_BCAST(2)
    LXA_ROW_BCAST(3)
    LXA_ROW_BCAST(4)
    LXA_ROW_BCAST(5)
    LXA_ROW_BCAST(6)
    LXA_ROW_BCAST(7)
    LXA_ROW_BCAST(8)
    LXA_ROW_BCAST(9)
    LXA_ROW_BCAST(10)
    LXA_ROW_BCAST(11)
    LXA_ROW_BCAST(12)
    LXA_ROW_BCAST(13)
    LXA_ROW_BCAST(14)
    LXA_ROW_BCAST(15)
  }
#undef LXA_ROW_BCAST
  return v;
}

// The value of lane J of this lane's row of 16 (DPP row_newbcast; every lane
// must be active).
template <int J, typename T>
__device__ __forceinline__ T row_bcast(T v) {
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x150 + J, 0xF, 0xF, true));
  } else {
    return __builtin_bit_cast(T, row_bcast64(__builtin_bit_cast(long long, v), J));
  }
}

// larfg in double: from alpha and the squared norm ss > 0 below it, beta =
// -sign(alpha) |[alpha; x]|, tau = (beta - alpha) / beta and 1 / (alpha - beta).
// Every wave repeats it for every column, so the instructions count: hardware
// reciprocals and Newton steps to full precision, a third of the operations
// of a square root and two divisions.
__device__ __forceinline__ void reflector(double alpha, double ss, double& beta, double& tau, double& scale) {
  const double t = fma(alpha, alpha, ss);
  if (t >= 0x1p-800 && t <= 0x1p800) {  // uniform
    double r = __builtin_amdgcn_rsq(t);
    r = fma(r, fma(-t * r, 0.5 * r, 0.5), r);
    r = fma(r, fma(-t * r, 0.5 * r, 0.5), r);
    double norm = t * r;
    norm = fma(fma(-norm, norm, t), 0.5 * r, norm);
    const double den = fabs(alpha) + norm;
    double c = __builtin_amdgcn_rcp(den);
    c = fma(fma(-den, c, 1.0), c, c);
    c = fma(fma(-den, c, 1.0), c, c);
    beta = -copysign(norm, alpha);
    tau = den * r;  // 1 + |alpha| / norm
    scale = copysign(c, alpha);
  } else {
    beta = -copysign(sqrt(t), alpha);
    tau = (beta - alpha) / beta;
    scale = 1.0 / (alpha - beta);
  }
}

// Whether v_q^T v_j may be formed as the scales of v_q and v_j times a sum over
// the unscaled columns (larft in qr_step_kernel).  The sum has at most 2^12
// products and the columns' norms are below 1 / |scale|: with both scales in
// this range nothing overflows, and what is lost below the smallest normal
// number is below rounding.
__device__ __forceinline__ bool unscaled_sums(float scale) {
  return fabsf(scale) >= 0x1p-50f && fabsf(scale) <= 0x1p40f;
}
__device__ __forceinline__ bool unscaled_sums(double scale) {
  return fabs(scale) >= 0x1p-480 && fabs(scale) <= 0x1p450;
}

// Columns of a workgroup that does not keep them in registers: V is read once
// per 64 columns instead of once per 16.
constexpr int kWideTiles = 4;
constexpr int kWideCols = 16 * kWideTiles;
constexpr int kWideLd = kWideCols + 1;

// Column blocks of a launch that updates `right` columns.  All blocks of a
// KR = 4 lookahead launch (panels of up to 512 rows) have 16 columns in
// registers; taller ones have the next panel's 16 and wide blocks after it.
// Updates of about twenty systems of up to 4096 rows: 160 us in wide blocks,
// 180 us with 16 columns in registers everywhere (one workgroup a CU then).
constexpr bool step_wide(int KR, int mode) { return mode == kStepUpdate || KR > 4; }
inline int step_blocks(int KR, int mode, int right) {
  if (mode == kStepPanel) return 1;
  if (mode == kStepUpdate) return (right + kWideCols - 1) / kWideCols;
  if (!step_wide(KR, mode)) return (right + 15) / 16;
  return 1 + (std::max(0, right - 16) + kWideCols - 1) / kWideCols;
}

// KR: 16-row tiles per wave held in registers (slot s of wave w is tile
// w + 8 s of the rows from k on); KL: further ones in LDS (28 slots, 3584 rows,
// in float and 24, 3072 rows, in double are what 256 registers hold beside the
// products' operands, the 24 with a few dozen bytes of scratch a lane).
// KR = 0: wide blocks only, any height.
template <typename T, int KR, int KL>
__global__ __launch_bounds__(kPanelThreads) void qr_step_kernel(const lxa_qr_desc* __restrict__ descs, int64_t count,
                                                                int mode, int k_all,
                                                                const int32_t* __restrict__ kcol, T* __restrict__ a,
                                                                T* __restrict__ tau, T* __restrict__ tblk) {
  // the panel's column: k_all, past kcol[s] where that is given
  constexpr int NB = QrCfg<T>::NB;
  static_assert(NB == 16 && KR % 4 == 0, "16-column panels; slots go in groups of four");
  constexpr int kWaves = kPanelWaves, kSpan = 16 * kWaves;  // rows per slot over the waves
  using M4 = typename Mma<T>::acc;
  extern __shared__ __align__(16) unsigned char step_smem[];
  T* far_slots = reinterpret_cast<T*>(step_smem);  // [KL][4][kPanelThreads]
  __shared__ T s_w[kWaves][NB][NB + 1];
  __shared__ T s_part[2][kWaves][NB];
  __shared__ double s_norm[2][kWaves];
  __shared__ T s_diag[2][NB];
  __shared__ T s_g[NB][NB];  // s_g[c][j] = v_c^T v_j, c < j
  __shared__ T s_tau[NB];

  const int64_t sys = blockIdx.x % count;
  const int blk = (int)(blockIdx.x / count);
  const lxa_qr_desc d = descs[sys];
  const int m = d.m, n = d.n, lda = d.lda;
  const int kmax = min(m, n);
  const int kc = kcol ? kcol[sys] : 0;
  if (kc >= kmax - k_all) return;  // no sum here: a system that is done may say so by any large column
  const int k = kc + k_all;
  const int nb = min(NB, kmax - k);
  const bool wide = mode == kStepUpdate || (mode == kStepLookahead && KR > 4 && blk > 0);
  const int c0 = mode == kStepPanel      ? k
                 : mode == kStepUpdate   ? k + nb + kWideCols * blk
                 : KR > 4 && blk > 0     ? k + nb + 16 + kWideCols * (blk - 1)
                                         : k + nb + 16 * blk;
  if (c0 >= n) return;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane & 15, g = lane >> 4;
  T* A = a + d.a_offset;
  const int col = c0 + q;
  const bool cv = col < n;
  const int rows = m - k;                                    // this step's rows
  const int ns = max(0, ((rows + 15) / 16 - wv + kWaves - 1) / kWaves);  // this wave's tiles

  // lane offsets of the four rows of a tile, from the row (k + kSpan * s)
  int rel[4];
  int64_t off[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    rel[e] = 16 * wv + Mma<T>::row(g, e);
    off[e] = (int64_t)rel[e] * lda;
  }
  auto base = [&](int s) { return A + (int64_t)min(k + kSpan * s, m - 1) * lda; };  // uniform
  auto exists = [&](int s, int e) { return kSpan * s + rel[e] < rows; };
  // T^T as the A operand of T^T W; rows of V as the A operands of V^T C
  // (project_v) and of V (T^T W) (expand_v)
  T tt[4] = {T(0), T(0), T(0), T(0)};
  if (mode != kStepPanel) {
    const T* Tp = tblk + d.t_offset + (int64_t)(k / NB) * NB * NB;
#pragma unroll
    for (int e = 0; e < 4; ++e) tt[e] = Tp[Mma<T>::row(g, e) * NB + q];
  }
  auto project_v = [&](int s, T (&x)[4]) {
    const T* p = base(s) + k + min(q, nb - 1);
    T v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = p[exists(s, e) ? off[e] : 0];
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = exists(s, e) && q < nb ? vpick(kSpan * s + rel[e], q, v[e]) : T(0);
  };
  const int rq = 16 * wv + q;
  const int64_t offq = (int64_t)rq * lda;
  auto expand_v = [&](int s, T (&x)[4]) {
    const bool in = kSpan * s + rq < rows;
    const T* p = base(s) + (in ? offq : 0) + k;
    T v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = p[min(Mma<T>::row(g, e), nb - 1)];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int j = Mma<T>::row(g, e);
      x[e] = in && j < nb ? -vpick(kSpan * s + rq, j, v[e]) : T(0);
    }
  };
  if (KR != 4 && wide) {
    // ---- 64 columns, C read for W = V^T C and again for C - V (T^T W)
    T(*s_wide)[NB][kWideLd] = reinterpret_cast<T(*)[NB][kWideLd]>(step_smem);  // [kWaves]
    auto load_wide = [&](int s, M4 (&c)[kWideTiles]) {
      const T* p = base(s);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const T* r = p + (exists(s, e) ? off[e] : 0);
#pragma unroll
        for (int u = 0; u < kWideTiles; ++u) c[u][e] = r[min(c0 + 16 * u + q, n - 1)];
      }
    };
    M4 w[kWideTiles];
#pragma unroll
    for (int u = 0; u < kWideTiles; ++u) w[u] = M4{T(0), T(0), T(0), T(0)};
#pragma unroll 2
    for (int s = 0; s < ns; ++s) {
      M4 c[kWideTiles];
      T x[4];
      load_wide(s, c);
      project_v(s, x);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int u = 0; u < kWideTiles; ++u) w[u] = Mma<T>::mul(x[e], exists(s, e) ? c[u][e] : T(0), w[u]);
    }
#pragma unroll
    for (int u = 0; u < kWideTiles; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) s_wide[wv][Mma<T>::row(g, e)][16 * u + q] = w[u][e];
    __syncthreads();
    M4 tw[kWideTiles];
#pragma unroll
    for (int u = 0; u < kWideTiles; ++u) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        T x = T(0);
#pragma unroll
        for (int i = 0; i < kWaves; ++i) x += s_wide[i][Mma<T>::row(g, e)][16 * u + q];
        w[u][e] = x;
      }
      tw[u] = M4{T(0), T(0), T(0), T(0)};
#pragma unroll
      for (int e = 0; e < 4; ++e) tw[u] = Mma<T>::mul(tt[e], w[u][e], tw[u]);
    }
#pragma unroll 2
    for (int s = 0; s < ns; ++s) {
      M4 c[kWideTiles];
      T x[4];
      load_wide(s, c);
      expand_v(s, x);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int u = 0; u < kWideTiles; ++u) c[u] = Mma<T>::mul(x[e], tw[u][e], c[u]);
      T* p = base(s);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int u = 0; u < kWideTiles; ++u)
          if (exists(s, e) && c0 + 16 * u + q < n) p[off[e] + c0 + 16 * u + q] = c[u][e];
    }
    return;
  }
  auto load = [&](int s) {
    const T* p = base(s) + min(col, n - 1);
    M4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = p[exists(s, e) ? off[e] : 0];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = cv && exists(s, e) ? v[e] : T(0);
    return v;
  };
  auto store = [&](int s, const M4& v) {
    T* p = base(s) + col;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (cv && exists(s, e)) p[off[e]] = v[e];
  };
  // f(slot, value) over this wave's tiles
  M4 acc[KR > 0 ? KR : 1];
  auto each = [&](auto&& f) __attribute__((always_inline)) {
    static_for<0, KR / 4>([&](auto G_) __attribute__((always_inline)) {
      constexpr int s4 = 4 * decltype(G_)::value;
      if (s4 < ns) {  // uniform; slots past the rows hold zeros
#pragma unroll
        for (int u = 0; u < 4; ++u) f(s4 + u, acc[s4 + u]);
      }
    });
    for (int s = KR; s < (KL > 0 ? ns : 0); ++s) {
      T* far = far_slots + (int64_t)(s - KR) * 4 * kPanelThreads + tid;
      M4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = far[e * kPanelThreads];
      f(s, v);
#pragma unroll
      for (int e = 0; e < 4; ++e) far[e * kPanelThreads] = v[e];
    }
  };
  auto each_read = [&](auto&& f) __attribute__((always_inline)) {
    static_for<0, KR / 4>([&](auto G_) __attribute__((always_inline)) {
      constexpr int s4 = 4 * decltype(G_)::value;
      if (s4 < ns) {
#pragma unroll
        for (int u = 0; u < 4; ++u) f(s4 + u, acc[s4 + u]);
      }
    });
    for (int s = KR; s < (KL > 0 ? ns : 0); ++s) {
      const T* far = far_slots + (int64_t)(s - KR) * 4 * kPanelThreads + tid;
      M4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = far[e * kPanelThreads];
      f(s, v);
    }
  };
  if constexpr (KR > 0) each([&](int s, M4& v) __attribute__((always_inline)) { v = load(s); });

  if (KR > 0 && mode != kStepPanel) {
    // ---- W = V^T C
    M4 w = {T(0), T(0), T(0), T(0)};
    each_read([&](int s, const M4& c) __attribute__((always_inline)) {
      T x[4];
      project_v(s, x);
#pragma unroll
      for (int e = 0; e < 4; ++e) w = Mma<T>::mul(x[e], c[e], w);
    });
#pragma unroll
    for (int e = 0; e < 4; ++e) s_w[wv][Mma<T>::row(g, e)][q] = w[e];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      T x = T(0);
#pragma unroll
      for (int i = 0; i < kWaves; ++i) x += s_w[i][Mma<T>::row(g, e)][q];
      w[e] = x;
    }
    // ---- T^T W, then C - V (T^T W)
    M4 tw = {T(0), T(0), T(0), T(0)};
#pragma unroll
    for (int e = 0; e < 4; ++e) tw = Mma<T>::mul(tt[e], w[e], tw);
    each([&](int s, M4& c) __attribute__((always_inline)) {
      T x[4];
      expand_v(s, x);
#pragma unroll
      for (int e = 0; e < 4; ++e) c = Mma<T>::mul(x[e], tw[e], c);
    });
  }
  if constexpr (KR > 0) {
    const int kn = mode == kStepPanel ? k : k + NB;  // the panel to factor
    if (blk != 0 || kn >= kmax) {
      each_read([&](int s, const M4& v) __attribute__((always_inline)) { store(s, v); });
      return;
    }
    const int nbn = min(NB, kmax - kn);
    const int t0 = (kn - k) / 16;  // tile with the panel's diagonal: slot 0 of wave t0
    T sc = T(1);                   // scaling of this lane's column below its diagonal, applied when stored
    static_for<0, NB>([&](auto J_) __attribute__((always_inline)) {
      constexpr int j = decltype(J_)::value;
      if (j >= nbn) return;  // uniform
      constexpr int b = j & 1;  // double-buffered: readers of column j - 1 may lag
      // x = column j below the diagonal: x^T (column q) and, in double, |column q|^2
      T dot[4] = {T(0), T(0), T(0), T(0)};
      double nrm[2] = {0.0, 0.0};
      each_read([&](int s, const M4& v) __attribute__((always_inline)) {
        if (s == 0 && wv < t0) return;  // uniform: rows above the panel
        M4 y = v;
        if (s == 0 && wv == t0) {       // uniform: rows above the diagonal and on it stay out
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = Mma<T>::row(g, e) > j ? v[e] : T(0);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          dot[e] = fma(row_bcast<j>(y[e]), y[e], dot[e]);
          if constexpr (sizeof(T) == 4) nrm[e & 1] = fma((double)y[e], (double)y[e], nrm[e & 1]);
        }
      });
      T dq = (dot[0] + dot[1]) + (dot[2] + dot[3]);
      dq += lane_xor<16>(dq);
      dq += lane_xor<32>(dq);
      double nq = nrm[0] + nrm[1];
      if constexpr (sizeof(T) == 4) {
        nq += lane_xor<16>(nq);
        nq += lane_xor<32>(nq);
      }
      if (g == 0) s_part[b][wv][q] = dq;
      if (sizeof(T) == 4 && lane == j) s_norm[b][wv] = nq;
      constexpr int gj = sizeof(T) == 4 ? j / 4 : j % 4, ej = sizeof(T) == 4 ? j % 4 : j / 4;  // row(gj, ej) = j
      if (wv == t0 && g == gj) s_diag[b][q] = acc[0][ej];
      lds_barrier();
      T dots = T(0);
      double ss = 0.0;
#pragma unroll
      for (int i = 0; i < kWaves; ++i) {
        dots += s_part[b][i][q];
        ss += sizeof(T) == 4 ? s_norm[b][i] : (double)s_part[b][i][j];
      }
      const T dv = s_diag[b][q];
      const double alpha = (double)s_diag[b][j];
      T tj = T(0), beta = (T)alpha, scale = T(1);
      if (ss != 0.0) {
        double bd, td, sd;
        reflector(alpha, ss, bd, td, sd);
        beta = (T)bd;
        tj = (T)td;
        scale = (T)sd;
      }
      // v = [1; scale x]: v^T (column q) for q > j (larf), v_q^T v for q < j
      // (larft; columns left of j are still unscaled)
      const T prod = dv + scale * dots;
      if (tid < j) s_g[tid][j] = sc * prod;
      if (tid == j) s_tau[j] = tj;
      if (q == j) sc = scale;
      // larf on the columns right of j; beta on the diagonal
      const bool right = q > j && q < nbn;
      const T on_diag = right ? -tj * prod : T(0);
      const T coef = on_diag * scale;
      each([&](int s, M4& v) __attribute__((always_inline)) {
        if (s == 0 && wv < t0) return;  // uniform
        if (s == 0 && wv == t0) {       // uniform
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const T moved = fma(row_bcast<j>(v[e]), coef, v[e]);
            v[e] = Mma<T>::row(g, e) > j ? moved : v[e];
          }
          if (g == gj) acc[0][ej] = q == j ? beta : acc[0][ej] + on_diag;
          return;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = fma(row_bcast<j>(v[e]), coef, v[e]);
      });
    });
    // column q of V from here on, with R above it
    each([&](int s, M4& v) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool below = s > 0 || wv > t0 || (wv == t0 && Mma<T>::row(g, e) > q);
        v[e] = below ? v[e] * sc : v[e];
      }
      store(s, v);
    });
    if (__any(!unscaled_sums(sc))) {  // uniform over the workgroup: every wave holds all columns' scales
      // ---- V^T V from the scaled columns: a result register is both operands
      // (1 % of the factor's time at 256 x 512 x 256 in float, 7 % at 4000 x 400)
      M4 w = {T(0), T(0), T(0), T(0)};
      each_read([&](int s, const M4& v) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = kSpan * s + rel[e] - 16 * t0;
          const T x = q < nbn ? vpick(r, q, v[e]) : T(0);
          w = Mma<T>::mul(x, x, w);
        }
      });
#pragma unroll
      for (int e = 0; e < 4; ++e) s_w[wv][Mma<T>::row(g, e)][q] = w[e];
      __syncthreads();
      if (tid < NB * NB) {
        T x = T(0);
#pragma unroll
        for (int i = 0; i < kWaves; ++i) x += s_w[i][tid / NB][tid % NB];
        s_g[tid / NB][tid % NB] = x;
      }
    }
    __syncthreads();  // s_g and s_tau complete

    // ---- T (larft, forward, columnwise): lane a owns row a of T.
    if (tid < NB) {
      const int ra = tid;
      T trow[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        T v = T(0);
        if (i < nbn) {
          if (ra == i) {
            v = s_tau[i];
          } else if (ra < i) {
            T x = T(0);
#pragma unroll
            for (int c = 0; c < NB; ++c)
              if (c >= ra && c < i) x += trow[c] * s_g[c][i];
            v = -s_tau[i] * x;
          }
        }
        trow[i] = v;
      }
      T* Tp = tblk + d.t_offset + (int64_t)(kn / NB) * NB * NB + ra * NB;
#pragma unroll
      for (int i = 0; i < NB; ++i) Tp[i] = trow[i];
      if (ra < nbn) tau[d.tau_offset + kn + ra] = s_tau[ra];
    }
  }
}

template <typename T, int KR, int KL>
int launch_step(hipStream_t st, int64_t count, const lxa_qr_desc* desc, int mode, int k, const int32_t* kcol,
                int right, T* a, T* tau, T* tblk) {
  const int blocks = step_blocks(KR, mode, right);
  const size_t far_bytes = sizeof(T) * (size_t)KL * 4 * kPanelThreads;
  const size_t wide_bytes = KR == 4 ? 0 : sizeof(T) * (size_t)kPanelWaves * 16 * kWideLd;
  const size_t smem = std::max(far_bytes, wide_bytes);
  if (smem) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&qr_step_kernel<T, KR, KL>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return hip_error(e, "hipFuncSetAttribute(qr_step_kernel)");
  }
  // a grid holds fewer than 2^32 threads: launches of at most 2^22 workgroups
  // of 512, whole column blocks of systems at a time
  const int64_t chunk = std::max<int64_t>(1, (int64_t(1) << 22) / blocks);
  for (int64_t s0 = 0; s0 < count; s0 += chunk) {
    const int64_t cnt = std::min(chunk, count - s0);
    qr_step_kernel<T, KR, KL><<<dim3((unsigned)(cnt * blocks)), kPanelThreads, smem, st>>>(
        desc + s0, cnt, mode, k, kcol ? kcol + s0 : nullptr, a, tau, tblk);
  }
  LXA_LAUNCH_CHECK("qr_step_kernel");
  return LXA_OK;
}

}  // namespace
}  // namespace lxa
