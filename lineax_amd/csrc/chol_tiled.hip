// Cholesky factorisation (potrf, upper: A = U^T U) in 64-column panels over
// all workgroups, in place, float32 and float64 (chol.hip says which calls
// come here), and the solve of the orders past its LDS tier.
//
// Factor: one launch per 64-column panel, all systems of the batch and all
// 64 x 64 tiles of the upper triangle at once.  Launch k
//   panel tiles (k, j), j >= k: apply panel k - 1 to the diagonal tile and to
//     tile (k, j), factor the diagonal tile (every workgroup repeats this, so
//     no second launch and no exchange is needed) and solve U_kj with it;
//   trailing tiles (i, j), i > k: apply panel k - 1, A_ij -= U_(k-1)i^T U_(k-1)j,
//     on the matrix cores.
// Panel tiles read only rows of panel k - 1, which the launch before finished;
// the factored diagonal tile may not replace A_kk while other workgroups read
// it, so it waits one launch in storage that nothing reads as matrix data:
// its strictly upper part transposed in the strictly lower triangle of the
// same tile, its diagonal in the row below that tile.
//
// What bounds it: the chain of n pivots (square root, reciprocal, scaling,
// update of the next row), about 0.1 us (float) each inside a launch, plus
// the launches.  A 16-row strip of a panel is therefore factored and solved
// by the same instructions: lanes 0..15 of every wave hold the strip's
// diagonal block, lanes 16..63 other columns, pivots and multipliers travel
// by readlane and no barrier lies inside a strip.  (All waves read the diagonal
// block, so wave 0 stores the factored one behind the barrier that ends the
// strip.)  One system of order 1000: 17.8 us (float) and 24.1 us (double) a
// launch; one workgroup in global memory, which this replaces, took 280 ms for
// the float one.
//
// Reference: lineax/_solver/cholesky.py:43-78 (cho_factor / cho_solve).
#include <algorithm>
#include <type_traits>

#include "lxa_common.h"

namespace lxa {
namespace {

constexpr int kT = 64;        // tile
constexpr int kS = 16;        // strip
constexpr int kThreads = 256;
constexpr int kLd = 2 * kT + 2;  // LDS row: diagonal tile, then the solved tile

// Square root and its reciprocal of a pivot, from the hardware reciprocal
// square root and Newton steps (the correctly rounded sqrt and division cost
// about four times as many dependent instructions on the chain): within an
// ulp or two of both.
__device__ __forceinline__ void pivot_root(float d, float& u, float& inv) {
  float r = __builtin_amdgcn_rsqf(d);
  r = fmaf(r, fmaf(-d * r, 0.5f * r, 0.5f), r);
  u = d * r;
  u = fmaf(fmaf(-u, u, d), 0.5f * r, u);
  inv = r;
}
__device__ __forceinline__ void pivot_root(double d, double& u, double& inv) {
  double r = __builtin_amdgcn_rsq(d);
  r = fma(r, fma(-d * r, 0.5 * r, 0.5), r);
  r = fma(r, fma(-d * r, 0.5 * r, 0.5), r);
  u = d * r;
  u = fma(fma(-u, u, d), 0.5 * r, u);
  inv = r;
}
// Pivots for which every step above stays normal.
__device__ __forceinline__ bool root_range(float d) { return d >= 0x1p-80f && d <= 0x1p80f; }
__device__ __forceinline__ bool root_range(double d) { return d >= 0x1p-800 && d <= 0x1p800; }

// Rows k0 .. k0 + 63 of the factor (all exist), columns c0 .. c0 + 63 (zero
// past column n): to registers, then to LDS columns at .. at + 63 of P, so
// that all of a workgroup's loads can be issued before any is waited for.
constexpr int kRowsPer = kT / (kThreads / kWave);
template <typename T>
__device__ __forceinline__ void fetch_rows(const T* A, int64_t ld, int n, int k0, int c0, T (&v)[kRowsPer]) {
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned cc = min(c0 + lane, n - 1);
  const T* p = A + (int64_t)(k0 + wv) * ld;  // uniform: stepped on the scalar unit
#pragma unroll
  for (int u = 0; u < kRowsPer; ++u, p += 4 * ld) v[u] = p[cc];
}
template <typename T>
__device__ __forceinline__ void stash_rows(const T (&v)[kRowsPer], int n, int c0, T* P, int at) {
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int u = 0; u < kRowsPer; ++u) P[(wv + 4 * u) * kLd + at + lane] = c0 + lane < n ? v[u] : T(0);
}

// Advances p by `steps` rows, but not past row n - 1 (row: p's row).  Row
// addresses are stepped instead of multiplied out: a 64-bit product per
// load costs more issue slots than the rest of the tile's arithmetic.
template <typename P>
__device__ __forceinline__ void step_rows(P& p, int& row, int steps, int n, int64_t ld) {
  const int to = min(row + steps, n - 1);
  p += (to - row == steps) ? steps * ld : (int64_t)(to - row) * ld;
  row = to;
}

// Launch k of the factorisation; nt tiles per side.  Workgroups [0, batch *
// (nt - k)) are the panel tiles; the next batch of them moves the diagonal
// tile of launch k - 1 into place; the rest are the trailing tiles.
template <typename T>
__global__ __launch_bounds__(kThreads, sizeof(T) == 4 ? 4 : 2) void chol_tile_kernel(int64_t batch, int n, int k, int nt, T* __restrict__ a,
                                                             int64_t a_stride, int negate,
                                                             int32_t* __restrict__ info) {
  using M4 = typename Mma<T>::acc;
  extern __shared__ __align__(16) unsigned char lxa_smem[];
  // [64][kLd]: P, rows of panel k - 1; then M, the diagonal tile and tile (k, j)
  // (sharing the space lets two double workgroups onto a CU: 256 systems of
  // order 150 take 34 us a launch instead of 48)
  T* P = reinterpret_cast<T*>(lxa_smem);
  T* M = P;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane & 15, g = lane >> 4;
  const int64_t sys = blockIdx.x % batch;
  int t = (int)(blockIdx.x / batch);
  T* A = a + sys * a_stride;
  const int64_t ld = n;
  const int k0 = k * kT;
  // the matrix itself is read for the first time by launch 0 (row 0 of tiles)
  // and launch 1 (all others)
  const T sign = (negate && k <= 1) ? T(-1) : T(1);

  if (k > 0 && t == nt - k) {
    // ---- the diagonal tile of the launch before moves to its place: row r of its
    // strictly lower triangle holds column r of the factor above the diagonal
    const int p0 = k0 - kT;
    T v[kRowsPer];
    const T* p = A + (int64_t)(p0 + wv) * ld + p0 + lane;
#pragma unroll
    for (int u = 0; u < kRowsPer; ++u, p += 4 * ld) v[u] = *p;
    const T dg = A[(int64_t)k0 * ld + p0 + lane];
#pragma unroll
    for (int u = 0; u < kRowsPer; ++u) {
      const int r = wv + 4 * u;
      if (lane < r) P[lane * kLd + r] = v[u];
      if (lane > r) P[lane * kLd + r] = T(0);
      if (lane == r) P[lane * kLd + r] = dg;
    }
    __syncthreads();  // every stored value is read before it is overwritten
    T* d = A + (int64_t)(p0 + wv) * ld + p0 + lane;
#pragma unroll 4
    for (int u = 0; u < kRowsPer; ++u, d += 4 * ld) *d = P[(wv + 4 * u) * kLd + lane];
    if (tid < kT) A[(int64_t)k0 * ld + p0 + tid] = T(0);
    return;
  }
  if (t > nt - k) {
    // ---- trailing tile (i, j), k < i <= j
    t -= nt - k + 1;
    int i = k + 1;
    while (t >= nt - i) {
      t -= nt - i;
      ++i;
    }
    const int j = i + t;
    T vi[kRowsPer], vj[kRowsPer];
    fetch_rows(A, ld, n, k0 - kT, i * kT, vi);
    fetch_rows(A, ld, n, k0 - kT, j * kT, vj);
    M4 acc[4];
    {
      int row = min(i * kT + 16 * wv + Mma<T>::row(g, 0), n - 1);
      const T* p = A + (int64_t)row * ld;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // entries below the diagonal (tile i = j) are loaded and not stored
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c][e] = sign * p[min(j * kT + 16 * c + q, n - 1)];
        if (e < 3) step_rows(p, row, Mma<T>::row(0, e + 1) - Mma<T>::row(0, e), n, ld);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the stores
    stash_rows(vi, n, i * kT, P, 0);
    stash_rows(vj, n, j * kT, P, kT);
    __syncthreads();
#pragma unroll 2
    for (int s = 0; s < kT; s += 4) {
      const T* Ps = P + (s + g) * kLd;
      const T av = -Ps[16 * wv + q];
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[c] = Mma<T>::mul(av, Ps[kT + 16 * c + q], acc[c]);
    }
    {
      const bool whole = i < j && j + 1 < nt;  // uniform
      int row = i * kT + 16 * wv + Mma<T>::row(g, 0);
      T* p = A + (int64_t)row * ld;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int col = j * kT + 16 * c + q;
          if (whole || (col < n && row <= col)) p[col] = acc[c][e];
        }
        if (e < 3) {
          const int d = Mma<T>::row(0, e + 1) - Mma<T>::row(0, e);
          row += d;
          p += d * ld;
        }
      }
    }
    return;
  }

  // ---- panel tile (k, j): M = [A_kk | A_kj] with panel k - 1 applied
  const int j = k + t;
  const int kb = min(kT, n - k0);
  const int ctiles = j > k ? 8 : 4;
  auto load_apply = [&](auto Tiles_) __attribute__((always_inline)) {
    constexpr int kTiles = decltype(Tiles_)::value;  // 16-column tiles: 4, or 8 with tile (k, j)
    T vk[kRowsPer], vj[kRowsPer];
    if (k > 0) {
      fetch_rows(A, ld, n, k0 - kT, k0, vk);
      if (kTiles == 8) fetch_rows(A, ld, n, k0 - kT, j * kT, vj);
    }
    M4 acc[kTiles];
    int row = min(k0 + 16 * wv + Mma<T>::row(g, 0), n - 1);
    const T* p = A + (int64_t)row * ld;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma unroll
      for (int c = 0; c < kTiles; ++c) acc[c][e] = p[min((c < 4 ? k0 : j * kT) + 16 * (c & 3) + q, n - 1)];
      if (e < 3) step_rows(p, row, Mma<T>::row(0, e + 1) - Mma<T>::row(0, e), n, ld);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 16 * wv + Mma<T>::row(g, e);
#pragma unroll
      for (int c = 0; c < kTiles; ++c) {
        const int cl = 16 * (c & 3) + q;
        const bool in = c < 4 ? (r <= cl && cl < kb) : j * kT + cl < n;
        // past the last row the diagonal tile continues as the identity; what
        // lies below the diagonal is not used (16 x 16 tiles there are
        // carried along: leaving them out would split the loops by wave)
        acc[c][e] = in ? sign * acc[c][e] : (c < 4 && r == cl) ? T(1) : T(0);
      }
    }
    if (k > 0) {
      stash_rows(vk, n, k0, P, 0);
      if (kTiles == 8) stash_rows(vj, n, j * kT, P, kT);
      __syncthreads();
#pragma unroll 4
      for (int s = 0; s < kT; s += 4) {
        const T* Ps = P + (s + g) * kLd;
        const T av = -Ps[16 * wv + q];
#pragma unroll
        for (int c = 0; c < kTiles; ++c) acc[c] = Mma<T>::mul(av, Ps[16 * c + q], acc[c]);
      }
      __syncthreads();  // P is M from here on
    }
#pragma unroll
    for (int c = 0; c < kTiles; ++c) {
#pragma unroll
      for (int e = 0; e < 4; ++e) M[(16 * wv + Mma<T>::row(g, e)) * kLd + 16 * c + q] = acc[c][e];
    }
  };
  if (j > k) {
    load_apply(std::integral_constant<int, 8>{});
  } else {
    load_apply(std::integral_constant<int, 4>{});
  }
  __syncthreads();

  int fail = 0;
#pragma unroll 1
  for (int s = 0; s < kT / kS; ++s) {
    // ---- strip s: lanes 0..15 of each wave hold its diagonal block, lanes
    // 16..63 the wave's share of the columns right of it
    const int r0 = s * kS;
    const int others = 16 * ctiles - r0 - kS;
    const int oc = wv * 48 + lane - kS;
    const int col = lane < kS ? r0 + lane : r0 + kS + min(oc, others - 1);
    const bool diag = wv == 0 && lane < kS;  // wave 0 keeps the factored block, the others work on copies
    T* Ms = M + r0 * kLd + (others > 0 ? col : min(col, r0 + kS - 1));
    T c[kS];
    if (wv == 0 || wv * 48 < others) {  // uniform
      // opaque per strip: the 16 lane masks are formed where they are used
      // instead of being held, and spilled, across the strips
      int ln = lane;
      asm volatile("" : "+v"(ln));
#pragma unroll
      for (int i = 0; i < kS; ++i) c[i] = Ms[i * kLd];
      static_for<0, kS>([&](auto T_) __attribute__((always_inline)) {
        constexpr int p = decltype(T_)::value;
        const T d = from_lane(c[p], p);
        if (!(d > T(0)) && fail == 0) fail = k0 + r0 + p + 1;
        T u, inv;
        if (root_range(d)) {  // uniform
          pivot_root(d, u, inv);
        } else {
          u = sqrt(d);  // NaN for a negative pivot
          inv = T(1) / u;
        }
        c[p] = ln == p ? u : c[p] * inv;
        static_for<p + 1, kS>([&](auto I_) __attribute__((always_inline)) {
          constexpr int i = decltype(I_)::value;
          c[i] -= from_lane(c[p], i) * c[p];
        });
      });
      if (lane >= kS && oc < others) {
#pragma unroll
        for (int i = 0; i < kS; ++i) Ms[i * kLd] = c[i];
      }
    }
    __syncthreads();
    // the factored diagonal block goes over the one that every wave has read
    // above, so behind the barrier; the update below takes no column of it
    if (diag) {
#pragma unroll
      for (int i = 0; i < kS; ++i) Ms[i * kLd] = c[i];
    }
    // ---- the rows below: M_rc -= M_sr^T M_sc, 16 x 16 tiles dealt to the
    // waves (row strip r, column tile c >= r)
    int idx = wv;
#pragma unroll 1
    for (int r = s + 1; r < 4; ++r) {
      const int cnt = ctiles - r;
#pragma unroll 1
      for (; idx < cnt; idx += 4) {
        const int c = r + idx;
        M4 acc;
        T* Mt = M + 16 * r * kLd + 16 * c + q;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = Mt[Mma<T>::row(g, e) * kLd];
#pragma unroll
        for (int h = 0; h < kS; h += 4) {
          const T* Mh = M + (r0 + h + g) * kLd;
          acc = Mma<T>::mul(-Mh[16 * r + q], Mh[16 * c + q], acc);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) Mt[Mma<T>::row(g, e) * kLd] = acc[e];
      }
      idx -= cnt;
    }
    __syncthreads();
  }

  if (j > k) {
    // U_kj (all 64 rows exist), and zeros below the diagonal in tile (j, k);
    // row 0 of tile (k + 1, k) holds the diagonal of U_kk until the next launch
    const int col = j * kT + lane;
    T* up = A + (int64_t)(k0 + wv) * ld + col;
    T* lo = A + (int64_t)(j * kT + wv) * ld + k0 + lane;
#pragma unroll 4
    for (int r = wv; r < kT; r += 4, up += 4 * ld, lo += 4 * ld) {
      if (col < n) *up = M[r * kLd + kT + lane];
      if (j * kT + r < n && !(j == k + 1 && r == 0)) *lo = T(0);
    }
    return;
  }
  const bool last = k == nt - 1;
  T* d = A + (int64_t)(k0 + wv) * ld + k0 + lane;
#pragma unroll 4
  for (int r = wv; r < kT; r += 4, d += 4 * ld) {
    if (r >= kb || lane >= kb) continue;
    if (last) {
      *d = r <= lane ? M[r * kLd + lane] : T(0);
    } else if (r > lane) {
      *d = M[lane * kLd + r];
    } else if (r == lane) {
      A[(int64_t)(k0 + kT) * ld + k0 + lane] = M[r * kLd + lane];
    }
  }
  if (tid == 0 && (k == 0 || (fail && info[sys] == 0))) info[sys] = fail;
}

// The whole factor of a system that failed becomes NaN.
template <typename T>
__global__ __launch_bounds__(kThreads) void chol_fail_kernel(int n, T* __restrict__ a, int64_t a_stride,
                                                             const int32_t* __restrict__ info, int64_t sys0) {
  const int64_t sys = sys0 + blockIdx.x;
  if (info[sys] == 0) return;
  T* A = a + sys * a_stride;
  const int64_t nn = (int64_t)n * n;
  for (int64_t e = threadIdx.x; e < nn; e += kThreads) A[e] = quiet_nan<T>();
}

// ---------------------------------------------------------------------------
// U^T U x = b, one right-hand side per system, one 512-thread workgroup each.
// The vector is in LDS; thread t takes every 512th column right of the block
// at hand and reads rows of U (coalesced) in both directions:
//   forward   y_j -= sum over the block's rows i of U_ij y_i, right-looking;
//   backward  sum over columns j of U_ij x_j for the block's rows, left-looking,
//             a wave reduce-scatter and a sum over waves in a fixed order.
// What a thread needs for its first two columns of the next block, and the next
// but one diagonal block, are loaded one block ahead, and the barriers order
// LDS only, so no block waits for memory.  The chain of R steps by one wave,
// multipliers in registers, bounds the solve: 186 us in float and 298 us in
// double at order 1000.
// ---------------------------------------------------------------------------
constexpr int kSolveThreads = 512;
constexpr int kSolveCols = 2;  // columns per thread that are loaded ahead
constexpr int kSolveWaves = kSolveThreads / kWave;

template <typename T>
struct SolveRows {
  static constexpr int value = sizeof(T) == 4 ? 32 : 16;
};

template <typename T, bool InLds>
__global__ __launch_bounds__(kSolveThreads) void chol_tile_solve_kernel(int n, const T* __restrict__ u,
                                                                        int64_t u_stride, T* __restrict__ b,
                                                                        int64_t b_stride, int negate) {
  constexpr int R = SolveRows<T>::value;
  extern __shared__ __align__(16) unsigned char lxa_smem[];
  T* ys = reinterpret_cast<T*>(lxa_smem);  // [n rounded up to R]
  __shared__ T part[kSolveWaves][R];
  __shared__ T D[2][R][R + 1];            // diagonal blocks, double-buffered
  __shared__ T rd[2][R];                  // reciprocals of their diagonals, 0 where that is no normal number
  const T* U = u + (int64_t)blockIdx.x * u_stride;
  T* B = b + (int64_t)blockIdx.x * b_stride;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t ld = n;
  const int blocks = (n + R - 1) / R;
  // the vector: in LDS, or in place in global memory where it would not fit
  // beside the buffers above
  auto get = [&](int i) -> T {
    if constexpr (InLds) return ys[i];
    return i < n ? B[i] : T(0);
  };
  auto put = [&](int i, T x) {
    if constexpr (InLds) {
      ys[i] = x;
    } else {
      if (i < n) B[i] = x;
    }
  };
  if constexpr (InLds) {
    for (int i = tid; i < blocks * R; i += kSolveThreads) ys[i] = i < n ? B[i] : T(0);
  }

  // the diagonal block of block p passes through dv
  constexpr int kDv = (R * R + kSolveThreads - 1) / kSolveThreads;
  T dv[kDv] = {};
  const int dj = tid % R;
  auto fetch_diag = [&](int p) {
#pragma unroll
    for (int h = 0; h < kDv; ++h) {
      const int di = (tid + h * kSolveThreads) / R;
      if (di < R) {
        const int j = min(p * R + dj, n - 1);
        dv[h] = U[(int64_t)min(p * R + di, j) * ld + j];
      }
    }
  };
  auto stash_diag = [&](int p) {
#pragma unroll
    for (int h = 0; h < kDv; ++h) {
      const int di = (tid + h * kSolveThreads) / R;
      if (di < R) {
        const bool in = p * R + dj < n && dj >= di;
        D[p & 1][di][dj] = in ? dv[h] : T(0);
        if (di == dj) rd[p & 1][di] = in && plain_range(dv[h]) ? T(1) / dv[h] : T(0);  // padding solves to 0
      }
    }
  };
  // column c, the R rows of block p (rows clamped; clamped ones meet y = 0)
  T v[kSolveCols][R], nx[kSolveCols][R];
  auto fetch = [&](int p, int c, T (&to)[R]) {
    const int rows = n - p * R;  // rows that exist from the block's first one on
    const unsigned cc = min(c, n - 1);
    const T* at = U + (int64_t)(p * R) * ld;  // uniform: stepped on the scalar unit
#pragma unroll
    for (int i = 0; i < R; ++i) {
      to[i] = at[cc];
      at += i + 1 < rows ? ld : 0;
    }
  };
  // the columns loaded ahead, of block p, from column c on
  auto fetch_ahead = [&](int p, int c) {
#pragma unroll
    for (int h = 0; h < kSolveCols; ++h)
      if (c + h * kSolveThreads < n) fetch(p, c + h * kSolveThreads + tid, nx[h]);  // uniform
  };
  auto take_ahead = [&]() {
#pragma unroll
    for (int h = 0; h < kSolveCols; ++h)
#pragma unroll
      for (int i = 0; i < R; ++i) v[h][i] = nx[h][i];
  };
#pragma unroll
  for (int h = 0; h < kSolveCols; ++h)
#pragma unroll
    for (int i = 0; i < R; ++i) nx[h][i] = T(0);
  // runs f(divide by this lane's diagonal entry of block p): by reciprocals, or
  // as divisions where one of the block's entries has none that is normal
  // (never a factor of lxa_chol_factor, whose entries are square roots)
  auto chain = [&](int p, auto&& f) __attribute__((always_inline)) {
    const T r = rd[p & 1][lane % R];
    const bool pad = p * R + lane % R >= n;
    if (__all(pad || r != T(0))) {
      f([&](T z) { return z * r; });
    } else {
      const T d = D[p & 1][lane % R][lane % R];
      f([&](T z) { return pad ? T(0) : z / d; });
    }
  };
  // the vector in global memory needs the barrier that orders global memory
  auto barrier = [&]() {
    if constexpr (InLds) {
      lds_barrier();
    } else {
      __syncthreads();
    }
  };

  // ---- U^T y = b
  fetch_diag(0);
  stash_diag(0);
  fetch_diag(min(1, blocks - 1));
  fetch_ahead(0, R);
  __syncthreads();
  for (int p = 0; p < blocks; ++p) {
    const int c0 = p * R + R;
    take_ahead();
    if (p + 1 < blocks) {
      stash_diag(p + 1);
      fetch_ahead(p + 1, c0 + R);
      fetch_diag(min(p + 2, blocks - 1));
    }
    if (wv == 0) {
      T z = get(p * R + lane % R);
      int ln = lane % R;  // lanes past R repeat the others; opaque per block: lane masks are not held across blocks
      asm volatile("" : "+v"(ln));
      T m[R];
#pragma unroll
      for (int i = 0; i < R; ++i) m[i] = D[p & 1][i][lane % R];
      chain(p, [&](auto over) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
          if (ln == i) z = over(z);
          const T zi = from_lane(z, i);
          if (ln > i) z -= m[i] * zi;
        }
      });
      if (lane < R && p * R + lane < n) put(p * R + lane, z);  // padding stays 0, also beside infinities
    }
    barrier();
    if (c0 + (wv << 6) < n) {  // uniform
      T yb[R];
#pragma unroll
      for (int i = 0; i < R; ++i) yb[i] = get(p * R + i);
      auto push = [&](int c, const T (&e)[R]) {
        T s = T(0);
#pragma unroll
        for (int i = 0; i < R; ++i) s += e[i] * yb[i];
        if (c < n) put(c, get(c) - s);
      };
#pragma unroll
      for (int h = 0; h < kSolveCols; ++h) push(c0 + h * kSolveThreads + tid, v[h]);
      for (int c = c0 + kSolveCols * kSolveThreads + tid; c < n; c += kSolveThreads) {
        fetch(p, c, v[0]);
        push(c, v[0]);
      }
    }
    barrier();
  }

  // ---- U x = y
  fetch_diag(blocks - 1);
  stash_diag(blocks - 1);
  fetch_diag(max(blocks - 2, 0));
  fetch_ahead(max(blocks - 2, 0), (blocks - 1) * R);
  if (tid < kSolveWaves * R) part[tid / R][tid % R] = T(0);
  __syncthreads();
  for (int p = blocks - 1; p >= 0; --p) {
    // the products with the columns solved so far, except those of the block
    // solved last, are in part; this block's rows of those columns follow
    if (p > 0) {
      take_ahead();
      stash_diag(p - 1);
      fetch_ahead(max(p - 2, 0), (p - 1) * R);
      fetch_diag(max(p - 2, 0));
    }
    if (wv == 0) {
      int ln = lane % R;
      asm volatile("" : "+v"(ln));
      T z = get(p * R + lane % R);
      {
        T s = T(0);
#pragma unroll
        for (int w = 0; w < kSolveWaves; ++w) s += part[w][lane % R];
        z -= s;
      }
      T m[R];
#pragma unroll
      for (int i = 0; i < R; ++i) m[i] = D[p & 1][lane % R][i];
      chain(p, [&](auto over) __attribute__((always_inline)) {
#pragma unroll
        for (int i = R - 1; i >= 0; --i) {
          if (ln == i) z = over(z);
          const T zi = from_lane(z, i);
          if (ln < i) z -= m[i] * zi;
        }
      });
      if (lane < R && p * R + lane < n) put(p * R + lane, z);  // padding stays 0, also beside infinities
    }
    barrier();
    if (p > 0) {
      T s[R];
#pragma unroll
      for (int i = 0; i < R; ++i) s[i] = T(0);
      const int c0 = p * R;
      auto pull = [&](int c, const T (&e)[R]) {
        const T x = c < n ? get(c) : T(0);
#pragma unroll
        for (int i = 0; i < R; ++i) s[i] += e[i] * x;
      };
#pragma unroll
      for (int h = 0; h < kSolveCols; ++h)
        if (c0 + h * kSolveThreads < n) pull(c0 + h * kSolveThreads + tid, v[h]);
      for (int c = c0 + kSolveCols * kSolveThreads + tid; c < n; c += kSolveThreads) {
        fetch(p - 1, c, v[0]);
        pull(c, v[0]);
      }
      if (c0 + wv * kWave < n || p == blocks - 1) {
        const T t = wave_reduce_scatter<R>(s, lane);
        constexpr int kShift = 6 - Log2<R>::value;
        if ((lane & ((1 << kShift) - 1)) == 0) part[wv][lane >> kShift] = t;
      }
    }
    barrier();
  }
  for (int i = tid; i < n; i += kSolveThreads) {
    const T x = get(i);
    B[i] = negate ? -x : x;
  }
}

template <typename T>
int factor_t(hipStream_t st, int64_t batch, int n, T* a, int64_t stride, int negate, int32_t* info) {
  const size_t smem = sizeof(T) * kT * kLd;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&chol_tile_kernel<T>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  if (e != hipSuccess) return hip_error(e, "hipFuncSetAttribute(chol_tile_kernel)");
  const int nt = (n + kT - 1) / kT;
  const int64_t most = (int64_t)nt + 1 + (int64_t)nt * (nt - 1) / 2;  // tiles of launch 1, the widest, or of launch 0
  // a grid holds fewer than 2^32 threads
  const int64_t chunk = std::max<int64_t>(1, (int64_t(1) << 23) / most);
  for (int64_t s0 = 0; s0 < batch; s0 += chunk) {
    const int64_t cnt = std::min(chunk, batch - s0);
    for (int k = 0; k < nt; ++k) {
      const int64_t rest = nt - k - 1;
      const int64_t tiles = nt - k + (k > 0 ? 1 + rest * (rest + 1) / 2 : 0);
      chol_tile_kernel<T><<<dim3((unsigned)(tiles * cnt)), kThreads, smem, st>>>(cnt, n, k, nt, a + s0 * stride, stride,
                                                                                  negate, info + s0);
    }
    chol_fail_kernel<T><<<dim3((unsigned)cnt), kThreads, 0, st>>>(n, a, stride, info, s0);
  }
  LXA_LAUNCH_CHECK("chol_tile_kernel");
  return LXA_OK;
}

template <typename T, bool InLds>
int solve_launch(hipStream_t st, int64_t batch, int n, const T* u, int64_t us, T* b, int64_t bs, int negate) {
  constexpr int R = SolveRows<T>::value;
  const size_t smem = InLds ? sizeof(T) * (size_t)((n + R - 1) / R * R) : 0;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&chol_tile_solve_kernel<T, InLds>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  if (e != hipSuccess) return hip_error(e, "hipFuncSetAttribute(chol_tile_solve_kernel)");
  chol_tile_solve_kernel<T, InLds><<<dim3((unsigned)batch), kSolveThreads, smem, st>>>(n, u, us, b, bs, negate);
  LXA_LAUNCH_CHECK("chol_tile_solve_kernel");
  return LXA_OK;
}

template <typename T>
int solve_t(hipStream_t st, int64_t batch, int n, const T* u, int64_t us, T* b, int64_t bs, int negate) {
  if (sizeof(T) * (size_t)n <= 128 * 1024) return solve_launch<T, true>(st, batch, n, u, us, b, bs, negate);
  return solve_launch<T, false>(st, batch, n, u, us, b, bs, negate);
}

}  // namespace

int chol_tile_factor(hipStream_t s, int64_t batch, int n, float* a, int64_t stride, int negate, int32_t* info) {
  return factor_t<float>(s, batch, n, a, stride, negate, info);
}
int chol_tile_factor(hipStream_t s, int64_t batch, int n, double* a, int64_t stride, int negate, int32_t* info) {
  return factor_t<double>(s, batch, n, a, stride, negate, info);
}
int chol_tile_solve(hipStream_t s, int64_t batch, int n, const float* u, int64_t us, float* b, int64_t bs,
                    int negate) {
  return solve_t<float>(s, batch, n, u, us, b, bs, negate);
}
int chol_tile_solve(hipStream_t s, int64_t batch, int n, const double* u, int64_t us, double* b, int64_t bs,
                    int negate) {
  return solve_t<double>(s, batch, n, u, us, b, bs, negate);
}

}  // namespace lxa
