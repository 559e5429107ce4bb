// linalg.hip -- batched dense factorizations for cp.linalg, one workgroup
// per matrix of a contiguous row-major batch, float32 and float64.
//
// Replaces the reference's NumPy/LAPACK host calls in linalg.py
// (solve / inv / det / slogdet :37-61, 149-159; cholesky :83-88; qr
// :97-105; eigh / eigvalsh :63-69, 122-127; svd / svdvals / pinv /
// matrix_rank / cond / lstsq :71-81, 129-183, 269-274).
//
//  * mmp_lu: blocked right-looking LU with partial pivoting (the first row of
//    largest |a| in the column, as LAPACK's getrf picks), unit-lower L and
//    U packed in place, pivots as LAPACK's 0-based row swaps, info = first
//    exactly-zero pivot (1-based) or 0.
//  * mmp_lu_solve: row swaps, forward then backward substitution for nrhs
//    right-hand sides (threads over rows x rhs per elimination step).
//  * mmp_cholesky: right-looking lower Cholesky; info = first non-positive
//    pivot (1-based); the strict upper triangle is zeroed.
//  * mmp_qr / mmp_qr_q: Householder QR with LAPACK's reflector convention
//    (beta = -sign(alpha) * ||x||, tau = (beta - alpha) / beta, v(0) = 1),
//    R in the upper triangle, reflectors below it, then Q accumulated
//    backwards into the first qcols columns of I (one wavefront per column).
//  * mmp_eigh: cyclic two-sided Jacobi for symmetric matrices, disjoint
//    rotation pairs per round (round-robin ordering), rows then columns
//    updated per round, eigenvectors accumulated in V.
//  * mmp_svd: one-sided (Hestenes) Jacobi orthogonalising the rows of W
//    (rows <= len), one wavefront per row pair, row rotations mirrored in
//    VT; the row norms are the singular values.
// Every loop is bounded (the Jacobi sweeps by kMaxSweeps), so each
// workgroup exits.
#include <limits>

#include "mmp_ops.h"
#include "mmp_internal.h"

namespace {

constexpr int kT = 256;           // LU / Cholesky / QR workgroup
constexpr int kJ = 1024;          // Jacobi workgroup (16 wavefronts)
constexpr int kMaxSweeps = 60;
constexpr int kMaxEighN = 2048;   // rotation table in LDS: kMaxEighN / 2 pairs
constexpr int kMaxSvdRows = 8192;
constexpr int kNb = 64;             // panel width in memory (Cholesky, tall LU panels)
constexpr int kBlockedMinN = 256;   // from this order a few matrices use products of blocks
constexpr int kBlockedMaxBatch = 64;
constexpr int kRhsChunk = 32;       // right-hand sides per workgroup in the substitution

// dst[r] -= src[r] * f for rows r = r0, r0 + S, ... < m of two columns of
// row-major matrices (leading dimensions ldd, lds): eight rows are loaded
// before any is stored (the stores never touch the loaded source column),
// so the loads overlap instead of waiting one by one.
template <typename T, int S>
__device__ __forceinline__ void axpy_rows(T *__restrict__ dst, long long ldd, const T *__restrict__ src,
                                          long long lds, int r0, int m, T f) {
  constexpr int U = 8;
  int r = r0;
  for (; r + (U - 1) * S < m; r += U * S) {
    T x[U], y[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      x[u] = src[(long long)(r + u * S) * lds];
      y[u] = dst[(long long)(r + u * S) * ldd];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) dst[(long long)(r + u * S) * ldd] = y[u] - x[u] * f;
  }
  for (; r < m; r += S) dst[(long long)r * ldd] -= src[(long long)r * lds] * f;
}

// Rows x, y (length len) := (c x - s y, s x + c y), lanes striding by 64,
// eight elements per lane loaded before any is stored.
template <typename T>
__device__ __forceinline__ void rotate_rows(T *__restrict__ x, T *__restrict__ y, int len, int lane, T c,
                                            T s) {
  constexpr int U = 8;
  int j = lane;
  for (; j + (U - 1) * 64 < len; j += U * 64) {
    T a[U], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      a[u] = x[j + u * 64];
      b[u] = y[j + u * 64];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      x[j + u * 64] = c * a[u] - s * b[u];
      y[j + u * 64] = s * a[u] + c * b[u];
    }
  }
  for (; j < len; j += 64) {
    const T a = x[j], b = y[j];
    x[j] = c * a - s * b;
    y[j] = s * a + c * b;
  }
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Sum over the workgroup, the same value in every thread (fixed order).
template <int NT, typename T>
__device__ T block_sum(T v, T *lds) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  T r = T(0);
  for (int i = 0; i < NT / 64; ++i) r += lds[i];
  return r;
}

// Round-robin pairing of N (even) indices: N - 1 rounds, N / 2 disjoint
// pairs per round, every pair met once per sweep.
__device__ __forceinline__ void pair_of(int r, int pi, int N, int &p, int &q) {
  if (pi == 0) {
    p = N - 1;
    q = r;
  } else {
    p = (r + pi) % (N - 1);
    q = (r - pi + (N - 1)) % (N - 1);
  }
}

// ------------------------------------------------------------------- LU
// Blocked right-looking LU of every matrix of a batch, three launches per
// panel of kLuW (or fewer) columns: k_lu_panel factors the panel with its
// rows in registers, k_lu_swap applies the panel's row swaps to the other
// columns and forms U12 = L11^-1 A12, and the trailing update
// A22 -= L21 U12 is k_lu_update, or for a few large matrices the
// matrix-product kernel subtracting in place.
//
// With k_lu_update every element goes through the operations of elimination
// column by column, in their order, each rounded by itself: the factors do not
// depend on the blocks, and a row that repeats another one ends in exact zeros,
// so that the matrix is reported as singular.  Sums in the matrix cores round
// differently from the triangular solve, and leave such a row a last place off
// zero.
//
// What bounds it is the chain of n pivot steps (each an argmax over the
// column, a row handed round, a division), not arithmetic: float64 n = 500
// 5.4 -> 1.2 ms, n = 1024 17.6 -> 3.1, n = 100 0.48 -> 0.20, 100 matrices of
// 200 3.1 -> 0.49, against panels in memory and one-workgroup elimination.

constexpr int kLuW = 32;  // most columns of a panel

// N contiguous values, as 16-byte loads at element alignment; the first
// `have` of them and zeros where that is fewer (a uniform choice: guarded
// loads are taken only where a block is cut off).
template <int N, typename T>
__device__ __forceinline__ void load_row(T (&v)[N], const T *p, int have) {
  constexpr int V = 16 / sizeof(T);
  if (have >= N) {
#pragma unroll
    for (int j = 0; j < N; j += V) __builtin_memcpy(&v[j], p + j, 16);
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = j < have ? p[j] : T(0);
  }
}

// Lane `l` (wave-uniform) of v.
__device__ __forceinline__ int lane_of(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ float lane_of(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
__device__ __forceinline__ double lane_of(double v, int l) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, l);
  const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), l);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Largest v of a wave, in every lane, through DPP moves (no LDS round trips):
// rows of 16 shifted by 1, 2, 4, 8, then the rows' last lanes passed on.  NaN
// never wins against a number; callers pass numbers.
template <int CTRL, int ROWS> __device__ __forceinline__ float dpp_mov(float v) {
  const int i = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, CTRL, ROWS, 0xf, false));
}
template <int CTRL, int ROWS> __device__ __forceinline__ double dpp_mov(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const int lo = (int)(unsigned)u, hi = (int)(unsigned)(u >> 32);
  const unsigned l2 = (unsigned)__builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false);
  const unsigned h2 = (unsigned)__builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)h2 << 32) | l2);
}
template <typename T> __device__ __forceinline__ T wave_max(T v) {
  v = fmax(v, dpp_mov<0x111, 0xf>(v));  // row_shr:1
  v = fmax(v, dpp_mov<0x112, 0xf>(v));  // row_shr:2
  v = fmax(v, dpp_mov<0x114, 0xf>(v));  // row_shr:4
  v = fmax(v, dpp_mov<0x118, 0xf>(v));  // row_shr:8
  v = fmax(v, dpp_mov<0x142, 0xa>(v));  // row_bcast:15
  v = fmax(v, dpp_mov<0x143, 0xc>(v));  // row_bcast:31
  return lane_of(v, 63);
}

// Lanes of one wave as the rows that the swaps k <-> piv[k], k = k0 .. k0 +
// jb - 1 (jb <= 32) touch: lane q < jb is row k0 + q, lane 32 + q the row
// piv[k0 + q] below the block, once.  Returns in `from` the row whose content
// this lane's row holds after all of them (applied in order); lanes without a
// row have row < 0.
__device__ __forceinline__ void swap_lanes(const int *__restrict__ piv, int k0, int jb, int lane,
                                           int &row, int &from) {
  const int q = lane & 31;
  const int pv = q < jb ? piv[k0 + q] : -1;
  row = -1;
  if (q < jb) row = lane < 32 ? k0 + q : (pv >= k0 + jb ? pv : -1);
  // a row that several swaps name belongs to the first of them
  for (int t = 0; t < jb; ++t) {
    const int r = lane_of(row, 32 + t);
    if (lane > 32 + t && r >= 0 && row == r) row = -1;
  }
  from = row;
  for (int t = 0; t < jb; ++t) {
    const int p = lane_of(pv, t);
    if (p == k0 + t) continue;  // uniform
    const int lp = __ffsll((long long)__ballot(row == p)) - 1;
    const int x = lane_of(from, t), y = lane_of(from, lp);
    from = lane == t ? y : lane == lp ? x : from;
  }
}

// One panel: rows j0 .., columns j0 .. j0 + jb - 1 (jb <= W), partial
// pivoting as LAPACK's getf2 (the first row of largest |a|).  Thread t holds
// rows t, t + blockDim, ... (R of them) in registers and never gives one
// away: a row keeps the position that the swaps have moved it to, and goes
// there when the panel is written.  A step is the column's largest value by
// shuffles and LDS, the pivot row through LDS, and each row's update; two
// barriers.  Four steps make one turn of the loop, after which the row turns
// by four, so that the columns in hand are always its first: straight code
// for every column would spend its time fetching instructions (64 us for 32
// steps of 128 rows, against 44).
template <typename T, int W, int R>
__global__ __launch_bounds__(512) void k_lu_panel(T *__restrict__ a, int n, int j0, int jb,
                                                  int *__restrict__ piv, int *__restrict__ info) {
  T *P = a + (long long)blockIdx.x * n * n + (long long)j0 * n + j0;
  const int m = n - j0, nt = blockDim.x;
  __shared__ T sval[8];
  __shared__ int sidx[8];
  __shared__ __attribute__((aligned(16))) T prow[W];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = nt >> 6;
  T v[R][W];
  int pos[R];  // row position; >= m: no row
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = tid + r * nt;
    pos[r] = i;
    load_row<W>(v[r], P + (long long)(i < m ? i : 0) * n, jb);
  }
  int first_zero = 0;
#pragma unroll 1
  for (int kk = 0; kk < W; kk += 4) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = kk + s;
      if (k < jb) {  // uniform
        T best = T(-1);
        int bi = m;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const T av = fabs(v[r][s]);
          if (pos[r] >= k && pos[r] < m && (av > best || (av == best && pos[r] < bi))) {
            best = av;
            bi = pos[r];
          }
        }
        // the wave's largest, and of the lanes that hold it the first position
        {
          const T top = wave_max(best);
          unsigned long long at = __ballot(best == top);
          best = top;
          int first = m;
          for (; at; at &= at - 1) {  // one lane, ties aside
            const int q = lane_of(bi, __ffsll((long long)at) - 1);
            first = q < first ? q : first;
          }
          bi = first;
        }
        if (nw > 1) {
          if (lane == 0) {
            sval[wave] = best;
            sidx[wave] = bi;
          }
          __syncthreads();
          T ov[8];
          int oi[8];
#pragma unroll
          for (int w = 0; w < 8; ++w) {
            ov[w] = sval[w];
            oi[w] = sidx[w];
          }
          best = ov[0];
          bi = oi[0];
#pragma unroll
          for (int w = 1; w < 8; ++w)
            if (w < nw && (ov[w] > best || (ov[w] == best && oi[w] < bi))) {
              best = ov[w];
              bi = oi[w];
            }
        } else {
          __syncthreads();  // the last step's pivot row has been read
        }
        const int p = bi < m ? bi : k;  // an all-NaN column keeps its row
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if (pos[r] == p) {
            pos[r] = k;
#pragma unroll
            for (int j = 0; j < W; ++j) prow[j] = v[r][j];
          } else if (pos[r] == k) {
            pos[r] = p;
          }
        }
        if (tid == 0) piv[(long long)blockIdx.x * n + j0 + k] = j0 + p;
        __syncthreads();
        const T u = prow[lane & (W - 1)];  // a value per lane, read into scalars below
        const T d = lane_of(u, s);
        if (d == T(0)) {  // the whole column is zero: nothing to eliminate
          if (!first_zero) first_zero = j0 + k + 1;
        } else {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            if (pos[r] > k && pos[r] < m) {
              const T l = v[r][s] / d;
              v[r][s] = l;
#pragma unroll
              for (int j = s + 1; j < 4; ++j) v[r][j] -= l * lane_of(u, j);
#pragma unroll
              for (int j = 4; j < W; j += 4) {
                if (j >= W - kk) break;  // uniform: the columns done with
#pragma unroll
                for (int e = 0; e < 4; ++e) v[r][j + e] -= l * lane_of(u, j + e);
              }
            }
          }
        }
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      T t[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) t[e] = v[r][e];
#pragma unroll
      for (int j = 0; j + 4 < W; ++j) v[r][j] = v[r][j + 4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[r][W - 4 + e] = t[e];
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int j = 0; j < W; ++j)
      if (pos[r] < m && j < jb) P[(long long)pos[r] * n + j] = v[r][j];
  if (tid == 0) {
    int *I = info + blockIdx.x;
    if (j0 == 0) *I = first_zero;
    else if (*I == 0) *I = first_zero;
  }
}

// The panel's row swaps on 64 of the other columns, all rows moved at once,
// and on those right of it the unit lower triangular solve U12 = L11^-1 A12
// (a column per lane, in registers, turned by four as in k_lu_panel).  Grid
// (ceil((n - jb) / 64), batch).
template <typename T>
__global__ __launch_bounds__(kT) void k_lu_swap(T *__restrict__ a, int n, int j0, int jb,
                                                const int *__restrict__ piv) {
  T *A = a + (long long)blockIdx.y * n * n;
  __shared__ __attribute__((aligned(16))) T Lt[kLuW][kLuW];  // L11 transposed
  __shared__ int srow[64], sfrom[64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c0 = blockIdx.x * 64 + lane;
  const int c = c0 < j0 ? c0 : c0 + jb;
  const bool on = c < n;
  if (wave == 0) {
    int row, from;
    swap_lanes(piv + (long long)blockIdx.y * n, j0, jb, lane, row, from);
    srow[lane] = row == from ? -1 : row;  // rows that stay put need no move
    sfrom[lane] = from;
  } else {
    // two waves, four threads a row
    if (wave < 3) {
      T l[8];
      const int i = (tid - 64) >> 2, k = ((tid - 64) & 3) * 8;
      load_row<8>(l, A + (long long)(j0 + (i < jb ? i : 0)) * n + j0 + k, jb - k);
#pragma unroll
      for (int e = 0; e < 8; ++e) Lt[k + e][i] = i < jb && k + e < i ? l[e] : T(0);
    }
  }
  __syncthreads();
  // every row moved is read before any is written
  T t[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int q = wave + u * (kT / 64);
    t[u] = A[(long long)(srow[q] >= 0 ? sfrom[q] : j0) * n + (on ? c : 0)];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int q = wave + u * (kT / 64);
    if (srow[q] >= 0 && on) A[(long long)srow[q] * n + c] = t[u];
  }
  __syncthreads();
  if (wave != 0) return;
  const int dk = j0 + (lane < jb ? lane : 0);  // a zero pivot eliminates nothing
  const unsigned long long zero = __ballot(lane < jb && A[(long long)dk * n + dk] == T(0));
  if (!on || c < j0 + jb) return;
  T x[kLuW];
#pragma unroll
  for (int i = 0; i < kLuW; ++i) {
    x[i] = A[(long long)(j0 + (i < jb ? i : 0)) * n + c];
    if (i >= jb) x[i] = T(0);
  }
#pragma unroll 1
  for (int kk = 0; kk < kLuW; kk += 4) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (kk + s < jb && !((zero >> (kk + s)) & 1)) {
        const T *l = &Lt[kk + s][kk];
        const T xk = x[s];
#pragma unroll
        for (int i = s + 1; i < 4; ++i) x[i] -= l[i] * xk;
#pragma unroll
        for (int i = 4; i < kLuW; i += 4) {
          if (i >= kLuW - kk) break;  // uniform: unknowns done with
#pragma unroll
          for (int e = 0; e < 4; ++e) x[i + e] -= l[i + e] * xk;
        }
      }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
      if (kk + s < jb) A[(long long)(j0 + kk + s) * n + c] = x[s];
#pragma unroll
    for (int i = 0; i + 4 < kLuW; ++i) x[i] = x[i + 4];
  }
}

// A22 -= L21 U12 by the panel's `jb` columns (8, 16 or 32) from `j0`, whose rows
// end at row `r1`: 64 x 64 outputs per workgroup, 4 x 4 per thread, L21 and U12
// in LDS.  Each product and each difference is rounded, column after column; a
// column whose pivot is zero eliminates nothing.  Grid (tiles^2, batch).
// Determinants by sums in the matrix cores / by this: 200 float64 matrices of
// 300 1146 / 1171 us, 100 of 100 242 / 254, float32 300 of 128 275 / 286.
template <typename T>
__global__ __launch_bounds__(kT) void k_lu_update(T *__restrict__ a, int n, int j0, int jb, int r1,
                                                  int tiles) {
  constexpr int TS = 64;
  __shared__ __attribute__((aligned(16))) T Ls[kLuW][TS + 4];  // L21 transposed
  __shared__ __attribute__((aligned(16))) T Us[kLuW][TS];
  T *A = a + (long long)blockIdx.y * n * n;
  const int tid = threadIdx.x, lane = tid & 63, tx = tid & 15, ty = tid >> 4;
  const int r0 = r1 + (int)(blockIdx.x / (unsigned)tiles) * TS;
  const int c0 = r1 + (int)(blockIdx.x % (unsigned)tiles) * TS;
  {
    const int i = tid >> 2, k = (tid & 3) * 8;
    T l[8];
    if (k < jb) {
      load_row<8>(l, A + (long long)(r0 + i < n ? r0 + i : n - 1) * n + j0 + k, 8);
#pragma unroll
      for (int e = 0; e < 8; ++e) Ls[k + e][i] = l[e];
    }
  }
  {
    const int k = tid >> 3, c = (tid & 7) * 8;
    T u[8];
    if (k < jb) {
      load_row<8>(u, A + (long long)(j0 + k) * n + c0 + c, n - c0 - c);
#pragma unroll
      for (int e = 0; e < 8; ++e) Us[k][c + e] = u[e];
    }
  }
  const int dk = j0 + (lane < jb ? lane : 0);
  const unsigned long long zero = __ballot(lane < jb && A[(long long)dk * n + dk] == T(0));
  T acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = r0 + ty + 16 * i;
    load_row<4>(acc[i], A + (long long)(r < n ? r : n - 1) * n + c0 + tx * 4, n - c0 - tx * 4);
  }
  __syncthreads();
  for (int k0 = 0; k0 < jb; k0 += 8) {
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      const int k = k0 + kk;
      if (zero && ((zero >> k) & 1)) continue;  // uniform
      T l[4], u[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) l[i] = Ls[k][ty + 16 * i];
#pragma unroll
      for (int j = 0; j < 4; ++j) u[j] = Us[k][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] -= l[i] * u[j];
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = r0 + ty + 16 * i;
    if (r >= n) continue;
    T *o = A + (long long)r * n + c0 + tx * 4;
    if (c0 + tx * 4 + 4 <= n) {
      __builtin_memcpy(o, acc[i], sizeof(acc[i]));
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (c0 + tx * 4 + j < n) o[j] = acc[i][j];
    }
  }
}

// Row swaps, then forward and backward substitution, of kRhs right-hand sides
// of one matrix in LDS, in blocks of 32 unknowns: one wave per right-hand side
// solves the block's triangle with its rows in registers (a lane each, the
// solved value read from its lane), then the threads subtract the block from
// the other rows, four threads on the 32 contiguous values of a row each.
// A block's values are loaded ahead of the solve that they wait for, and the
// next triangle ahead of the subtraction.  The backward solve's divisions go
// through each diagonal element's reciprocal, corrected by the remainder in
// fused multiply-adds (Markstein's method: the correctly rounded quotient but
// for rare last places), since a division proper in each of the chain's steps
// would be most of its time.  Grid (batch, ceil(nrhs / kRhs)).
// Bound by the chain of blocks: float64 n = 500 450 -> 215 us, n = 1024 with
// 1024 right-hand sides 19 -> 1.3 ms, against a barrier per unknown.
constexpr int kRhs = 8;
constexpr int kSolveLds = 128 * 1024;  // right-hand sides in LDS up to this
template <typename T>
__global__ __launch_bounds__(512) void k_lu_solve(const T *__restrict__ lu, const int *__restrict__ piv,
                                                  T *__restrict__ b, int n, int nrhs) {
  typedef std::numeric_limits<T> Lim;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  T *X = reinterpret_cast<T *>(smem);  // X[c * n + i]
  const T *A = lu + (long long)blockIdx.x * n * n;
  const int *P = piv + (long long)blockIdx.x * n;
  const int c0 = blockIdx.y * kRhs;
  const int cw = nrhs - c0 < kRhs ? nrhs - c0 : kRhs;
  T *B = b + (long long)blockIdx.x * n * nrhs + c0;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nt = blockDim.x, nw = nt >> 6;
  const int nb = (n + 31) / 32;
  for (int t = tid; t < n * cw; t += nt) X[(t % cw) * n + t / cw] = B[(long long)(t / cw) * nrhs + t % cw];
  T l[32];  // this lane's row of the triangle
  auto load_triangle = [&](int q) {
    const int i = q * 32 + (lane & 31);
    load_row<32>(l, A + (long long)(i < n ? i : n - 1) * n + q * 32, n - q * 32);
  };
  if (wave < cw) load_triangle(0);
  __syncthreads();
  for (int c = wave; c < cw; c += nw) {  // a wave swaps its own columns, in order
    for (int k0 = 0; k0 < n; k0 += 32) {
      int row, from;
      swap_lanes(P, k0, n - k0 < 32 ? n - k0 : 32, lane, row, from);
      const T x = row >= 0 ? X[c * n + from] : T(0);
      __builtin_amdgcn_wave_barrier();
      if (row >= 0) X[c * n + row] = x;
      __builtin_amdgcn_wave_barrier();
    }
  }
  __syncthreads();
  for (int pass = 0; pass < 2; ++pass) {  // unit lower, then upper
    for (int bq = 0; bq < nb; ++bq) {
      const int q = pass == 0 ? bq : nb - 1 - bq;
      const int k0 = q * 32, jb = n - k0 < 32 ? n - k0 : 32;
      const int i00 = pass == 0 ? k0 + 32 : 0, r1 = pass == 0 ? n : k0;  // rows to update
      constexpr int U = 4;
      const int part = tid & 3;  // columns 8 part .. 8 part + 7 of the block
      T m[U][8];
      auto load_rows = [&](int i0) {
#pragma unroll
        for (int w = 0; w < U; ++w) {
          const int i = i0 + w * (nt / 4) + (tid >> 2);
          load_row<8>(m[w], A + (long long)(i < n ? i : n - 1) * n + k0 + part * 8, jb - part * 8);
        }
      };
      auto update = [&](int i0) {
        for (int c = 0; c < cw; ++c) {
          T xb[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) xb[k] = part * 8 + k < jb ? X[c * n + k0 + part * 8 + k] : T(0);
#pragma unroll
          for (int w = 0; w < U; ++w) {
            const int i = i0 + w * (nt / 4) + (tid >> 2);
            T sum = T(0);
#pragma unroll
            for (int k = 0; k < 8; ++k)
              if (part * 8 + k < jb) sum += m[w][k] * xb[k];
            sum += __shfl_xor(sum, 1, 64);
            sum += __shfl_xor(sum, 2, 64);
            if (part == 0 && i < r1) X[c * n + i] -= sum;
          }
        }
      };
      load_rows(i00);
      if (wave < cw) {
        const int i = lane & 31;
        for (int c = wave; c < cw; c += nw) {
          T x = i < jb ? X[c * n + k0 + i] : T(0);
          if (pass == 0) {
#pragma unroll
            for (int k = 0; k < 32; ++k) {
              const T xk = lane_of(x, k);
              if (i > k) x -= l[k] * xk;
            }
          } else {
            T u = T(1);  // this lane's diagonal element
#pragma unroll
            for (int k = 0; k < 32; ++k) u = i == k && k < jb ? l[k] : u;
            const T r = T(1) / u;
            const bool plain = fabs(r) > Lim::min() * 4 && fabs(u) > Lim::min() * 4;
#pragma unroll
            for (int k = 31; k >= 0; --k) {
              if (k < jb) {  // uniform
                const T q0 = x * r, q1 = fma(fma(-q0, u, x), r, q0);
                T qx = q1;
                if (!plain || !(fabs(q1) <= Lim::max()) || fabs(x) < Lim::min() * 4 / Lim::epsilon())
                  qx = x / u;  // extremes (also where nothing is left: 0)
                if (i == k) x = qx;
                const T xk = lane_of(x, k);
                if (i < k) x -= l[k] * xk;
              }
            }
          }
          if (lane < 32 && i < jb) X[c * n + k0 + i] = x;
        }
        // the last block of the forward pass is the first of the backward one
        if (pass == 0 ? q + 1 < nb : q > 0) load_triangle(pass == 0 ? q + 1 : q - 1);
      }
      __syncthreads();
      update(i00);
      for (int i0 = i00 + U * (nt / 4); i0 < r1; i0 += U * (nt / 4)) {
        load_rows(i0);
        update(i0);
      }
      __syncthreads();
    }
  }
  for (int t = tid; t < n * cw; t += nt) B[(long long)(t / cw) * nrhs + t % cw] = X[(t % cw) * n + t / cw];
}

// Few unknowns (mmpi::solve_block_waves), and orders whose right-hand sides do
// not fit LDS: workgroup (b, y) handles right-hand sides [y * kRhsChunk, ...) of
// matrix b.
template <typename T>
__global__ __launch_bounds__(kT) void k_getrs(const T *__restrict__ lu, const int *__restrict__ piv,
                                              T *__restrict__ b, int n, int nrhs) {
  const T *A = lu + (long long)blockIdx.x * n * n;
  const int *P = piv + (long long)blockIdx.x * n;
  const int c0 = blockIdx.y * kRhsChunk;
  const int cw = nrhs - c0 < kRhsChunk ? nrhs - c0 : kRhsChunk;
  T *B = b + (long long)blockIdx.x * n * nrhs + c0;
  const int tid = threadIdx.x;
  for (int c = tid; c < cw; c += kT)
    for (int k = 0; k < n; ++k) {
      const int p = P[k];
      if (p != k) {
        const T t = B[(long long)k * nrhs + c];
        B[(long long)k * nrhs + c] = B[(long long)p * nrhs + c];
        B[(long long)p * nrhs + c] = t;
      }
    }
  __syncthreads();
  // thread -> (row group r0, column c) once, no division per element; the
  // r0 < rstep threads cover every (row group, column) pair exactly once
  const int c = tid % cw, r0 = tid / cw, rstep = kT / cw;
  for (int k = 0; k < n - 1; ++k) {
    if (r0 < rstep) {
      const T bk = B[(long long)k * nrhs + c];
      for (int i = k + 1 + r0; i < n; i += rstep) B[(long long)i * nrhs + c] -= A[(long long)i * n + k] * bk;
    }
    __syncthreads();
  }
  for (int k = n - 1; k >= 0; --k) {
    if (tid < cw) B[(long long)k * nrhs + tid] /= A[(long long)k * n + k];
    __syncthreads();
    if (r0 < rstep) {
      const T bk = B[(long long)k * nrhs + c];
      for (int i = r0; i < k; i += rstep) B[(long long)i * nrhs + c] -= A[(long long)i * n + k] * bk;
    }
    __syncthreads();
  }
}

// Panels of more rows than k_lu_panel holds: columns j0..j0+jb factored in
// memory with partial pivoting (one workgroup), k_laswp applies the row swaps
// to the other columns and k_trsm_ll forms U12 = L11^-1 A12 (one thread per
// column).
template <typename T>
__global__ __launch_bounds__(kT) void k_getf2_panel(T *__restrict__ a, int n, int j0, int jb,
                                                    int *__restrict__ piv, int *__restrict__ info) {
  T *P = a + (long long)j0 * n + j0;
  const int m = n - j0;
  __shared__ T sval[kT / 64];
  __shared__ int sidx[kT / 64];
  const int tid = threadIdx.x;
  int first_zero = 0;
  for (int k = 0; k < jb; ++k) {
    T best = T(-1);
    int bi = m;
    for (int i = k + tid; i < m; i += kT) {
      const T v = fabs(P[(long long)i * n + k]);
      if (v > best) {
        best = v;
        bi = i;
      }
    }
    for (int o = 32; o > 0; o >>= 1) {
      const T ov = __shfl_xor(best, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ov > best || (ov == best && oi < bi)) {
        best = ov;
        bi = oi;
      }
    }
    __syncthreads();
    if ((tid & 63) == 0) {
      sval[tid >> 6] = best;
      sidx[tid >> 6] = bi;
    }
    __syncthreads();
    best = sval[0];
    bi = sidx[0];
    for (int w = 1; w < kT / 64; ++w)
      if (sval[w] > best || (sval[w] == best && sidx[w] < bi)) {
        best = sval[w];
        bi = sidx[w];
      }
    const int p = bi < m ? bi : k;
    if (tid == 0) piv[j0 + k] = j0 + p;
    if (p != k)
      for (int j = tid; j < jb; j += kT) {
        const T t = P[(long long)k * n + j];
        P[(long long)k * n + j] = P[(long long)p * n + j];
        P[(long long)p * n + j] = t;
      }
    __syncthreads();
    const T d = P[(long long)k * n + k];
    if (d == T(0)) {
      if (!first_zero) first_zero = j0 + k + 1;
      continue;
    }
    for (int i = k + 1 + tid; i < m; i += kT) P[(long long)i * n + k] /= d;
    __syncthreads();
    // rank-1 update: lane = column (jb <= 64), wavefronts take rows in turn
    const int lane = tid & 63, wave = tid >> 6;
    if (lane < jb - k - 1) {
      const int j = k + 1 + lane;
      const T ukj = P[(long long)k * n + j];
      axpy_rows<T, kT / 64>(P + j, n, P + k, n, k + 1 + wave, m, ukj);
    }
    __syncthreads();
  }
  if (tid == 0) {
    if (j0 == 0) info[0] = first_zero;
    else if (info[0] == 0) info[0] = first_zero;
  }
}

template <typename T>
__global__ __launch_bounds__(kT) void k_laswp(T *__restrict__ a, int n, const int *__restrict__ piv,
                                              int k0, int k1) {
  const int c = blockIdx.x * kT + threadIdx.x;
  if (c >= n || (c >= k0 && c < k1)) return;  // the panel's own columns are swapped already
  for (int k = k0; k < k1; ++k) {
    const int p = piv[k];
    if (p != k) {
      const T t = a[(long long)k * n + c];
      a[(long long)k * n + c] = a[(long long)p * n + c];
      a[(long long)p * n + c] = t;
    }
  }
}

template <typename T>
__global__ __launch_bounds__(kT) void k_trsm_ll(T *__restrict__ a, int n, int j0, int jb) {
  const int c = j0 + jb + blockIdx.x * kT + threadIdx.x;
  if (c >= n) return;
  const T *L = a + (long long)j0 * n + j0;
  T *B = a + (long long)j0 * n;
  for (int i = 1; i < jb; ++i) {
    T s = B[(long long)i * n + c];
    for (int k = 0; k < i; ++k) s -= L[(long long)i * n + k] * B[(long long)k * n + c];
    B[(long long)i * n + c] = s;
  }
}

template <typename T, int W, int R>
void launch_panel(T *A, long long batch, int n, int j0, int jb, int *piv, int *info) {
  const int m = n - j0, nt = (mmpi::ceil_div(mmpi::ceil_div(m, R), 64)) * 64;
  hipLaunchKernelGGL((k_lu_panel<T, W, R>), dim3((unsigned)batch), dim3((unsigned)nt), 0,
                     mmpi::stream(), A, n, j0, jb, piv, info);
}

template <typename T>
int lu_blocked(int dtype, T *A, long long batch, int n, int *piv, int *info, bool in_order) {
  constexpr int F = 8 / (int)sizeof(T);  // float rows in the registers of a double row
  const long long nn = (long long)n * n;
  for (int j0 = 0, jb; j0 < n; j0 += jb) {
    const int m = n - j0;
    if (m > 2048 * F) {  // more rows than registers hold: in memory, matrix by matrix
      jb = kNb;
      const unsigned cgrid = (unsigned)mmpi::ceil_div(n, kT);
      for (long long b = 0; b < batch; ++b) {
        T *Ab = A + b * nn;
        int *Pb = piv + b * n;
        hipLaunchKernelGGL(k_getf2_panel<T>, dim3(1), dim3(kT), 0, mmpi::stream(), Ab, n, j0, jb, Pb,
                           info + b);
        hipLaunchKernelGGL(k_laswp<T>, dim3(cgrid), dim3(kT), 0, mmpi::stream(), Ab, n,
                           (const int *)Pb, j0, j0 + jb);
        hipLaunchKernelGGL(k_trsm_ll<T>, dim3((unsigned)mmpi::ceil_div(m - jb, kT)), dim3(kT), 0,
                           mmpi::stream(), Ab, n, j0, jb);
      }
    } else {
      // rows per thread by the panel's height; the width keeps a thread's
      // rows within 64 registers (of 256, pivot rows and loads beside them)
      const int w = m <= 512 * F ? 32 : m <= 1024 * F ? 16 : 8;
      jb = m < w ? m : w;
      if (m <= 512) launch_panel<T, 32, 1>(A, batch, n, j0, jb, piv, info);
      else if (m <= 512 * F) launch_panel<T, 32, F>(A, batch, n, j0, jb, piv, info);
      else if (m <= 1024 * F) launch_panel<T, 16, 2 * F>(A, batch, n, j0, jb, piv, info);
      else launch_panel<T, 8, 4 * F>(A, batch, n, j0, jb, piv, info);
      if (n > jb)
        hipLaunchKernelGGL(k_lu_swap<T>, dim3((unsigned)mmpi::ceil_div(n - jb, 64), (unsigned)batch),
                           dim3(kT), 0, mmpi::stream(), A, n, j0, jb, (const int *)piv);
    }
    if (int st = mmpi::check_launch("mmp_lu")) return st;
    const int n2 = n - j0 - jb;
    if (n2 > 0 && in_order) {
      const unsigned tiles = (unsigned)mmpi::ceil_div(n2, 64);
      for (int k = 0; k < jb; k += kLuW)
        hipLaunchKernelGGL(k_lu_update<T>, dim3(tiles * tiles, (unsigned)batch), dim3(kT), 0,
                           mmpi::stream(), A, n, j0 + k, jb - k < kLuW ? jb - k : kLuW, j0 + jb,
                           (int)tiles);
      if (int st = mmpi::check_launch("mmp_lu")) return st;
    } else if (n2 > 0) {
      T *P = A + (long long)j0 * n + j0;
      if (int st = mmpi::matmul_sub(dtype, batch, n2, n2, jb, P + (long long)jb * n, n, nn, P + jb, n,
                                    nn, P + (long long)jb * n + jb, n, nn))
        return st;
    }
  }
  return MMP_OK;
}

// -------------------------------------------------------------- Cholesky
template <typename T>
__global__ __launch_bounds__(kT) void k_sub_block(T *__restrict__ a, int n, int r0, int mr, int nc,
                                                  const T *__restrict__ c) {
  const long long tot = (long long)mr * nc;
  for (long long t = (long long)blockIdx.x * kT + threadIdx.x; t < tot; t += (long long)gridDim.x * kT) {
    const int i = (int)(t / nc), j = (int)(t % nc);
    a[(long long)(r0 + i) * n + r0 + j] -= c[t];
  }
}

template <typename T>
__global__ __launch_bounds__(kT) void k_potrf(T *__restrict__ a, int n, int *__restrict__ info) {
  T *A = a + (long long)blockIdx.x * n * n;
  const int tid = threadIdx.x;
  int bad = 0;
  for (int k = 0; k < n; ++k) {
    const T d = A[(long long)k * n + k];
    if (!(d > T(0))) {  // same value in every thread: a uniform exit
      bad = k + 1;
      break;
    }
    const T l = sqrt(d);
    __syncthreads();
    if (tid == 0) A[(long long)k * n + k] = l;
    for (int i = k + 1 + tid; i < n; i += kT) A[(long long)i * n + k] /= l;
    __syncthreads();
    const int m = n - k - 1;
    const long long mm = (long long)m * m;
    for (long long t = tid; t < mm; t += kT) {
      const int i = k + 1 + (int)(t / m), j = k + 1 + (int)(t % m);
      if (j <= i) A[(long long)i * n + j] -= A[(long long)i * n + k] * A[(long long)j * n + k];
    }
    __syncthreads();
  }
  const long long nn = (long long)n * n;
  for (long long t = tid; t < nn; t += kT)
    if ((int)(t % n) > (int)(t / n)) A[t] = T(0);
  if (tid == 0) info[blockIdx.x] = bad;
}

// ------------------------------------------------------ blocked Cholesky
// One n x n matrix, panels of kNb columns: the diagonal block is factored
// by one workgroup (k_potrf_diag), L21 = A21 L11^-T row by row
// (k_trsm_rlt, one thread per row), A22 -= L21 L21^T through the device
// matmul (L21^T staged by k_transpose_block) and k_sub_block; the strict
// upper triangle is zeroed at the end.
template <typename T>
__global__ __launch_bounds__(kT) void k_potrf_diag(T *__restrict__ a, int n, int j0, int jb,
                                                   int *__restrict__ info) {
  T *A = a + (long long)j0 * n + j0;
  const int tid = threadIdx.x;
  int bad = 0;
  if (info[0] != 0) return;  // an earlier panel failed: leave the rest
  for (int k = 0; k < jb; ++k) {
    const T d = A[(long long)k * n + k];
    if (!(d > T(0))) {
      bad = j0 + k + 1;
      break;
    }
    const T l = sqrt(d);
    __syncthreads();
    if (tid == 0) A[(long long)k * n + k] = l;
    for (int i = k + 1 + tid; i < jb; i += kT) A[(long long)i * n + k] /= l;
    __syncthreads();
    const int m = jb - k - 1;
    for (int t = tid; t < m * m; t += kT) {
      const int i = k + 1 + t / m, j = k + 1 + t % m;
      if (j <= i) A[(long long)i * n + j] -= A[(long long)i * n + k] * A[(long long)j * n + k];
    }
    __syncthreads();
  }
  if (tid == 0 && bad) info[0] = bad;
}

template <typename T>
__global__ __launch_bounds__(kT) void k_trsm_rlt(T *__restrict__ a, int n, int j0, int jb) {
  const int r = j0 + jb + blockIdx.x * kT + threadIdx.x;
  if (r >= n) return;
  const T *L = a + (long long)j0 * n + j0;
  T *X = a + (long long)r * n + j0;
  for (int k = 0; k < jb; ++k) {
    T s = X[k];
    for (int l = 0; l < k; ++l) s -= X[l] * L[(long long)k * n + l];
    X[k] = s / L[(long long)k * n + k];
  }
}

// out (jb x m2, contiguous) = transpose of A[r0 .. r0+m2)[j0 .. j0+jb)
template <typename T>
__global__ __launch_bounds__(kT) void k_transpose_block(const T *__restrict__ a, int n, int r0, int j0,
                                                        int m2, int jb, T *__restrict__ out) {
  const long long tot = (long long)m2 * jb;
  for (long long t = (long long)blockIdx.x * kT + threadIdx.x; t < tot; t += (long long)gridDim.x * kT) {
    const int k = (int)(t / m2), i = (int)(t % m2);
    out[t] = a[(long long)(r0 + i) * n + j0 + k];
  }
}

template <typename T>
__global__ __launch_bounds__(kT) void k_zero_upper(T *__restrict__ a, int n) {
  const long long tot = (long long)n * n;
  for (long long t = (long long)blockIdx.x * kT + threadIdx.x; t < tot; t += (long long)gridDim.x * kT)
    if ((int)(t % n) > (int)(t / n)) a[t] = T(0);
}

template <typename T>
__global__ void k_set_zero(int *__restrict__ p, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}

template <typename T>
int cholesky_blocked(int dtype, T *a, long long batch, int n, int *info) {
  const long long m2max = (long long)(n - kNb);
  void *tmp = nullptr, *tr = nullptr;
  if (m2max > 0) {
    if (int st = mmp_alloc((size_t)(m2max * m2max) * sizeof(T), &tmp)) return st;
    if (int st = mmp_alloc((size_t)(m2max * kNb) * sizeof(T), &tr)) {
      mmp_free(tmp);
      return st;
    }
  }
  hipLaunchKernelGGL(k_set_zero<T>, dim3(1), dim3(kT), 0, mmpi::stream(), info, (int)batch);
  int st = mmpi::check_launch("mmp_cholesky (blocked)");
  for (long long b = 0; b < batch && st == MMP_OK; ++b) {
    T *A = a + b * (long long)n * n;
    int *I = info + b;
    for (int j0 = 0; j0 < n && st == MMP_OK; j0 += kNb) {
      const int jb = n - j0 < kNb ? n - j0 : kNb;
      hipLaunchKernelGGL(k_potrf_diag<T>, dim3(1), dim3(kT), 0, mmpi::stream(), A, n, j0, jb, I);
      const int m2 = n - j0 - jb;
      if (m2 > 0) {
        hipLaunchKernelGGL(k_trsm_rlt<T>, dim3((unsigned)mmpi::ceil_div(m2, kT)), dim3(kT), 0,
                           mmpi::stream(), A, n, j0, jb);
        const long long g1 = mmpi::ceil_div((long long)m2 * jb, kT);
        hipLaunchKernelGGL(k_transpose_block<T>, dim3((unsigned)(g1 < 4096 ? g1 : 4096)), dim3(kT), 0,
                           mmpi::stream(), (const T *)A, n, j0 + jb, j0, m2, jb, (T *)tr);
        st = mmp_matmul(dtype, 1, m2, m2, jb, A + (long long)(j0 + jb) * n + j0, n, 0, tr, m2, 0, tmp,
                        m2, 0);
        if (st == MMP_OK) {
          const long long g = mmpi::ceil_div((long long)m2 * m2, kT);
          hipLaunchKernelGGL(k_sub_block<T>, dim3((unsigned)(g < 4096 ? g : 4096)), dim3(kT), 0,
                             mmpi::stream(), A, n, j0 + jb, m2, m2, (const T *)tmp);
        }
      }
      if (st == MMP_OK) st = mmpi::check_launch("mmp_cholesky (blocked)");
    }
    if (st == MMP_OK) {
      const long long g = mmpi::ceil_div((long long)n * n, kT);
      hipLaunchKernelGGL(k_zero_upper<T>, dim3((unsigned)(g < 4096 ? g : 4096)), dim3(kT), 0,
                         mmpi::stream(), A, n);
      st = mmpi::check_launch("mmp_cholesky (blocked)");
    }
  }
  if (tmp) mmp_free(tmp);
  if (tr) mmp_free(tr);
  return st;
}

// -------------------------------------------------------------------- QR
template <typename T>
__global__ __launch_bounds__(kT) void k_geqrf(T *__restrict__ a, int m, int n, T *__restrict__ tau) {
  const int kmin = m < n ? m : n;
  T *A = a + (long long)blockIdx.x * m * n;
  T *TAU = tau + (long long)blockIdx.x * kmin;
  __shared__ T red[kT / 64];
  __shared__ T part_lds[kT / 64][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int k = 0; k < kmin; ++k) {
    T part = T(0);
    for (int i = k + 1 + tid; i < m; i += kT) {
      const T v = A[(long long)i * n + k];
      part += v * v;
    }
    const T xn2 = block_sum<kT>(part, red);
    const T alpha = A[(long long)k * n + k];
    T t = T(0);
    if (xn2 != T(0)) {
      const T beta = -copysign(sqrt(alpha * alpha + xn2), alpha);
      t = (beta - alpha) / beta;
      const T sc = T(1) / (alpha - beta);
      __syncthreads();  // alpha read everywhere before A[k][k] changes
      for (int i = k + 1 + tid; i < m; i += kT) A[(long long)i * n + k] *= sc;
      if (tid == 0) A[(long long)k * n + k] = beta;
    }
    if (tid == 0) TAU[k] = t;
    __syncthreads();
    if (t != T(0)) {
      // lane = column of a 64-column chunk, wavefronts split the rows; the
      // four partial dot products meet in LDS
      for (int jc = k + 1; jc < n; jc += 64) {
        const int j = jc + lane;
        T part = T(0);
        if (j < n) {
#pragma unroll 8
          for (int i = k + 1 + wave; i < m; i += kT / 64) part += A[(long long)i * n + k] * A[(long long)i * n + j];
        }
        // A[k][j] is read by every wavefront before the barrier and
        // written by wavefront 0 after it
        const T akj = j < n ? A[(long long)k * n + j] : T(0);
        part_lds[wave][lane] = part;
        __syncthreads();
        if (j < n) {
          T w = akj;
          for (int q = 0; q < kT / 64; ++q) w += part_lds[q][lane];
          axpy_rows<T, kT / 64>(A + j, n, A + k, n, k + 1 + wave, m, t * w);
          if (wave == 0) A[(long long)k * n + j] = akj - t * w;
        }
        __syncthreads();
      }
    }
  }
}

template <typename T>
__global__ __launch_bounds__(kT) void k_orgqr(const T *__restrict__ a, const T *__restrict__ tau, int m,
                                              int n, int qc, T *__restrict__ q) {
  const int kmin = m < n ? m : n;
  const T *A = a + (long long)blockIdx.x * m * n;
  const T *TAU = tau + (long long)blockIdx.x * kmin;
  T *Q = q + (long long)blockIdx.x * m * qc;
  __shared__ T part_lds[kT / 64][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long long tot = (long long)m * qc;
  for (long long t = tid; t < tot; t += kT) Q[t] = (t / qc == t % qc) ? T(1) : T(0);
  __syncthreads();
  for (int k = kmin - 1; k >= 0; --k) {
    const T t = TAU[k];
    if (t == T(0)) continue;
    for (int jc = k; jc < qc; jc += 64) {
      const int j = jc + lane;
      T part = T(0);
      if (j < qc) {
#pragma unroll 8
        for (int i = k + 1 + wave; i < m; i += kT / 64) part += A[(long long)i * n + k] * Q[(long long)i * qc + j];
      }
      const T qkj = j < qc ? Q[(long long)k * qc + j] : T(0);
      part_lds[wave][lane] = part;
      __syncthreads();
      if (j < qc) {
        T w = qkj;
        for (int q = 0; q < kT / 64; ++q) w += part_lds[q][lane];
        axpy_rows<T, kT / 64>(Q + j, qc, A + k, n, k + 1 + wave, m, t * w);
        if (wave == 0) Q[(long long)k * qc + j] = qkj - t * w;
      }
      __syncthreads();
    }
  }
}

// ------------------------------------------------------ symmetric Jacobi
template <typename T>
__global__ __launch_bounds__(kJ) void k_syevj(T *__restrict__ a, T *__restrict__ v, int n,
                                              int *__restrict__ sweeps_out) {
  T *A = a + (long long)blockIdx.x * n * n;
  T *V = v + (long long)blockIdx.x * n * n;
  __shared__ T cs[kMaxEighN];  // (c, s) of each pair of the round
  __shared__ int s_rot;
  const int tid = threadIdx.x;
  const int N = n + (n & 1);
  const int npair = N / 2;
  const T eps = std::numeric_limits<T>::epsilon();
  const long long nn = (long long)n * n;
  for (long long t = tid; t < nn; t += kJ) V[t] = (t / n == t % n) ? T(1) : T(0);
  int sweep = 0;
  for (; sweep < kMaxSweeps; ++sweep) {
    if (tid == 0) s_rot = 0;
    __syncthreads();
    for (int r = 0; r < N - 1; ++r) {
      for (int pi = tid; pi < npair; pi += kJ) {
        int p, q;
        pair_of(r, pi, N, p, q);
        T c = T(1), s = T(0);
        if (p < n && q < n) {
          const T app = A[(long long)p * n + p], aqq = A[(long long)q * n + q];
          const T apq = A[(long long)p * n + q];
          if (apq != T(0) && fabs(apq) > eps * sqrt(fabs(app * aqq))) {
            const T th = (aqq - app) / (T(2) * apq);
            const T tt = (th >= T(0) ? T(1) : T(-1)) / (fabs(th) + sqrt(T(1) + th * th));
            c = T(1) / sqrt(T(1) + tt * tt);
            s = tt * c;
            if (s != T(0)) s_rot = 1;
          }
        }
        cs[2 * pi] = c;
        cs[2 * pi + 1] = s;
      }
      __syncthreads();
      const int work = npair * n;  // <= 2^21
      for (int t = tid; t < work; t += kJ) {
        const int pi = t / n, j = t - pi * n;  // lanes along a row: coalesced
        const T s = cs[2 * pi + 1];
        if (s == T(0)) continue;
        int p, q;
        pair_of(r, pi, N, p, q);
        const T c = cs[2 * pi];
        const T x = A[(long long)p * n + j], y = A[(long long)q * n + j];
        A[(long long)p * n + j] = c * x - s * y;
        A[(long long)q * n + j] = s * x + c * y;
      }
      __syncthreads();
      for (int t = tid; t < work; t += kJ) {
        // lanes over consecutive pairs of one row: the round-robin pairs
        // are runs of consecutive columns, so the accesses coalesce
        const int i = t / npair, pi = t - i * npair;
        const T s = cs[2 * pi + 1];
        if (s == T(0)) continue;
        int p, q;
        pair_of(r, pi, N, p, q);
        const T c = cs[2 * pi];
        const T x = A[(long long)i * n + p], y = A[(long long)i * n + q];
        A[(long long)i * n + p] = c * x - s * y;
        A[(long long)i * n + q] = s * x + c * y;
        const T vx = V[(long long)i * n + p], vy = V[(long long)i * n + q];
        V[(long long)i * n + p] = c * vx - s * vy;
        V[(long long)i * n + q] = s * vx + c * vy;
      }
      __syncthreads();
    }
    const int rotated = s_rot;
    __syncthreads();
    if (!rotated) break;
  }
  if (tid == 0) sweeps_out[blockIdx.x] = sweep;
}

// ------------------------------------------------------ one-sided Jacobi
template <typename T>
__global__ __launch_bounds__(kJ) void k_gesvj(T *__restrict__ w, T *__restrict__ vt, int r, int L,
                                              int *__restrict__ sweeps_out) {
  T *W = w + (long long)blockIdx.x * r * L;
  T *VT = vt + (long long)blockIdx.x * r * r;
  __shared__ int s_rot;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int N = r + (r & 1);
  const int npair = N / 2;
  const T eps = std::numeric_limits<T>::epsilon();
  const long long rr = (long long)r * r;
  for (long long t = tid; t < rr; t += kJ) VT[t] = (t / r == t % r) ? T(1) : T(0);
  int sweep = 0;
  for (; sweep < kMaxSweeps; ++sweep) {
    if (tid == 0) s_rot = 0;
    __syncthreads();
    for (int rd = 0; rd < N - 1; ++rd) {
      for (int pi = wave; pi < npair; pi += kJ / 64) {
        int p, q;
        pair_of(rd, pi, N, p, q);
        if (p >= r || q >= r) continue;
        T al = T(0), be = T(0), ga = T(0);
#pragma unroll 8
        for (int j = lane; j < L; j += 64) {
          const T x = W[(long long)p * L + j], y = W[(long long)q * L + j];
          al += x * x;
          be += y * y;
          ga += x * y;
        }
        al = wave_sum(al);
        be = wave_sum(be);
        ga = wave_sum(ga);
        if (ga != T(0) && fabs(ga) > eps * sqrt(al * be)) {
          const T ze = (be - al) / (T(2) * ga);
          const T tt = (ze >= T(0) ? T(1) : T(-1)) / (fabs(ze) + sqrt(T(1) + ze * ze));
          const T c = T(1) / sqrt(T(1) + tt * tt), s = c * tt;
          if (s != T(0)) {
            rotate_rows(W + (long long)p * L, W + (long long)q * L, L, lane, c, s);
            rotate_rows(VT + (long long)p * r, VT + (long long)q * r, r, lane, c, s);
            if (lane == 0) s_rot = 1;
          }
        }
      }
      __syncthreads();
    }
    const int rotated = s_rot;
    __syncthreads();
    if (!rotated) break;
  }
  if (tid == 0) sweeps_out[blockIdx.x] = sweep;
}

int check_common(const char *what, int dtype, long long batch) {
  if (dtype != MMP_F32 && dtype != MMP_F64)
    return mmpi::fail(MMP_E_UNSUPPORTED, "%s: dtype %d (float32 / float64 only)", what, dtype);
  if (batch < 0 || batch > 0x7fffffffll) return mmpi::fail(MMP_E_ARG, "%s: batch %lld", what, batch);
  return MMP_OK;
}

}  // namespace

extern "C" int mmp_lu(int dtype, void *a, int64_t batch, int64_t n, int32_t *piv, int32_t *info) {
  if (int st = mmpi::ensure_init()) return st;
  if (int st = check_common("mmp_lu", dtype, batch)) return st;
  if (n < 0 || n > 32768) return mmpi::fail(MMP_E_ARG, "mmp_lu: n %lld", (long long)n);
  if (batch == 0 || n == 0) return MMP_OK;
  if (!a || !piv || !info) return mmpi::fail(MMP_E_ARG, "mmp_lu: null pointer");
  // few large matrices: their arithmetic is worth the matrix cores
  const bool in_order = n < kBlockedMinN || batch > kBlockedMaxBatch;
  for (int64_t b0 = 0; b0 < batch; b0 += 65535) {  // a grid dimension's limit
    const int64_t nb = batch - b0 < 65535 ? batch - b0 : 65535;
    int *P = (int *)piv + b0 * n, *I = (int *)info + b0;
    const int st = dtype == MMP_F32
                       ? lu_blocked<float>(dtype, (float *)a + b0 * n * n, nb, (int)n, P, I, in_order)
                       : lu_blocked<double>(dtype, (double *)a + b0 * n * n, nb, (int)n, P, I, in_order);
    if (st) return st;
  }
  return MMP_OK;
}

extern "C" int mmp_lu_solve(int dtype, const void *lu, const int32_t *piv, void *b, int64_t batch,
                            int64_t n, int64_t nrhs) {
  if (int st = mmpi::ensure_init()) return st;
  if (int st = check_common("mmp_lu_solve", dtype, batch)) return st;
  if (n < 0 || n > 32768 || nrhs < 0 || nrhs > 0x7fffffffll)
    return mmpi::fail(MMP_E_ARG, "mmp_lu_solve: n %lld nrhs %lld", (long long)n, (long long)nrhs);
  if (batch == 0 || n == 0 || nrhs == 0) return MMP_OK;
  if (!lu || !piv || !b) return mmpi::fail(MMP_E_ARG, "mmp_lu_solve: null pointer");
  const size_t lds = (size_t)n * (size_t)(nrhs < kRhs ? nrhs : kRhs) * (dtype == MMP_F32 ? 4 : 8);
  const int waves = mmpi::solve_block_waves(batch, (int)n, (int)(nrhs < 0x7fffffff ? nrhs : 0x7fffffff),
                                            dtype == MMP_F32 ? 4 : 8,
                                            mmpi::cu_count() > 0 ? mmpi::cu_count() : 256);
  if (waves && lds <= kSolveLds && mmpi::ceil_div(nrhs, kRhs) <= 65535) {
    const dim3 g((unsigned)batch, (unsigned)mmpi::ceil_div(nrhs, kRhs));
    const dim3 t(64 * waves);
    if (dtype == MMP_F32)
      hipLaunchKernelGGL(k_lu_solve<float>, g, t, lds, mmpi::stream(), (const float *)lu,
                         (const int *)piv, (float *)b, (int)n, (int)nrhs);
    else
      hipLaunchKernelGGL(k_lu_solve<double>, g, t, lds, mmpi::stream(), (const double *)lu,
                         (const int *)piv, (double *)b, (int)n, (int)nrhs);
    return mmpi::check_launch("mmp_lu_solve");
  }
  const dim3 grid((unsigned)batch, (unsigned)mmpi::ceil_div(nrhs, kRhsChunk));
  if (grid.y > 65535) return mmpi::fail(MMP_E_ARG, "mmp_lu_solve: nrhs %lld too large", (long long)nrhs);
  if (dtype == MMP_F32)
    hipLaunchKernelGGL(k_getrs<float>, grid, dim3(kT), 0, mmpi::stream(),
                       (const float *)lu, (const int *)piv, (float *)b, (int)n, (int)nrhs);
  else
    hipLaunchKernelGGL(k_getrs<double>, grid, dim3(kT), 0, mmpi::stream(),
                       (const double *)lu, (const int *)piv, (double *)b, (int)n, (int)nrhs);
  return mmpi::check_launch("mmp_lu_solve");
}

extern "C" int mmp_cholesky(int dtype, void *a, int64_t batch, int64_t n, int32_t *info) {
  if (int st = mmpi::ensure_init()) return st;
  if (int st = check_common("mmp_cholesky", dtype, batch)) return st;
  if (n < 0 || n > 32768) return mmpi::fail(MMP_E_ARG, "mmp_cholesky: n %lld", (long long)n);
  if (batch == 0 || n == 0) return MMP_OK;
  if (!a || !info) return mmpi::fail(MMP_E_ARG, "mmp_cholesky: null pointer");
  if (n >= kBlockedMinN && batch <= kBlockedMaxBatch)
    return dtype == MMP_F32 ? cholesky_blocked<float>(dtype, (float *)a, batch, (int)n, (int *)info)
                            : cholesky_blocked<double>(dtype, (double *)a, batch, (int)n, (int *)info);
  if (dtype == MMP_F32)
    hipLaunchKernelGGL(k_potrf<float>, dim3((unsigned)batch), dim3(kT), 0, mmpi::stream(), (float *)a,
                       (int)n, (int *)info);
  else
    hipLaunchKernelGGL(k_potrf<double>, dim3((unsigned)batch), dim3(kT), 0, mmpi::stream(), (double *)a,
                       (int)n, (int *)info);
  return mmpi::check_launch("mmp_cholesky");
}

extern "C" int mmp_qr(int dtype, void *a, void *tau, int64_t batch, int64_t m, int64_t n) {
  if (int st = mmpi::ensure_init()) return st;
  if (int st = check_common("mmp_qr", dtype, batch)) return st;
  if (m < 0 || n < 0 || m > 0x7fffffffll || n > 0x7fffffffll)
    return mmpi::fail(MMP_E_ARG, "mmp_qr: shape %lld x %lld", (long long)m, (long long)n);
  if (batch == 0 || m == 0 || n == 0) return MMP_OK;
  if (!a || !tau) return mmpi::fail(MMP_E_ARG, "mmp_qr: null pointer");
  if (dtype == MMP_F32)
    hipLaunchKernelGGL(k_geqrf<float>, dim3((unsigned)batch), dim3(kT), 0, mmpi::stream(), (float *)a,
                       (int)m, (int)n, (float *)tau);
  else
    hipLaunchKernelGGL(k_geqrf<double>, dim3((unsigned)batch), dim3(kT), 0, mmpi::stream(), (double *)a,
                       (int)m, (int)n, (double *)tau);
  return mmpi::check_launch("mmp_qr");
}

extern "C" int mmp_qr_q(int dtype, const void *a, const void *tau, int64_t batch, int64_t m, int64_t n,
                        int64_t qcols, void *q) {
  if (int st = mmpi::ensure_init()) return st;
  if (int st = check_common("mmp_qr_q", dtype, batch)) return st;
  const long long kmin = m < n ? m : n;
  if (m < 0 || n < 0 || m > 0x7fffffffll || n > 0x7fffffffll || qcols < kmin || qcols > m)
    return mmpi::fail(MMP_E_ARG, "mmp_qr_q: shape %lld x %lld, qcols %lld", (long long)m,
                      (long long)n, (long long)qcols);
  if (batch == 0 || m == 0 || qcols == 0) return MMP_OK;
  if (!a || !tau || !q) return mmpi::fail(MMP_E_ARG, "mmp_qr_q: null pointer");
  if (dtype == MMP_F32)
    hipLaunchKernelGGL(k_orgqr<float>, dim3((unsigned)batch), dim3(kT), 0, mmpi::stream(),
                       (const float *)a, (const float *)tau, (int)m, (int)n, (int)qcols, (float *)q);
  else
    hipLaunchKernelGGL(k_orgqr<double>, dim3((unsigned)batch), dim3(kT), 0, mmpi::stream(),
                       (const double *)a, (const double *)tau, (int)m, (int)n, (int)qcols, (double *)q);
  return mmpi::check_launch("mmp_qr_q");
}

extern "C" int mmp_eigh(int dtype, void *a, void *v, int64_t batch, int64_t n, int32_t *sweeps) {
  if (int st = mmpi::ensure_init()) return st;
  if (int st = check_common("mmp_eigh", dtype, batch)) return st;
  if (n < 0 || n > kMaxEighN) return mmpi::fail(MMP_E_ARG, "mmp_eigh: n %lld (at most %d)", (long long)n, kMaxEighN);
  if (batch == 0 || n == 0) return MMP_OK;
  if (!a || !v || !sweeps) return mmpi::fail(MMP_E_ARG, "mmp_eigh: null pointer");
  if (dtype == MMP_F32)
    hipLaunchKernelGGL(k_syevj<float>, dim3((unsigned)batch), dim3(kJ), 0, mmpi::stream(), (float *)a,
                       (float *)v, (int)n, (int *)sweeps);
  else
    hipLaunchKernelGGL(k_syevj<double>, dim3((unsigned)batch), dim3(kJ), 0, mmpi::stream(), (double *)a,
                       (double *)v, (int)n, (int *)sweeps);
  return mmpi::check_launch("mmp_eigh");
}

extern "C" int mmp_svd(int dtype, void *w, void *vt, int64_t batch, int64_t rows, int64_t len,
                       int32_t *sweeps) {
  if (int st = mmpi::ensure_init()) return st;
  if (int st = check_common("mmp_svd", dtype, batch)) return st;
  if (rows < 0 || rows > kMaxSvdRows || len < rows || len > 0x7fffffffll)
    return mmpi::fail(MMP_E_ARG, "mmp_svd: rows %lld len %lld (rows <= len, rows <= %d)", (long long)rows,
                      (long long)len, kMaxSvdRows);
  if (batch == 0 || rows == 0) return MMP_OK;
  if (!w || !vt || !sweeps) return mmpi::fail(MMP_E_ARG, "mmp_svd: null pointer");
  if (dtype == MMP_F32)
    hipLaunchKernelGGL(k_gesvj<float>, dim3((unsigned)batch), dim3(kJ), 0, mmpi::stream(), (float *)w,
                       (float *)vt, (int)rows, (int)len, (int *)sweeps);
  else
    hipLaunchKernelGGL(k_gesvj<double>, dim3((unsigned)batch), dim3(kJ), 0, mmpi::stream(), (double *)w,
                       (double *)vt, (int)rows, (int)len, (int *)sweeps);
  return mmpi::check_launch("mmp_svd");
}
