// Upper Cholesky A = R^T R of one matrix by one 512-thread workgroup with the
// trailing triangle in registers (n <= 16 * PR_MAXT).
//
// What bounds it is the chain of 16-column steps: diagonal factor, the block
// row, the next diagonal tile's update.  The upper triangle's 16 x 16 tiles
// live in the accumulator registers of wavefronts 1..7 (tile t of the
// row-by-row enumeration belongs to wavefront 1 + t % 7, so every step's
// remaining tiles are spread evenly) from the load to the step that finishes
// them, and nothing but the finished row passes through LDS.  The result
// layout of v_mfma_f64_16x16x4f64 (lane l, item r: row l / 16 + 4 r, column
// l % 16) is both its A^T and its B operand layout, so a row tile X = R_kj
// is stored to LDS as it lies in the registers and read back as either
// operand of the updates A_ij -= R_ki^T R_kj without a transpose.
// Wavefront 0 owns no tile: it factors the next diagonal tile, handed over
// through LDS as soon as it is updated, while the others finish the step.
//
// A diagonal tile is factored with one column per lane (16 lanes, the four
// rows of the wavefront redundant): the row of R and the pivot reach the other
// lanes by DPP broadcast, one instruction each.  Its inverse is applied in two
// 8-row halves, x_a = Ra^-T g_a, x_b = Rb^-T (g_b - C^T x_a), as two K = 8
// products; only 8 x 8 blocks are inverted, so the block row has the accuracy
// of substitution up to kappa(8 x 8 block).
//
// Measured: 97 -> 47 us at n = 200, 46 -> 19 at 100, 21 -> 10 at 64, against
// the trailing matrix in global memory, 32-column blocks factored through LDS
// (440 cycles a column, here 130) and substitution by one thread per column.
// A step is about 6500 cycles, 3200 of them the diagonal tile; n = 200 spends
// a third of its time on the first four steps' products.
#pragma once

#include "common.h"

typedef double d4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int PR_B = 16;
constexpr int PR_MAXT = 13;                    // tiles per dimension: n <= 208
constexpr int PR_MAXN = PR_B * PR_MAXT;
constexpr int PR_WORKERS = 7;
constexpr int PR_THREADS = 64 * (1 + PR_WORKERS);

struct PrShared {
  double row[PR_MAXT][64 * 4];  // the finished row's tiles, lane by lane
  double diag[PR_B][PR_B + 1];  // the tile wavefront 0 factors, diag[column][row]
  double m1[8][PR_B];           // [k][m]: (Ra^-1)[k][m] for m < 8, -(Ra^-1 C)[k][m - 8] for m >= 8
  double m2[8][PR_B];           // [k][m]: 0 for m < 8, (Rb^-1)[k][m - 8] for m >= 8
  int handed;                   // diagonal tiles handed to wavefront 0
  int bad;
};

// v in lane C of this lane's 16-lane row
template <int C>
__device__ __forceinline__ double pr_bcast(double v) {
  return __longlong_as_double(__builtin_amdgcn_update_dpp(0LL, __double_as_longlong(v), 0x150 + C, 0xf, 0xf, true));
}

// v of lane (l + 8) % 16 of this lane's row (row_ror:8)
__device__ __forceinline__ double pr_swap8(double v) { return dpp_f64<0x128>(v); }

template <int J, int I>
struct PrUpd {  // col[i] -= R[j][i] R[j][c] for i = I..15
  static __device__ __forceinline__ void run(double (&col)[PR_B], double v) {
    if constexpr (I < PR_B) {
      col[I] = fma(-pr_bcast<I>(v), v, col[I]);
      PrUpd<J, I + 1>::run(col, v);
    }
  }
};

// columns J..15 of the 16 x 16 factor; col: this lane's column, row J.. of it
// still to be reduced; on return col[j] = R[j][c] (junk for j > c) and
// rinv[j] = 1 / R_jj.  A pivot that is not positive and finite leaves rinv[j]
// zero, infinite or NaN (pr_fail).  The step is a chain of latencies, so 1 /
// sqrt(d) takes one third-order correction of the hardware estimate (relative
// error e^3 of about 2^-26 cubed) instead of two Newton steps: four dependent
// operations instead of six.
template <int J>
__device__ __forceinline__ void pr_factor(double (&col)[PR_B], double (&rinv)[PR_B]) {
  if constexpr (J < PR_B) {
    const double d = pr_bcast<J>(col[J]);
    const double y0 = __builtin_amdgcn_rsq(d);
    const double e = fma(-d * y0, y0, 1.0);
    const double y = fma(y0 * e, fma(e, 0.375, 0.5), y0);
    rinv[J] = y;
    const double v = col[J] * y;
    col[J] = v;
    PrUpd<J, J + 1>::run(col, v);
    pr_factor<J + 1>(col, rinv);
  }
}

// the first column whose pivot failed, plus one, or 0.  A failed pivot makes
// its row NaN in every lane and so every later pivot: the last one tells
__device__ __forceinline__ int pr_fail(const double (&rinv)[PR_B]) {
  const bool ok = rinv[PR_B - 1] > 0.0 && rinv[PR_B - 1] < INFINITY;
  if (__builtin_amdgcn_readfirstlane(ok)) return 0;
  int fail = 0;
#pragma unroll
  for (int j = PR_B - 1; j >= 0; --j) fail = (rinv[j] > 0.0 && rinv[j] < INFINITY) ? fail : j + 1;
  return __builtin_amdgcn_readfirstlane(fail);
}

// z <- (8 x 8 upper triangle with column k in lane k's h)^-1 z, one right-hand
// side per lane; ri[i] the diagonal's reciprocals
template <int I>
__device__ __forceinline__ void pr_back8(const double (&h)[8], const double (&ri)[8], double (&z)[8]) {
  if constexpr (I >= 0) {
    z[I] *= ri[I];
    // rows above: z_i -= R[i][I] z_I
    [&]<int... Q>(std::integer_sequence<int, Q...>) {
      ((z[Q] = fma(-pr_bcast<I>(h[Q]), z[I], z[Q])), ...);
    }(std::make_integer_sequence<int, I>{});
    pr_back8<I - 1>(h, ri, z);
  }
}

// Wavefront 0: factors the tile in s.diag; col: this lane's column of R's
// tile; the operands of the block row to s.m1, s.m2.  Returns 0 or the failing
// column + 1.
__device__ __forceinline__ int pr_diag(PrShared& s, int lane, double (&col)[PR_B]) {
  const int c = lane & 15, row = lane >> 4;
  double rinv[PR_B];
#pragma unroll
  for (int i = 0; i < PR_B; ++i) col[i] = s.diag[c][i];
  pr_factor<0>(col, rinv);
  // lane row 0 works on Ra with the right-hand sides e_c (c < 8) and C's
  // columns (c >= 8); lane row 1 on Rb, its columns moved down eight lanes
  double h[8], ri[8], z[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const double hb = pr_swap8(col[8 + i]);
    h[i] = row == 0 ? col[i] : hb;
    ri[i] = row == 0 ? rinv[i] : rinv[8 + i];
    z[i] = (row == 0 && c >= 8) ? col[i] : (c == i ? 1.0 : 0.0);
  }
  pr_back8<7>(h, ri, z);
  if (row == 0) {
#pragma unroll
    for (int k = 0; k < 8; ++k) s.m1[k][c] = c < 8 ? z[k] : -z[k];
  } else if (row == 1 && c < 8) {
#pragma unroll
    for (int k = 0; k < 8; ++k) s.m2[k][8 + c] = z[k];
  }
  return pr_fail(rinv);
}

// R's tile (rows / columns i0.., inside n) to A; lane row q stores rows 4 q .. 4 q + 3
__device__ __forceinline__ void pr_store_diag(const double (&col)[PR_B], double* __restrict__ A, int64_t lda, int n,
                                              int i0, int lane) {
  const int c = lane & 15, row = lane >> 4;
  if (i0 + c >= n) return;
  double* a = A + (int64_t)(i0 + 4 * row) * lda + i0 + c;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const double lo = (row & 1) ? col[4 + r] : col[r], hi = (row & 1) ? col[12 + r] : col[8 + r];
    if (4 * row + r <= c) a[r * lda] = (row & 2) ? hi : lo;
  }
}

// A tile index, opaque to the optimiser: the addresses formed from it inside
// the step loop are not hoisted out of it (two registers per tile and operand)
__device__ __forceinline__ int pr_opaque(int t) {
  asm volatile("" : "+s"(t));
  return t;
}

// one tile of the block row k: X = R_kk^-T A_kj to s.row and to A
__device__ __forceinline__ void pr_row_tile(PrShared& s, const d4& g, const double (&a1)[2], const double (&a2)[2],
                                            int k, int tj, int n, int lane, double* __restrict__ A, int64_t lda,
                                            int64_t off) {
  d4 u = {0.0, 0.0, g[2], g[3]};
  u = __builtin_amdgcn_mfma_f64_16x16x4f64(a1[0], g[0], u, 0, 0, 0);
  u = __builtin_amdgcn_mfma_f64_16x16x4f64(a1[1], g[1], u, 0, 0, 0);
  d4 x = {u[0], u[1], 0.0, 0.0};
  x = __builtin_amdgcn_mfma_f64_16x16x4f64(a2[0], u[2], x, 0, 0, 0);
  x = __builtin_amdgcn_mfma_f64_16x16x4f64(a2[1], u[3], x, 0, 0, 0);
  double* d = s.row[tj] + lane * 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) d[r] = x[r];
  if (PR_B * tj + (lane & 15) < n) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      (A + (int64_t)(PR_B * k + 4 * r) * lda + PR_B * tj)[off] = x[r];
  }
}

// A_ij -= R_ki^T R_kj for tile t
__device__ __forceinline__ void pr_update_tile(const PrShared& s, d4& acc, int t, int lane) {
  const double* x = s.row[t & 255] + lane * 4;
  const double* y = s.row[t >> 8] + lane * 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-x[r], y[r], acc, 0, 0, 0);
}

// diagonal tile k, fully updated, to wavefront 0
__device__ __forceinline__ void pr_hand_over(PrShared& s, const d4& acc, int k, int lane) {
#pragma unroll
  for (int r = 0; r < 4; ++r) s.diag[lane & 15][(lane >> 4) + 4 * r] = acc[r];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  if (lane == 0) __hip_atomic_store(&s.handed, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// SL tiles per worker wavefront: SL * 7 >= T (T + 1) / 2.  The two roles are
// separate code paths with the same barriers (2 + 2 per step), so that neither
// holds the other's registers.
template <int SL>
__device__ __forceinline__ void potrf_reg(int n, double* __restrict__ A, int64_t lda, int* __restrict__ info,
                                          int lead) {
  __shared__ PrShared s;
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int T = (n + PR_B - 1) / PR_B;
  if (wave == 0) {
    if (lane == 0) {
      s.handed = 0;
      s.bad = 0;
    }
    for (int e = lane; e < 8 * PR_B; e += 64) s.m2[e >> 4][e & 15] = 0.0;
    __syncthreads();
    double col[PR_B];
    int bad = pr_diag(s, lane, col);
    if (lane == 0) s.bad = bad;
    __syncthreads();
    for (int k = 0; k + 1 < T && !bad; ++k) {
      pr_store_diag(col, A, lda, n, PR_B * k, lane);  // while the workers form the block row
      __syncthreads();
      while (__hip_atomic_load(&s.handed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) <= k) {
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
      const int fail = pr_diag(s, lane, col);
      if (fail) bad = PR_B * (k + 1) + fail;
      if (lane == 0) s.bad = bad;
      __syncthreads();  // the workers' updates
    }
    if (!bad) pr_store_diag(col, A, lda, n, PR_B * (T - 1), lane);
    if (lane == 0) info[0] = bad ? lead + bad : 0;
    return;
  }

  // this wavefront's tiles, row + 256 * column; row T for a slot without one (never reached by a step)
  int tij[SL];
  d4 acc[SL];
  const int64_t off = lk * lda + lr;  // this lane inside a tile's first four rows
  {
    int i = 0, first = 0;  // row i's tiles are first .. first + T - i - 1
#pragma unroll
    for (int q = 0; q < SL; ++q) {
      const int t = wave - 1 + PR_WORKERS * q;
      while (i < T && t >= first + T - i) first += T - i++;
      const int j = i + t - first;
      tij[q] = i + 256 * j;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int a = PR_B * i + lk + 4 * r, b = PR_B * j + lr;
        // the upper triangle inside n, the identity beyond
        acc[q][r] = a == b ? 1.0 : 0.0;
        if (i < T && a <= b && b < n)
          acc[q][r] = (A + (int64_t)(PR_B * i + 4 * r) * lda + PR_B * j)[off];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (wave == 1) {  // tile 0
#pragma unroll
    for (int r = 0; r < 4; ++r) s.diag[lr][lk + 4 * r] = acc[0][r];
  }
  __syncthreads();
  __syncthreads();
  int first_open = 0;  // this wavefront's first slot of a row not yet finished
  for (int k = 0; k + 1 < T; ++k) {
    if (s.bad) return;
    // the block row: X = R_kk^-T A_kj
    double a1[2], a2[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      a1[q] = s.m1[4 * q + lk][lr];
      a2[q] = s.m2[4 * q + lk][lr];
    }
    // The wavefront's tiles are in row order, so a step's are consecutive
    // slots: a jump to the first one (a test per slot cost 50 cycles each).
#define PR_ROW(Q)                                                                             \
  case Q:                                                                                     \
    if constexpr (Q < SL) {                                                                   \
      const int t = pr_opaque(tij[Q]), tj = t >> 8;                                           \
      if ((t & 255) != k) break;                                                              \
      ++first_open;                                                                           \
      if (tj != k) pr_row_tile(s, acc[Q], a1, a2, k, tj, n, lane, A, lda, off);               \
    }                                                                                         \
    [[fallthrough]];
    switch (first_open) {
      PR_ROW(0) PR_ROW(1) PR_ROW(2) PR_ROW(3) PR_ROW(4) PR_ROW(5) PR_ROW(6) PR_ROW(7) PR_ROW(8) PR_ROW(9)
      PR_ROW(10) PR_ROW(11) PR_ROW(12)
      default: break;
    }
#undef PR_ROW
    __syncthreads();
    // the updates; the next diagonal tile, its owner's first open one, is handed over at once
#define PR_UPD(Q)                                                                             \
  case Q:                                                                                     \
    if constexpr (Q < SL) {                                                                   \
      const int t = pr_opaque(tij[Q]);                                                        \
      if ((t & 255) >= T) break;                                                              \
      pr_update_tile(s, acc[Q], t, lane);                                                     \
      if (t == 257 * (k + 1)) pr_hand_over(s, acc[Q], k + 1, lane);                           \
    }                                                                                         \
    [[fallthrough]];
    switch (first_open) {
      PR_UPD(0) PR_UPD(1) PR_UPD(2) PR_UPD(3) PR_UPD(4) PR_UPD(5) PR_UPD(6) PR_UPD(7) PR_UPD(8) PR_UPD(9)
      PR_UPD(10) PR_UPD(11) PR_UPD(12)
      default: break;
    }
#undef PR_UPD
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// n > PR_MAXN: right-looking over PR_LEAD rows at a time.  The leading rows by
// the kernel above, their block row R12 = R11^-T A12 (one workgroup per 16
// columns), A22 -= R12^T R12 (one wavefront per 16 x 16 tile), then the
// trailing matrix.  The middle steps use the whole chip and take about 8 us
// each; one workgroup's matrix cores would need 40 us for the updates of n =
// 266 alone (n = 266: 78 us this way, 87 with all of it in one workgroup's
// registers, 150 in one with the matrix in memory; n = 512: 165 against 736).
// ---------------------------------------------------------------------------
constexpr int PR_LEAD = 128;
constexpr int PR_LT = PR_LEAD / PR_B;

// tiles per dimension behind the leading rows
__host__ __device__ inline int pr_trailing(int n) { return (n - PR_LEAD + PR_B - 1) / PR_B; }

struct PrRowShared {
  double x[PR_LT][64 * 4];     // the solved tiles of this block column, lane by lane
  double part[3][64 * 4];      // partial sums of wavefronts 1..3
  double m1[PR_LT][8][PR_B], m2[PR_LT][8][PR_B];
};

// 16 columns c0.. of R12 by one 256-thread workgroup: X_I = R_II^-T (A_I -
// sum_{J < I} R_JI^T X_J), the sum split over the wavefronts by J
__device__ __forceinline__ void pr_block_column(int n, double* __restrict__ A, int64_t lda, int c0) {
  __shared__ PrRowShared s;
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the 8 x 8 inverses and couplings of R11's diagonal tiles, as in pr_diag
  for (int t = wave; t < PR_LT; t += 4) {
    double h[8], ri[8], z[8];
    const int o = PR_B * t + (lk == 1 ? 8 : 0);  // lane row 1: the lower half
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      h[i] = A[(int64_t)(o + i) * lda + o + (lr & 7)];
      z[i] = (lk == 0 && lr >= 8) ? A[(int64_t)(o + i) * lda + o + lr] : (lr == i ? 1.0 : 0.0);
    }
    double rd[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) rd[i] = 1.0 / h[i];  // lane i holds 1 / R_ii in rd[i]
    ri[0] = pr_bcast<0>(rd[0]);
    ri[1] = pr_bcast<1>(rd[1]);
    ri[2] = pr_bcast<2>(rd[2]);
    ri[3] = pr_bcast<3>(rd[3]);
    ri[4] = pr_bcast<4>(rd[4]);
    ri[5] = pr_bcast<5>(rd[5]);
    ri[6] = pr_bcast<6>(rd[6]);
    ri[7] = pr_bcast<7>(rd[7]);
    pr_back8<7>(h, ri, z);
    if (lk == 0) {
#pragma unroll
      for (int k = 0; k < 8; ++k) s.m1[t][k][lr] = lr < 8 ? z[k] : -z[k];
    } else if (lk == 1) {
#pragma unroll
      for (int k = 0; k < 8; ++k) s.m2[t][k][(lr + 8) & 15] = lr < 8 ? z[k] : 0.0;
    }
  }
  const bool in = c0 + lr < n;
  double* col = A + c0 + lr;
  __syncthreads();
  for (int I = 0; I < PR_LT; ++I) {
    constexpr int NU = (PR_LT + 3) / 4;  // tiles of a sum per wavefront
    double g[4], r[NU][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) g[q] = (wave == 0 && in) ? col[(int64_t)(PR_B * I + 4 * q + lk) * lda] : 0.0;
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int J = wave + 4 * u;
        r[u][q] = J < I ? A[(int64_t)(PR_B * J + 4 * q + lk) * lda + PR_B * I + lr] : 0.0;
      }
    d4 acc = {g[0], g[1], g[2], g[3]};
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int J = wave + 4 * u;
      if (J >= I) break;
      const double* x = s.x[J] + lane * 4;
#pragma unroll
      for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-r[u][q], x[q], acc, 0, 0, 0);
    }
    if (wave > 0) {
#pragma unroll
      for (int q = 0; q < 4; ++q) s.part[wave - 1][lane * 4 + q] = acc[q];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int w = 0; w < 3; ++w)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] += s.part[w][lane * 4 + q];
      d4 u = {0.0, 0.0, acc[2], acc[3]};
      u = __builtin_amdgcn_mfma_f64_16x16x4f64(s.m1[I][lk][lr], acc[0], u, 0, 0, 0);
      u = __builtin_amdgcn_mfma_f64_16x16x4f64(s.m1[I][4 + lk][lr], acc[1], u, 0, 0, 0);
      d4 x = {u[0], u[1], 0.0, 0.0};
      x = __builtin_amdgcn_mfma_f64_16x16x4f64(s.m2[I][lk][lr], u[2], x, 0, 0, 0);
      x = __builtin_amdgcn_mfma_f64_16x16x4f64(s.m2[I][4 + lk][lr], u[3], x, 0, 0, 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        s.x[I][lane * 4 + q] = x[q];
        if (in) col[(int64_t)(PR_B * I + 4 * q + lk) * lda] = x[q];
      }
    }
    __syncthreads();
  }
}

// tile t (row by row) of the trailing upper triangle A22 -= R12^T R12 by one wavefront
__device__ __forceinline__ void pr_trailing_tile(int n, double* __restrict__ A, int64_t lda, int t) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int T = pr_trailing(n);
  int i = 0;
  while (t >= T - i) t -= T - i++;
  const int a0 = PR_LEAD + PR_B * i, b0 = PR_LEAD + PR_B * (i + t);
  const bool ain = a0 + lr < n, bin = b0 + lr < n;
  d4 acc[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
  for (int k0 = 0; k0 < PR_LEAD; k0 += 32) {
    double a[8], b[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const double* r = A + (int64_t)(k0 + 4 * q + lk) * lda;
      a[q] = ain ? r[a0 + lr] : 0.0;
      b[q] = bin ? r[b0 + lr] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 8; ++q)
      acc[q & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q], b[q], acc[q & 1], 0, 0, 0);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = a0 + 4 * q + lk;
    if (r <= b0 + lr && bin) A[(int64_t)r * lda + b0 + lr] -= acc[0][q] + acc[1][q];
  }
}

// Whether an n x n matrix fits the small instantiation (6 tiles per worker
// wavefront, n <= 128; the large one has 13).  Fewer registers, so that
// several batched problems share a CU.
constexpr int PR_SMALL = 6, PR_LARGE = 13;
__host__ __device__ inline bool pr_small(int n) { return n <= 128; }
static_assert(PR_MAXT * (PR_MAXT + 1) / 2 <= PR_LARGE * PR_WORKERS && 8 * 9 / 2 <= PR_SMALL * PR_WORKERS, "tiles");

// Rows from j0 on that are factored in one go (0: all done before j0)
__host__ __device__ inline int pr_width(int n, int j0) {
  if (j0 > 0 && n - (j0 - PR_LEAD) <= PR_MAXN) return 0;
  return n - j0 <= PR_MAXN ? n - j0 : PR_LEAD;
}

}  // namespace
