// Triangular solves with an upper-triangular R whose data was packed once
// for the lanes that use it: R^T y = b ("adjoint") and R x = b ("forward"),
// n <= 64 * TP_MAX_NB, by one 512-thread workgroup.
//
// What bounds a solve is the chain through the diagonal, and past n of about
// 500 the rate at which one CU reads R (about 130 GB/s: 1.2 MB at n = 512 is 9
// us).  Both directions are lower-triangular solves L y = b with L = R^T, or
// L = R with rows and columns reversed over the padded size N = 64 nb.  Block
// row I (64 rows, lane = row) belongs to wavefront I % 8 and keeps its right-
// hand side in one register per lane.  As soon as block t's solution is in LDS
// (a flag there, no barrier), every later row subtracts its 64 x 64 product
// from registers that were loaded one block ahead, so the chain per block is
// one 64 x 64 product, the diagonal solve and one LDS hand-over.
//
// The packing makes every load 1 KiB of consecutive doubles: block (I, J) is
// stored two columns at a time (64 rows of two), blocks of a row one after
// another, row after row.  The diagonal block stores, in its columns 0..47, the columns of
// L below the 16 x 16 diagonal sub-blocks (zeros elsewhere), and in columns
// 48..63 the sub-block of the lane's own 16 rows: rows 0..7 hold the inverse
// of the upper 8 x 8 half in columns 0..7, rows 8..15 the coupling in columns
// 0..7 and the inverse of the lower half in columns 8..15.  The solve of 16
// rows is then three 8-term products inside a 16-lane DPP row.  Inverting 8 x
// 8 blocks only keeps the application error at u kappa(8 x 8 block), the
// accuracy of substitution for the triangles of a sketch (wider inverses,
// with u kappa(64 x 64 block), raised LSQR's attainable backward error).
//
// Measured, one solve (with its launch): 24 -> 8 us at n = 200, 40 -> 12.6 at
// 333, 60 -> 17.4 at 512, 164 -> 58 at 1024, against one workgroup that stages
// 64 x 64 diagonal blocks in LDS and solves them on one wavefront between
// barriers (trsv_dev.h, kept for larger n and for the batched solves).
// Packing both directions takes 7 us.
#pragma once

#include "common.h"

constexpr int TP_MAX_NB = 16;           // block rows: two per wavefront
constexpr int64_t TP_MAX_N = 64 * TP_MAX_NB;
constexpr int TP_WAVES = 8;
constexpr int TP_THREADS = 64 * TP_WAVES;
constexpr int TP_BLOCK = 64 * 64;       // doubles of one packed block

__host__ __device__ inline int tp_nb(int64_t n) { return (int)pamd_cdiv(n, 64); }
// doubles of one packed direction
__host__ __device__ inline int64_t tp_doubles(int64_t n) {
  const int64_t nb = tp_nb(n);
  return nb * (nb + 1) / 2 * TP_BLOCK;
}

namespace {

// v in lane C of this lane's 16-lane row, for every lane of the row
template <int C>
__device__ __forceinline__ double tp_row_bcast(double v) {
  return __longlong_as_double(__builtin_amdgcn_update_dpp(0LL, __double_as_longlong(v), 0x150 + C, 0xf, 0xf, true));
}

// lanes 16 Q .. 16 Q + 15 of v copied to every 16-lane row
template <int Q>
__device__ __forceinline__ double tp_spread_row(double v) {
  const long long b = __double_as_longlong(v);
  unsigned w[2] = {(unsigned)(b & 0xffffffffLL), (unsigned)((unsigned long long)b >> 32)};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    // halves (lo, lo) / (hi, hi), then even / odd rows doubled
    const auto h = __builtin_amdgcn_permlane32_swap(w[i], w[i], false, false);
    const unsigned x = (Q & 2) ? h[1] : h[0];
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    w[i] = (Q & 1) ? r[1] : r[0];
  }
  return __longlong_as_double((long long)(((unsigned long long)w[1] << 32) | w[0]));
}

template <int C0, int N>
struct TpDot {  // s[c & 1] += bcast_c(x) d[c], c = C0 .. C0 + N - 1 (two chains)
  static __device__ __forceinline__ void run(double x, const double* d, double& s0, double& s1) {
    if constexpr (N > 0) {
      if constexpr (C0 & 1)
        s1 = fma(tp_row_bcast<C0>(x), d[C0], s1);
      else
        s0 = fma(tp_row_bcast<C0>(x), d[C0], s0);
      TpDot<C0 + 1, N - 1>::run(x, d, s0, s1);
    }
  }
};

// sum_{c = C0}^{C0 + N - 1} x[c of this lane's row] d[c]
template <int C0, int N>
__device__ __forceinline__ double tp_dot(double x, const double* d) {
  double s0 = 0.0, s1 = 0.0;
  TpDot<C0, N>::run(x, d, s0, s1);
  return s0 + s1;
}

// rows 16 Q .. of the diagonal block: the solution of its 16 rows to y's
// lanes, the rows below updated in acc
template <int Q>
__device__ __forceinline__ void tp_diag16(const double (&buf)[64], int lane, double& acc, double& y) {
  const double* d = buf + 48;
  const double s = tp_dot<0, 8>(acc, d);              // rows 0..7: the solution
  const double u = acc - tp_dot<0, 8>(s, d);          // rows 8..15: right-hand side of the lower half
  const double z = tp_dot<8, 8>(u, d);                // rows 8..15: the solution
  const double xl = (lane & 8) ? z : s;
  y = ((lane >> 4) == Q) ? xl : y;
  if constexpr (Q < 3) acc -= tp_dot<0, 16>(tp_spread_row<Q>(xl), buf + 16 * Q);
}

// A packed direction as a buffer: one descriptor in scalar registers, the
// block's byte offset scalar, so 64 loads in flight need one address register.
typedef unsigned tp_u4 __attribute__((ext_vector_type(4)));

struct TpBuf {
  __amdgpu_buffer_rsrc_t r;
  int lane16;  // this lane's byte offset
};

__device__ __forceinline__ TpBuf tp_buf(const double* P, int nb, int lane) {
  const unsigned bytes = (unsigned)(nb * (nb + 1) / 2 * TP_BLOCK * sizeof(double));  // at most 4.5 MB
  return TpBuf{__builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(P), 0, bytes, 0x00020000), lane * 16};
}

// byte offset of block (I, J)
__device__ __forceinline__ int tp_off(int I, int J) { return (I * (I + 1) / 2 + J) * (TP_BLOCK * 8); }

// columns 16 C .. 16 C + 15 of the block at byte offset off
template <int C>
__device__ __forceinline__ void tp_load16(double (&buf)[64], const TpBuf& P, int off) {
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const tp_u4 v = __builtin_amdgcn_raw_buffer_load_b128(P.r, P.lane16, off + (8 * C + q) * 1024, 0);
    buf[16 * C + 2 * q] = __longlong_as_double((long long)(((unsigned long long)v[1] << 32) | v[0]));
    buf[16 * C + 2 * q + 1] = __longlong_as_double((long long)(((unsigned long long)v[3] << 32) | v[2]));
  }
}

__device__ __forceinline__ void tp_load(double (&buf)[64], const TpBuf& P, int off) {
  tp_load16<0>(buf, P, off);
  tp_load16<1>(buf, P, off);
  tp_load16<2>(buf, P, off);
  tp_load16<3>(buf, P, off);
}

// until block t's solution is in LDS
__device__ __forceinline__ void tp_wait(const int* ready, int t) {
  while (__hip_atomic_load(ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) <= t) {
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// acc -= (block in buf) x_t once block t's solution is there; buf is reloaded
// from byte offset `next` as it is used
template <int C>
__device__ __forceinline__ void tp_update16(double (&buf)[64], const TpBuf& P, int next, double xv, double& s) {
  s += tp_dot<0, 16>(xv, buf + 16 * C);
  __builtin_amdgcn_sched_barrier(0);  // the loads below go to the registers just used
  tp_load16<C>(buf, P, next);
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ void tp_update(double (&buf)[64], const TpBuf& P, int next, int t, const double* xs,
                                          const int* ready, int lane, double& acc) {
  tp_wait(ready, t);
  double xv[4], s = 0.0;
#pragma unroll
  for (int c = 0; c < 4; ++c) xv[c] = xs[64 * t + 16 * c + (lane & 15)];
  tp_update16<0>(buf, P, next, xv[0], s);
  tp_update16<1>(buf, P, next, xv[1], s);
  tp_update16<2>(buf, P, next, xv[2], s);
  tp_update16<3>(buf, P, next, xv[3], s);
  acc -= s;
}

// the diagonal block t: acc's solution, published in xs
__device__ __forceinline__ void tp_diag(const double (&buf)[64], int t, double* xs, int* ready, int lane,
                                        double& acc) {
  double y = 0.0;
  tp_diag16<0>(buf, lane, acc, y);
  tp_diag16<1>(buf, lane, acc, y);
  tp_diag16<2>(buf, lane, acc, y);
  tp_diag16<3>(buf, lane, acc, y);
  acc = y;
  xs[64 * t + lane] = y;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  if (lane == 0) __hip_atomic_store(ready, t + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// the first block of a wavefront's rows, started before its right-hand side is known
__device__ __forceinline__ void tp_prefetch(double (&buf)[64], const TpBuf& P, int nb, int wave) {
  if (wave < nb) tp_load(buf, P, tp_off(wave, 0));
}

// L y = acc for wavefront `wave` (uniform) of TP_WAVES.  buf holds its first
// block (tp_prefetch); acc[k] the right-hand side of block
// row wave + 8 k (0 past n), on return its solution.  xs: 64 nb doubles of
// LDS for the solution; ready: an LDS counter that is 0 on entry for every
// wavefront (the caller's barrier).  Block t's owner needs only blocks before
// t, so every wait ends.  A wavefront returns when its own rows are done: a
// barrier is needed before another wavefront's part of xs is overwritten.
template <int K>
__device__ __forceinline__ void tp_solve(int nb, const TpBuf& P, double (&buf)[64], double (&acc)[K], double* xs,
                                         int* ready, int wave, int lane) {
  static_assert(K == 1 || K == 2, "one or two block rows per wavefront");
  if (wave >= nb) return;
  const int I1 = wave, I2 = wave + TP_WAVES;
  if constexpr (K == 1) {
    for (int t = 0; t < I1; ++t) tp_update(buf, P, tp_off(I1, t + 1), t, xs, ready, lane, acc[0]);
    tp_diag(buf, I1, xs, ready, lane, acc[0]);
  } else {
    // the products in the order of the solution blocks they need: (I1, t) and
    // (I2, t) for t < I1, row I1's diagonal, (I2, t) for the rest, its diagonal.
    // One place reloads buf: with more the compiler keeps copies of it and spills.
    const bool two = I2 < nb;
    int row = 0, I = I1, t = 0;
#pragma unroll 1
    for (;;) {
      double a = row ? acc[1] : acc[0];
      int nI = I, nt = t + 1, nrow = row;
      if (t < I) {
        tp_wait(ready, t);
        double s = 0.0;
#pragma unroll
        for (int c = 0; c < 4; ++c) s += tp_dot<0, 16>(xs[64 * t + 16 * c + (lane & 15)], buf + 16 * c);
        a -= s;
        if (two && t < I1) {  // the other row's product while both are open
          nrow = 1 - row;
          nI = nrow ? I2 : I1;
          nt = t + row;
        }
      } else {
        tp_diag(buf, t, xs, ready, lane, a);
        nrow = 1;
        nI = I2;
        nt = t;
      }
      if (row)
        acc[1] = a;
      else
        acc[0] = a;
      if (t == I && (row || !two)) return;
      __builtin_amdgcn_sched_barrier(0);
      tp_load(buf, P, tp_off(nI, nt));
      __builtin_amdgcn_sched_barrier(0);
      row = nrow;
      I = nI;
      t = nt;
    }
  }
}

// Packing.  Workgroup b (256 threads) of tp_pack_blocks(nb) packs block b of
// both directions: the adjoint's first, then the forward's.
__host__ __device__ inline int tp_pack_blocks(int nb) { return nb * (nb + 1); }

// position of (row i, column c) inside a packed block
__device__ __forceinline__ int tp_pos(int i, int c) { return (c >> 1) * 128 + 2 * i + (c & 1); }

__global__ __launch_bounds__(256) void tp_pack_kernel(int n, const double* __restrict__ R, int64_t ldr,
                                                      double* __restrict__ Padj, double* __restrict__ Pfwd) {
  __shared__ double T[64][65];  // T[i][j] = L(64 I + i, 64 J + j)
  const int nb = tp_nb(n);
  const int per = nb * (nb + 1) / 2;
  const bool fwd = (int)blockIdx.x >= per;
  const int b = (int)blockIdx.x - (fwd ? per : 0);
  int I = 0;
  while ((I + 1) * (I + 2) / 2 <= b) ++I;
  const int J = b - I * (I + 1) / 2;
  double* __restrict__ P = (fwd ? Pfwd : Padj) + (int64_t)b * TP_BLOCK;
  // the block of R this is, read row by row: rows r0.., columns c0..
  const int r0 = 64 * (fwd ? nb - 1 - I : J), c0 = 64 * (fwd ? nb - 1 - J : I);
  double v[TP_BLOCK / 256];
#pragma unroll
  for (int q = 0; q < TP_BLOCK / 256; ++q) {
    const int r = r0 + ((threadIdx.x + 256 * q) >> 6), c = c0 + (threadIdx.x & 63);
    // the triangle inside n; the identity beyond
    v[q] = (r < n && c < n && r <= c) ? R[(int64_t)r * ldr + c] : (r == c && r >= n ? 1.0 : 0.0);
  }
#pragma unroll
  for (int q = 0; q < TP_BLOCK / 256; ++q) {
    const int i = (threadIdx.x + 256 * q) >> 6, j = threadIdx.x & 63;
    if (fwd)
      T[63 - i][63 - j] = v[q];
    else
      T[j][i] = v[q];
  }
  __syncthreads();
  if (I != J) {
    for (int e = threadIdx.x; e < TP_BLOCK; e += 256) {
      const int i = (e >> 1) & 63, c = 2 * (e >> 7) + (e & 1);
      P[e] = T[i][c];
    }
    return;
  }
  for (int e = threadIdx.x; e < 48 * 64; e += 256) {
    const int i = (e >> 1) & 63, c = 2 * (e >> 7) + (e & 1);
    P[e] = (i >> 4) > (c >> 4) ? T[i][c] : 0.0;
  }
  // 16 x 16 sub-blocks: thread = (sub-block q, half h, column j) inverts column j of one 8 x 8 half by forward
  // substitution and copies the coupling's column
  if (threadIdx.x < 64) {
    const int q = threadIdx.x >> 4, h = (threadIdx.x >> 3) & 1, j = threadIdx.x & 7;
    const int o = 16 * q + 8 * h;
    double z[8], rd[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) rd[i] = 1.0 / T[o + i][o + i];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      double s = (i == j) ? 1.0 : 0.0;
#pragma unroll
      for (int k = 0; k < i; ++k) s -= (k >= j) ? T[o + i][o + k] * z[k] : 0.0;
      z[i] = (i >= j) ? s * rd[i] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) P[tp_pos(o + i, 48 + 8 * h + j)] = z[i];
    // the other half's rows of these columns: the coupling (lower rows, columns of the upper half) or zero
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 16 * q + 8 * (1 - h) + i;
      P[tp_pos(r, 48 + 8 * h + j)] = (h == 0) ? T[r][o + j] : 0.0;
    }
  }
}

// out = R^{-T} in (trans) or R^{-1} in from the packed direction P; in may be out
template <int K>
__global__ __launch_bounds__(TP_THREADS) void tp_solve_kernel(int trans, int n, const double* __restrict__ P,
                                                              const double* in, double* out) {
  __shared__ double xs[64 * TP_WAVES * K];
  __shared__ int ready;
  const int nb = tp_nb(n), N = 64 * nb;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const TpBuf B = tp_buf(P, nb, lane);
  double buf[64], acc[K];
  tp_prefetch(buf, B, nb, wave);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int r = 64 * (wave + TP_WAVES * k) + lane;
    const int i = trans ? r : N - 1 - r;
    acc[k] = (i >= 0 && i < n) ? in[i] : 0.0;
  }
  if (threadIdx.x == 0) ready = 0;
  __syncthreads();
  tp_solve<K>(nb, B, buf, acc, xs, &ready, wave, lane);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int r = 64 * (wave + TP_WAVES * k) + lane;
    const int i = trans ? r : N - 1 - r;
    if (i >= 0 && i < n) out[i] = acc[k];
  }
}

inline int tp_launch_pack(int n, const double* R, int64_t ldr, double* Padj, double* Pfwd, hipStream_t st) {
  tp_pack_kernel<<<(unsigned)tp_pack_blocks(tp_nb(n)), 256, 0, st>>>(n, R, ldr, Padj, Pfwd);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

inline int tp_launch_solve(int trans, int n, const double* P, const double* in, double* out, hipStream_t st) {
  if (n <= 64 * TP_WAVES)
    tp_solve_kernel<1><<<1, TP_THREADS, 0, st>>>(trans, n, P, in, out);
  else
    tp_solve_kernel<2><<<1, TP_THREADS, 0, st>>>(trans, n, P, in, out);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

}  // namespace
