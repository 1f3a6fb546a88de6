// R and z = Q^T S b of a sketch M = [S A | S b] by CholeskyQR, every step a
// launch and nothing read back in between.
//
// A Householder QR of the sketch is bound by the latency of its panels (one
// barrier per column or more: 0.86 ms at 800 x 201, 2.5 ms at 2048 x 513).
// CholeskyQR2 does the same work as Gram products and strip solves over the
// whole chip and leaves only two k x k factorisations to latency:
//   G = Y^T Y, R1 = chol(G), Q1 = Y R1^{-1};  [Q1^T Q1 | w] = Q1^T [Q1 | S b];
//   R2 = chol(Q1^T Q1): Newton's two steps for I + E, or potrf;
//   R = R2 R1, z = R2^{-T} w.
// Y = S A, or, for an S A too ill conditioned for that, Y = S A R0^{-1} with
// R0 the Cholesky factor of the shifted Gram matrix (Fukaya, Kannan, Nakatsukasa,
// Yamamoto and Yanagisawa 2020: stable up to kappa about 1 / u), and R = R2 R1
// R0.  The caller reads four numbers once and decides whether the result
// stands: the failing pivots and ||Q1^T Q1 - I||_F, which measures what the
// first round lost.
//
// With that read, R and z of 400 x 101 / 800 x 201 / 2048 x 513 take 172 / 227
// / 495 us (Householder: 408 / 842 / 2498); in the shifted form, after the
// first form has failed, 345 / 487 / 1095; Householder after both 680 / 1223 /
// 3343.  A form that fails costs its Gram matrix and the pivots before the
// failing one; with the rest of its chain run to the end the last two rows were
// 395 / 539 / 1250 and 754 / 1344 / 3683.
#include "common.h"

namespace {

constexpr int64_t RZ_MAX_N = 1024;  // the strip solve and the packed triangular solve
constexpr int RZ_PARTS = 256;      // workgroups of the ||E|| partial sums

struct RzLayout {
  int64_t Q, G0, G, QtQ, T, U, dinv, gw, tri, part, info, total;  // offsets in doubles
  int64_t gw_bytes;
};

int64_t rz_round(int64_t x) { return (x + 31) / 32 * 32; }

int rz_layout(int64_t d, int64_t n, RzLayout* L) {
  int64_t b, gw = 0;
  const int64_t shapes[3][3] = {{n, n, d}, {n, n + 1, d}, {n, n, n}};
  for (const auto& s : shapes) {
    const int rc = pamd_gemm_workspace(s[0], s[1], s[2], &b);
    if (rc) return rc;
    gw = imax64(gw, b);
  }
  int64_t o = 0;
  auto take = [&](int64_t doubles) {
    const int64_t at = o;
    o += rz_round(doubles);
    return at;
  };
  L->Q = take(d * (n + 1));        // [Q1 | S b]; before, S A R0^{-1} of the shifted form in Q1's place
  L->G0 = take(n * n);             // R0 (shifted form)
  L->G = take(n * n);              // R1
  L->QtQ = take(n * (n + 1));      // [Q1^T Q1 | w]
  L->T = take(n * n);
  L->U = take(n * n);
  L->dinv = take(pamd_cdiv(n, 16) * 256);
  L->gw_bytes = gw;
  L->gw = take(gw / 8 + 1);
  const int rc = pamd_trsv_pack_workspace(n, &b);
  if (rc) return rc;
  L->tri = take(b / 8);
  L->part = take(RZ_PARTS);
  L->info = take(4);
  L->total = o;
  return PAMD_OK;
}

// [.. | S b]: column n of Q from column n of M; infos to 0
__global__ __launch_bounds__(256) void rz_init_kernel(int64_t d, int64_t n, const double* __restrict__ M, int64_t ldm,
                                                      double* __restrict__ Q, int* __restrict__ info) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < d) Q[i * (n + 1) + n] = M[i * ldm + n];
  if (blockIdx.x == 0 && threadIdx.x < 4) info[threadIdx.x] = 0;
}

// G += 11 (d n + n (n + 1)) u trace(G) I
__global__ __launch_bounds__(256) void rz_shift_kernel(int64_t d, int64_t n, double* __restrict__ G) {
  __shared__ double red[4];
  double t = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 256) t += G[i * n + i];
  t = block_sum(t, red);
  const double shift = 11.0 * ((double)d * (double)n + (double)n * (double)(n + 1)) * 0x1p-53 * t;
  for (int64_t i = threadIdx.x; i < n; i += 256) G[i * n + i] += shift;
}

// G's strictly lower part to zero (U <- triu(G)); with QtQ: X = H(QtQ - I)
// (upper triangle, halved diagonal) and this workgroup's part of ||QtQ - I||_F^2
__global__ __launch_bounds__(256) void rz_newton_kernel(int n, const double* __restrict__ QtQ, double* __restrict__ G,
                                                        double* __restrict__ X, double* __restrict__ part) {
  __shared__ double red[4];
  const int total = n * n;
  double ss = 0.0;
  for (int e = blockIdx.x * 256 + threadIdx.x; e < total; e += gridDim.x * 256) {
    const int i = e / n, j = e - i * n;
    if (j < i) G[e] = 0.0;
    const double v = QtQ[(int64_t)i * (n + 1) + j] - (i == j ? 1.0 : 0.0);
    ss += v * v;
    X[e] = j > i ? v : (j == i ? 0.5 * v : 0.0);
  }
  ss = block_sum(ss, red);
  if (threadIdx.x == 0) part[blockIdx.x] = ss;
}

// R2 = I + H(QtQ - I - X^T X)
__global__ __launch_bounds__(256) void rz_r2_kernel(int n, const double* __restrict__ QtQ,
                                                    const double* __restrict__ XtX, double* __restrict__ R2) {
  const int total = n * n;
  for (int e = blockIdx.x * 256 + threadIdx.x; e < total; e += gridDim.x * 256) {
    const int i = e / n, j = e - i * n;
    const double v = QtQ[(int64_t)i * (n + 1) + j] - (i == j ? 1.0 : 0.0) - XtX[e];
    R2[e] = j > i ? v : (j == i ? 1.0 + 0.5 * v : 0.0);
  }
}

// R2 <- triu(QtQ's n columns) (after its potrf)
__global__ __launch_bounds__(256) void rz_triu_kernel(int n, const double* __restrict__ QtQ, int64_t ld,
                                                      double* __restrict__ R2) {
  const int total = n * n;
  for (int e = blockIdx.x * 256 + threadIdx.x; e < total; e += gridDim.x * 256) {
    const int i = e / n, j = e - i * n;
    R2[e] = j >= i ? QtQ[(int64_t)i * ld + j] : 0.0;
  }
}

// stats = (min |R1_ii|, max |R1_ii|, ||Q1^T Q1 - I||_F, first failing pivot or 0);
// z <- w (column n of QtQ)
__global__ __launch_bounds__(256) void rz_stats_kernel(int n, const double* __restrict__ G,
                                                       const double* __restrict__ QtQ, int parts,
                                                       const double* __restrict__ part, const int* __restrict__ info,
                                                       double* __restrict__ z, double* __restrict__ stats) {
  __shared__ double red[4], smin[4], smax[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double mn = INFINITY, mx = 0.0;
  for (int i = tid; i < n; i += 256) {
    const double v = fabs(G[(int64_t)i * n + i]);
    mn = fmin(mn, v);
    mx = fmax(mx, v);
    z[i] = QtQ[(int64_t)i * (n + 1) + n];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    mn = fmin(mn, __shfl_xor(mn, off, 64));
    mx = fmax(mx, __shfl_xor(mx, off, 64));
  }
  if (lane == 0) {
    smin[wave] = mn;
    smax[wave] = mx;
  }
  const double ss = block_sum(tid < parts ? part[tid] : 0.0, red);
  if (tid == 0) {
    for (int w = 1; w < 4; ++w) {
      mn = fmin(mn, smin[w]);
      mx = fmax(mx, smax[w]);
    }
    stats[0] = mn;
    stats[1] = mx;
    stats[2] = sqrt(ss);
    stats[3] = (double)(info[0] ? info[0] : info[1] ? info[1] : info[2]);
  }
}

#define RZ_TRY(expr)         \
  do {                       \
    const int rc_ = (expr);  \
    if (rc_) return rc_;     \
  } while (0)

}  // namespace

extern "C" int pamd_sketch_rz_workspace(int64_t d, int64_t n, int64_t* bytes) {
  PAMD_ARG_CHECK(n >= 1 && n <= RZ_MAX_N, 2);
  PAMD_ARG_CHECK(d >= n && d < ((int64_t)1 << 31), 1);
  PAMD_ARG_CHECK(bytes != nullptr, 3);
  RzLayout L;
  RZ_TRY(rz_layout(d, n, &L));
  *bytes = L.total * (int64_t)sizeof(double);
  return PAMD_OK;
}

extern "C" int pamd_sketch_rz_f64(int64_t d, int64_t n, const double* M, int64_t ldm, int shifted, int newton,
                                  double* R, int64_t ldr, double* z, double* stats, void* workspace, void* stream) {
  PAMD_ARG_CHECK(n >= 1 && n <= RZ_MAX_N, 2);
  PAMD_ARG_CHECK(d >= n && d < ((int64_t)1 << 31), 1);
  PAMD_ARG_CHECK(M != nullptr, 3);
  PAMD_ARG_CHECK(ldm >= n + 1, 4);
  PAMD_ARG_CHECK(shifted == 0 || shifted == 1, 5);
  PAMD_ARG_CHECK(newton >= 0 && newton <= 2, 6);
  PAMD_ARG_CHECK(R != nullptr, 7);
  PAMD_ARG_CHECK(ldr >= n, 8);
  PAMD_ARG_CHECK(z != nullptr, 9);
  PAMD_ARG_CHECK(stats != nullptr, 10);
  PAMD_ARG_CHECK(workspace != nullptr, 11);
  hipStream_t st = (hipStream_t)stream;
  RzLayout L;
  RZ_TRY(rz_layout(d, n, &L));
  double* ws = (double*)workspace;
  double *Q = ws + L.Q, *G = ws + L.G, *QtQ = ws + L.QtQ, *T = ws + L.T, *U = ws + L.U;
  int* info = (int*)(ws + L.info);
  const unsigned eg = (unsigned)imin64(RZ_PARTS, pamd_cdiv(n * n, 1024));
  // Everything after the first round's potrf is left out on the device when a pivot failed there (info[0]), so that a
  // sketch that has to be factored otherwise pays for its Gram matrix and the pivots before the failing one
  auto gemm = [&](int ta, int64_t m, int64_t nn, int64_t k, const double* A, int64_t lda, const double* B, int64_t ldb,
                  double* C, int64_t ldc, const int* skip) {
    return pamd_gemm_cin_f64(ta, 0, m, nn, k, 1.0, A, lda, B, ldb, 0.0, C, ldc, C, ldc, ws + L.gw, L.gw_bytes, stream,
                             skip);
  };
  if (newton != 2) {
    rz_init_kernel<<<(unsigned)pamd_cdiv(d, 256), 256, 0, st>>>(d, n, M, ldm, Q, info);
    PAMD_LAUNCH_CHECK();
    const double* Y = M;
    int64_t ldy = ldm;
    if (shifted) {
      double* G0 = ws + L.G0;
      RZ_TRY(gemm(1, n, n, d, M, ldm, M, ldm, G0, n, nullptr));
      rz_shift_kernel<<<1, 256, 0, st>>>(d, n, G0);
      PAMD_LAUNCH_CHECK();
      RZ_TRY(pamd_potrf_run((int)n, G0, n, info + 2, stream));
      RZ_TRY(pamd_trsm_strip_run(d, (int)n, G0, n, M, ldm, Q, n + 1, ws + L.dinv, stream));
      Y = Q;  // the next strip solve is in place: a workgroup holds its 16 rows in LDS before it stores them
      ldy = n + 1;
    }
    RZ_TRY(gemm(1, n, n, d, Y, ldy, Y, ldy, G, n, nullptr));
    RZ_TRY(pamd_potrf_run((int)n, G, n, info, stream));
    RZ_TRY(pamd_trsm_strip_run(d, (int)n, G, n, Y, ldy, Q, n + 1, ws + L.dinv, stream, info));
    RZ_TRY(gemm(1, n, n + 1, d, Q, n + 1, Q, n + 1, QtQ, n + 1, info));
    rz_newton_kernel<<<eg, 256, 0, st>>>((int)n, QtQ, G, T, ws + L.part);  // T = X = H(E)
    PAMD_LAUNCH_CHECK();
  }
  // the first round stays in the workspace (G = R1, QtQ, the norm's parts) for a second call with newton = 2
  if (newton == 1) {
    RZ_TRY(gemm(1, n, n, n, T, n, T, n, U, n, info));
    rz_r2_kernel<<<eg, 256, 0, st>>>((int)n, QtQ, U, T);  // T = R2
    PAMD_LAUNCH_CHECK();
  } else {
    RZ_TRY(pamd_potrf_run((int)n, QtQ, n + 1, info + 1, stream));
    rz_triu_kernel<<<eg, 256, 0, st>>>((int)n, QtQ, n + 1, T);
    PAMD_LAUNCH_CHECK();
  }
  rz_stats_kernel<<<1, 256, 0, st>>>((int)n, G, QtQ, (int)eg, ws + L.part, info, z, stats);
  PAMD_LAUNCH_CHECK();
  RZ_TRY(pamd_trsv_pack_f64(n, T, n, ws + L.tri, stream));
  if (shifted) {
    RZ_TRY(gemm(0, n, n, n, T, n, G, n, U, n, info));
    rz_triu_kernel<<<eg, 256, 0, st>>>((int)n, ws + L.G0, n, T);
    PAMD_LAUNCH_CHECK();
    RZ_TRY(gemm(0, n, n, n, U, n, T, n, R, ldr, info));
  } else {
    RZ_TRY(gemm(0, n, n, n, T, n, G, n, R, ldr, info));
  }
  return pamd_trsv_packed_f64(1, n, ws + L.tri, z, stream);
}
