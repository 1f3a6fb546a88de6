// Thin SVD of a small dense matrix by one-sided block Jacobi (Hestenes'
// method), and the two helpers of the symmetric eigendecomposition built on
// it (the eigenvalues of a symmetric C are the singular values of C with the
// signs of u_j . v_j).
//
// Replaces the small LAPACK decompositions of the low-rank drivers: la.svd(B)
// of SVD1 (drivers/svd.py:164), la.eigh(C) of EVD1 (drivers/evd.py:279), the
// SVD preconditioner (comps/preconditioning.py:74) and the SVD-based solve of
// sketch-and-solve (drivers/least_squares.py:186).
//
// The callers precondition as Drmac and Veselic do: the Jacobi runs on R^T of
// a Householder QR, whose columns are far closer to orthogonal than A's (9
// sweeps instead of 27 for a 266 x 266 matrix with Haar singular vectors).
//
// Method.  The columns of W (m x n, m >= n, initially A) are rotated pairwise
// until every pair is orthogonal to tol = m * eps relative to the pair's
// norms; the rotations accumulate in V.  Then A = W V^T, the column norms of W
// are the singular values and its normalised columns the left singular
// vectors.  The Gram matrix of a pair of blocks is formed from the columns in
// every round and rotated with them inside it; its relative accuracy is that of
// the columns scaled to unit length (Demmel and Veselic 1992), so small singular
// values of graded matrices keep theirs, unlike with one Gram matrix of A.
//
// Parallel order.  The n columns (padded with zero columns) form nb blocks
// of w columns, nb even.  A sweep is nb - 1 rounds of the round-robin
// ("circle") tournament over the blocks: in a round every block meets one
// other block, and each block pair is one workgroup, which runs one full inner
// sweep over its 2w columns (2w - 1 steps of w disjoint column pairs) on their
// Gram matrix and applies the accumulated rotation to W and V (see the kernel).
//
// Convergence without host synchronisation.  A workgroup that rotated any
// pair increments the sweep's counter.  Every round kernel of sweep s > 0
// returns at once when sweep s - 1 rotated nothing, so the host can enqueue
// max_sweeps sweeps without reading anything back.
//
// Layout in the workspace: W as np columns of m doubles (column j at
// W + j*m), V as np columns of np doubles, then the column norms, the sorted
// positions and the per-sweep counters.  w = 8: narrow blocks spread a sweep
// over more workgroups at once (17 per round at n = 266).
#include <mutex>
#include <type_traits>

#include "common.h"

typedef double d4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int JAC_BW = 8;                 // columns per block: 16 per pair, one wavefront per column pair
constexpr int JAC_P = 2 * JAC_BW;         // columns of a pair
constexpr int JAC_THREADS = 512;          // one round workgroup
constexpr int JAC_MAX_SWEEPS = 64;
constexpr int64_t JAC_MAX_M = 1024;

__host__ __device__ inline int jac_block(int64_t) { return JAC_BW; }

__host__ __device__ inline int64_t jac_nblocks(int64_t n, int w) {
  int64_t nb = pamd_cdiv(n, w);
  nb += nb & 1;
  return nb < 2 ? 2 : nb;
}

struct JacLayout {
  int64_t W, V, sig, pos, cnt, total;  // offsets in doubles
};

__host__ __device__ inline JacLayout jac_layout(int64_t m, int64_t n) {
  const int w = jac_block(m);
  const int64_t np = jac_nblocks(n, w) * w;
  JacLayout L;
  L.W = 0;
  L.V = L.W + np * m;
  L.sig = L.V + np * np;
  L.pos = L.sig + np;                   // np int32 (np / 2 doubles, rounded up)
  L.cnt = L.pos + (np + 1) / 2 + 1;     // JAC_MAX_SWEEPS int32
  L.total = L.cnt + JAC_MAX_SWEEPS / 2 + 8;
  return L;
}

// the pair of participant k in round r of the circle tournament over L + 1
// players (L odd): player L sits still, the others rotate
__device__ __forceinline__ void circle_pair(int r, int k, int L, int& a, int& b) {
  if (k == 0) {
    a = L;
    b = r;
  } else {
    a = (r + k) % L;
    b = (r - k + L) % L;
  }
}

// W (column-major, ld m) <- A (row-major, lda) padded with zero columns to np;
// V <- I (np x np); sweep counters <- 0
__global__ void jac_init_kernel(int64_t m, int64_t n, int64_t np, const double* __restrict__ A, int64_t lda,
                                double* __restrict__ ws) {
  const JacLayout L = jac_layout(m, n);
  double* W = ws + L.W;
  double* V = ws + L.V;
  int* cnt = reinterpret_cast<int*>(ws + L.cnt);
  const int64_t j = blockIdx.y;  // column
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x) {
    W[j * m + i] = (j < n) ? A[i * lda + j] : 0.0;
  }
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < np; i += (int64_t)gridDim.x * blockDim.x)
    V[j * np + i] = (i == j) ? 1.0 : 0.0;
  if (j == 0 && blockIdx.x == 0 && threadIdx.x < JAC_MAX_SWEEPS) cnt[threadIdx.x] = 0;
}

// 1 / sqrt(x): hardware estimate (relative error about 2^-26) and one third-
// order correction
__device__ __forceinline__ double rsq_nr(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// c, s and t = s / c of the rotation a' = c a - s b, b' = s a + c b that makes
// a'.b' = 0, from al = a.a, be = b.b, ga = a.b; |theta| <= pi / 4.  With d = be -
// al, g = 2 ga, h = sqrt(d^2 + g^2): cos 2 theta = |d| / h, so c^2 = (1 + |d| / h)
// / 2 and s = sign(d) g / (2 h c): two reciprocal square roots in a row and no
// division (the step is a chain of latencies).  The identity unless rot.  h2 =
// d^2 + g^2 (d and g may share any factor).
__device__ __forceinline__ void jac_rotation(bool rot, double d, double g, double h2, double& c, double& s,
                                             double& t) {
  const double r = rsq_nr(h2);                // 1 / h
  const double c2 = fma(0.5 * fabs(d), r, 0.5);
  const double w = rsq_nr(c2);                // 1 / c
  const double ss = copysign(0.5 * g, d < 0.0 ? -g : g) * r * w;
  c = rot ? c2 * w : 1.0;
  s = rot ? ss : 0.0;
  t = rot ? ss * w : 0.0;
}

// Squared lengths whose products and squares (h^2 is of fourth order in the
// lengths) keep to FP64's range, down to what cancels in a round; 0 is a zero
// column.  Outside, h^2 loses its last bits or overflows, and c, s would not be
// a rotation.
__device__ __forceinline__ bool jac_in_range(double al) { return !(al > 0x1p480 || (al > 0.0 && al < 0x1p-400)); }

// The slow path for a round with columns outside that (1e-60 .. 1e72 in
// length): whether the pair is to be rotated, with al, be and ga scaled by a
// power of two where their products overflow, and d, g by the one that makes
// the larger of them about 1, with their h^2.  Where the products underflow the
// test stays as it is: a pair whose ga^2 is 0 is left alone, which ends the
// sweeps on the columns of a rank-one triangle (1e-16, 1e-32, .. in length) that
// cannot be made orthogonal to a relative tolerance among subnormal numbers.
__device__ __forceinline__ bool jac_wide(double al, double be, double ga, double tol2, double& d, double& g,
                                         double& h2) {
  d = be - al;
  g = 2.0 * ga;
  int e = al * be < 0x1p1000 ? 0 : -__builtin_amdgcn_frexp_exp(fmax(al, be));
  const double c = ldexp(ga, e);
  const bool rot = c * c > tol2 * (ldexp(al, e) * ldexp(be, e));
  e = -__builtin_amdgcn_frexp_exp(fmax(fabs(d), fabs(g)));
  d = ldexp(d, e);
  g = ldexp(g, e);
  h2 = fma(d, d, g * g);
  return rot;
}

// One round of sweep `sweep`: workgroup k orthogonalises block pair k (P = 16
// columns, rows in chunks of 16; CH >= ceil(max(m, np) / 128) chunks per
// wavefront).  What bounds it is the chain of 15 steps; so a step works on the
// pair's Gram matrix G = W^T W (one MFMA product per round) instead of the
// columns.  One wavefront holds G's 8 x 8 grid of (pair p, pair q) 2 x 2 blocks
// in its 64 lanes: a lane reads its block and both pairs' three inner products
// from LDS, forms both rotations and writes the rotated block, so the step has
// no barrier and no exchange of rotations: 1000 cycles, most of them the issue of
// one wavefront's 75 FP64 operations (reducing the inner products of the columns
// themselves took 2500).  The accumulated rotation J is
// then applied to the pair's columns of W and V by MFMA from registers that
// were loaded before the steps.  G is formed afresh in every round, so what is
// rotated and when the sweeps end is decided by the columns' own inner products.
// A working round at m = n = 160 takes 12 us, 6.5 of them the steps; the SVD of
// a 160 x 160 / 266 x 266 / 1000 x 1000 triangle 2.53 -> 1.45 / 5.6 -> 3.0 / 52 -> 28
// ms.
template <int CH>
__global__ __launch_bounds__(JAC_THREADS) void jac_round_kernel(int m, int nb, int sweep, int round, double tol,
                                                                double* __restrict__ W, double* __restrict__ V,
                                                                int* __restrict__ cnt) {
  constexpr int NW = JAC_THREADS / 64;
  __shared__ double part[NW][JAC_P * JAC_P];
  __shared__ double G[JAC_P][JAC_P + 8];   // the stride keeps a step's 64 accesses (nearly) off each other's banks
  __shared__ double Jm[JAC_P][JAC_P + 8];  // Jm[k][j]: column j of the result takes Jm[k][j] of column k
  __shared__ int any;
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int np = nb * JAC_BW;
  if (sweep > 0 && cnt[sweep - 1] == 0) return;  // an earlier sweep rotated nothing: converged
  int bp, bq;
  circle_pair(round, blockIdx.x, nb - 1, bp, bq);
  // global column of pair column c
  auto gcol = [&](int c) -> int64_t { return (c < JAC_BW) ? bp * JAC_BW + c : bq * JAC_BW + (c - JAC_BW); };

  // Gram operand: column lr, rows 16 Q + 4 lk + r; product operand: column 4 q + lk,
  // row 16 Q + lr.  Rows past the end are read from the last one and zeroed:
  // a branch per load made the 24 loads take 4000 cycles to issue.
  const double* wcol = W + gcol(lr) * m;
  const double *wprod[4], *vprod[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    wprod[q] = W + gcol(4 * q + lk) * m;
    vprod[q] = V + gcol(4 * q + lk) * np;
  }
  double wg[CH][4], wa[CH][4], va[CH][4];
#pragma unroll
  for (int u = 0; u < CH; ++u) {
    const int r0 = 16 * (wave + NW * u);
    const int ra = r0 + lr, rm = min(ra, m - 1), rv = min(ra, np - 1);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      wg[u][q] = wcol[min(r0 + 4 * lk + q, m - 1)];
      wa[u][q] = wprod[q][rm];
      va[u][q] = vprod[q][rv];
    }
  }
#pragma unroll
  for (int u = 0; u < CH; ++u)
#pragma unroll
    for (int q = 0; q < 4; ++q) wg[u][q] = (16 * (wave + NW * u) + 4 * lk + q < m) ? wg[u][q] : 0.0;
  d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int u = 0; u < CH; ++u)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(wg[u][q], wg[u][q], acc, 0, 0, 0);
#pragma unroll
  for (int r = 0; r < 4; ++r) part[wave][(lk + 4 * r) * JAC_P + lr] = acc[r];
  __syncthreads();
  if (threadIdx.x < JAC_P * JAC_P) {
    const int i = threadIdx.x / JAC_P, j = threadIdx.x % JAC_P;
    double g = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) g += part[w][threadIdx.x];
    G[i][j] = g;
    Jm[i][j] = i == j ? 1.0 : 0.0;
  }
  __syncthreads();
  if (wave == 0) {
    // pair p of step t is (15, t) for p = 0, else (t + p, t - p) modulo 15: rows
    // a, b by p = lane / 8 and columns e, f by q = lane % 8, stepped by one
    const int p = lane >> 3, q = lane & 7;
    int a = p ? p : JAC_P - 1, b = p ? JAC_P - 1 - p : 0;
    int e = q ? q : JAC_P - 1, f = q ? JAC_P - 1 - q : 0;
    const double tol2 = tol * tol;
    bool rotated = false;
    const bool wide = __any(!jac_in_range(G[lr][lr]));
    double* J0 = &Jm[2 * p][0];
    double* J1 = &Jm[2 * p + 1][0];
    auto steps = [&](auto WIDE) {
      for (int t = 0; t < JAC_P - 1; ++t) {
        double *Ga = &G[a][0], *Gb = &G[b][0];
        const double alq = G[e][e], beq = G[f][f], gaq = G[e][f];
        const double alp = Ga[a], bep = Gb[b], gap = Ga[b];
        const double gae = Ga[e], gaf = Ga[f], gbe = Gb[e], gbf = Gb[f];
        const double j0e = J0[e], j0f = J0[f], j1e = J1[e], j1f = J1[f];
        __builtin_amdgcn_sched_barrier(0);  // every read under way before the first is waited for
        double dp, gp, hp, dq, gq, hq;
        bool rp, rq;
        if constexpr (WIDE.value) {
          rp = jac_wide(alp, bep, gap, tol2, dp, gp, hp);
          rq = jac_wide(alq, beq, gaq, tol2, dq, gq, hq);
        } else {
          rq = gaq * gaq > tol2 * (alq * beq);
        }
        if (__any(rq)) {
          double cp, sp, tp, cq, sq, tq;
          if constexpr (!WIDE.value) {
            rp = gap * gap > tol2 * (alp * bep);
            dp = bep - alp, gp = 2.0 * gap, hp = fma(dp, dp, gp * gp);
            dq = beq - alq, gq = 2.0 * gaq, hq = fma(dq, dq, gq * gq);
          }
          jac_rotation(rp, dp, gp, hp, cp, sp, tp);
          jac_rotation(rq, dq, gq, hq, cq, sq, tq);
          rotated = true;
          // rows (a, b) by p's rotation, then columns (e, f) by q's
          const double rae = cp * gae - sp * gbe, raf = cp * gaf - sp * gbf;
          const double rbe = sp * gae + cp * gbe, rbf = sp * gaf + cp * gbf;
          double nae = cq * rae - sq * raf, naf = sq * rae + cq * raf;
          double nbe = cq * rbe - sq * rbf, nbf = sq * rbe + cq * rbf;
          if (p == q && tp != 0.0) {  // the pair's own block: al - t ga, be + t ga, orthogonal
            nae = fma(-tp, gap, alp);
            nbf = fma(tp, gap, bep);
            naf = nbe = 0.0;
          }
          PAMD_WAVE_SYNC();
          Ga[e] = nae;
          Ga[f] = naf;
          Gb[e] = nbe;
          Gb[f] = nbf;
          J0[e] = cq * j0e - sq * j0f;
          J0[f] = sq * j0e + cq * j0f;
          J1[e] = cq * j1e - sq * j1f;
          J1[f] = sq * j1e + cq * j1f;
          PAMD_WAVE_SYNC();
        }
        a = p ? (a == JAC_P - 2 ? 0 : a + 1) : a;
        b = b == JAC_P - 2 ? 0 : b + 1;
        e = q ? (e == JAC_P - 2 ? 0 : e + 1) : e;
        f = f == JAC_P - 2 ? 0 : f + 1;
      }
    };
    if (wide)
      steps(std::true_type{});
    else
      steps(std::false_type{});
    const bool r = __any(rotated);
    if (lane == 0) any = r;
  }
  __syncthreads();
  if (!any) return;  // the pair was already orthogonal: W and V unchanged
  double jb[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) jb[q] = Jm[4 * q + lk][lr];
#pragma unroll
  for (int u = 0; u < CH; ++u) {
    const int r0 = 16 * (wave + NW * u);
    d4 w = {0.0, 0.0, 0.0, 0.0}, v = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      w = __builtin_amdgcn_mfma_f64_16x16x4f64(wa[u][q], jb[q], w, 0, 0, 0);
      v = __builtin_amdgcn_mfma_f64_16x16x4f64(va[u][q], jb[q], v, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = r0 + lk + 4 * r;
      if (row < m) W[gcol(lr) * m + row] = w[r];
      if (row < np) V[gcol(lr) * np + row] = v[r];
    }
  }
  if (threadIdx.x == 0) atomicAdd(cnt + sweep, 1);
}

// sigma_j = ||W(:, j)|| for the first n columns, one workgroup per column
__global__ __launch_bounds__(256) void jac_norms_kernel(int64_t m, int64_t n, double* __restrict__ ws) {
  __shared__ double red[4];
  const JacLayout L = jac_layout(m, n);
  const double* W = ws + L.W;
  const int64_t j = blockIdx.x;
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < m; i += blockDim.x) {
    const double v = W[j * m + i];
    acc = fma(v, v, acc);
  }
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) ws[L.sig + j] = sqrt(red[0] + red[1] + red[2] + red[3]);
}

// position of column j in descending order of sigma (ties: lower index first),
// the sorted sigma, the convergence flag
__global__ __launch_bounds__(JAC_THREADS) void jac_sort_kernel(int64_t m, int64_t n, int max_sweeps,
                                                               double* __restrict__ s, double* __restrict__ ws,
                                                               int* __restrict__ info) {
  const JacLayout L = jac_layout(m, n);
  const double* sig = ws + L.sig;
  int* pos = reinterpret_cast<int*>(ws + L.pos);
  const int* cnt = reinterpret_cast<const int*>(ws + L.cnt);
  for (int64_t j = threadIdx.x; j < n; j += blockDim.x) {
    const double sj = sig[j];
    int p = 0;
    for (int64_t k = 0; k < n; ++k) {
      const double sk = sig[k];
      p += (sk > sj || (sk == sj && k < j)) ? 1 : 0;
    }
    pos[j] = p;
    s[p] = sj;
  }
  if (threadIdx.x == 0 && info) info[0] = (cnt[max_sweeps - 1] != 0) ? 1 : 0;
}

// U(:, pos_j) = W(:, j) / sigma_j (0 for sigma_j = 0); Vt(pos_j, :) = V(:, j)^T
__global__ void jac_output_kernel(int64_t m, int64_t n, int64_t np, double* __restrict__ U, int64_t ldu,
                                  double* __restrict__ Vt, int64_t ldvt, const double* __restrict__ ws) {
  const JacLayout L = jac_layout(m, n);
  const double* W = ws + L.W;
  const double* V = ws + L.V;
  const int* pos = reinterpret_cast<const int*>(ws + L.pos);
  const int64_t j = blockIdx.y;
  const int64_t p = pos[j];
  const double sj = ws[L.sig + j];
  const double inv = (sj > 0.0) ? 1.0 / sj : 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x) {
    if (U) U[i * ldu + p] = W[j * m + i] * inv;
  }
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    if (Vt) Vt[p * ldvt + i] = V[j * np + i];
  }
}

// eigenvalues of the symmetric matrix from its singular triplets: lambda_j =
// sigma_j sign(u_j . v_j) - shift; info[0] = 2 when, for a singular value
// above 1e-10 sigma_max, |u_j . v_j| falls short of 1 by more than 1e-6 (a
// pair lambda, -lambda of nearly equal magnitude mixed the vectors; below
// that size the sign of a null-space value is noise, as it is for eigh)
__global__ __launch_bounds__(256) void jac_eig_sign_kernel(int64_t n, const double* __restrict__ U, int64_t ldu,
                                                           const double* __restrict__ Vt, int64_t ldvt,
                                                           const double* __restrict__ s, double shift,
                                                           double* __restrict__ lamb, int* __restrict__ info) {
  __shared__ double red[4];
  const int64_t j = blockIdx.x;
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) acc = fma(U[i * ldu + j], Vt[j * ldvt + i], acc);
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    const double d = red[0] + red[1] + red[2] + red[3];
    const double sj = s[j];
    lamb[j] = (d < 0.0 ? -sj : sj) - shift;
    if (sj > 1e-10 * s[0] && fabs(fabs(d) - 1.0) > 1e-6 && info) atomicMax(info, 2);
  }
}

int jac_launch_sweeps(int64_t m, int64_t n, int max_sweeps, double* ws, hipStream_t st) {
  const int w = jac_block(m);
  const int nb = (int)jac_nblocks(n, w);
  const double tol = (double)imax64(m, 16) * 2.220446049250313e-16;
  const JacLayout L = jac_layout(m, n);
  double *W = ws + L.W, *V = ws + L.V;
  int* cnt = reinterpret_cast<int*>(ws + L.cnt);
  const int64_t rows = imax64(m, (int64_t)nb * w);
  for (int sw = 0; sw < max_sweeps; ++sw) {
    for (int r = 0; r < nb - 1; ++r) {
#define PAMD_JAC(CH) jac_round_kernel<CH><<<nb / 2, JAC_THREADS, 0, st>>>((int)m, nb, sw, r, tol, W, V, cnt)
      if (rows <= 128) PAMD_JAC(1);
      else if (rows <= 256) PAMD_JAC(2);
      else if (rows <= 384) PAMD_JAC(3);
      else if (rows <= 640) PAMD_JAC(5);
      else PAMD_JAC(8);
#undef PAMD_JAC
      PAMD_LAUNCH_CHECK();
    }
  }
  return PAMD_OK;
}

int jac_finish(int64_t m, int64_t n, int max_sweeps, double* U, int64_t ldu, double* s, double* Vt, int64_t ldvt,
               double* ws, int* info, hipStream_t st) {
  const int w = jac_block(m);
  const int64_t np = jac_nblocks(n, w) * w;
  jac_norms_kernel<<<(unsigned)n, 256, 0, st>>>(m, n, ws);
  PAMD_LAUNCH_CHECK();
  jac_sort_kernel<<<1, JAC_THREADS, 0, st>>>(m, n, max_sweeps, s, ws, info);
  PAMD_LAUNCH_CHECK();
  dim3 grid((unsigned)imin64(pamd_cdiv(imax64(m, n), 256), 4), (unsigned)n);
  jac_output_kernel<<<grid, 256, 0, st>>>(m, n, np, U, ldu, Vt, ldvt, ws);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

}  // namespace

extern "C" int pamd_svd_jacobi_workspace(int64_t m, int64_t n, int64_t* bytes) {
  PAMD_ARG_CHECK(m >= 1 && m <= JAC_MAX_M, 1);
  PAMD_ARG_CHECK(n >= 1 && n <= m, 2);
  PAMD_ARG_CHECK(bytes != nullptr, 3);
  *bytes = jac_layout(m, n).total * (int64_t)sizeof(double);
  return PAMD_OK;
}

namespace {

// the whole SVD on a caller-supplied or static workspace ws (arguments checked)
int jac_svd(int64_t m, int64_t n, const double* A, int64_t lda, double* U, int64_t ldu, double* s, double* Vt,
            int64_t ldvt, int max_sweeps, double* ws, int* info, hipStream_t st) {
  const int w = jac_block(m);
  const int64_t np = jac_nblocks(n, w) * w;
  dim3 grid((unsigned)imin64(pamd_cdiv(imax64(m, np), 256), 4), (unsigned)np);
  jac_init_kernel<<<grid, 256, 0, st>>>(m, n, np, A, lda, ws);
  PAMD_LAUNCH_CHECK();
  const int rc = jac_launch_sweeps(m, n, max_sweeps, ws, st);
  if (rc != PAMD_OK) return rc;
  return jac_finish(m, n, max_sweeps, U, ldu, s, Vt, ldvt, ws, info, st);
}

}  // namespace

// ---------------------------------------------------------------------------
// The allocation-free variant: the same kernels on a file-scope device array
// of JAC_SCRATCH_DOUBLES doubles (16.8 MB, the workspace of the largest SVD
// this file does, m = n = 1024).  Each GPU holds its own copy of the array
// until the process ends; its device address is looked up once per device
// (hipGetSymbolAddress with that device current) and used for every launch --
// the array's name is only a host-side stand-in.  Every call on one GPU
// shares that GPU's array: calls that overlap on one GPU race.  Nothing in it
// needs clearing between calls: the init kernel writes W, V and the sweep
// counters, and the norms and positions are written before they are read.
// ---------------------------------------------------------------------------
constexpr int64_t JAC_SCRATCH_DOUBLES = 2 * JAC_MAX_M * JAC_MAX_M + 4 * JAC_MAX_M + 256;
static __device__ __align__(256) double scratch[JAC_SCRATCH_DOUBLES];

namespace {

constexpr int JAC_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[JAC_MAX_DEVICES] = {};

// device address of the current device's copy of `scratch`
int jac_scratch(double** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= JAC_MAX_DEVICES) return PAMD_ERR_HIP;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) return PAMD_ERR_HIP;
    g_scratch_ptr[dev] = static_cast<double*>(p);
  }
  *out = g_scratch_ptr[dev];
  return PAMD_OK;
}

}  // namespace

extern "C" int pamd_svd_jacobi_noalloc_f64(int64_t m, int64_t n, const double* A, int64_t lda, double* U,
                                           int64_t ldu, double* s, double* Vt, int64_t ldvt, int max_sweeps,
                                           int* info, void* stream) {
  PAMD_ARG_CHECK(m >= 1 && m <= JAC_MAX_M, 1);
  PAMD_ARG_CHECK(n >= 1 && n <= m, 2);
  PAMD_ARG_CHECK(A != nullptr, 3);
  PAMD_ARG_CHECK(lda >= n, 4);
  PAMD_ARG_CHECK(U == nullptr || ldu >= n, 6);
  PAMD_ARG_CHECK(s != nullptr, 7);
  PAMD_ARG_CHECK(Vt == nullptr || ldvt >= n, 9);
  PAMD_ARG_CHECK(max_sweeps >= 1 && max_sweeps <= JAC_MAX_SWEEPS, 10);
  if (jac_layout(m, n).total > JAC_SCRATCH_DOUBLES) return PAMD_ERR_UNSUPPORTED;
  double* ws = nullptr;
  const int rc = jac_scratch(&ws);
  if (rc != PAMD_OK) return rc;
  return jac_svd(m, n, A, lda, U, ldu, s, Vt, ldvt, max_sweeps, ws, info, (hipStream_t)stream);
}

extern "C" int pamd_svd_jacobi_f64(int64_t m, int64_t n, const double* A, int64_t lda, double* U, int64_t ldu,
                                   double* s, double* Vt, int64_t ldvt, int max_sweeps, void* workspace, int* info,
                                   void* stream) {
  PAMD_ARG_CHECK(m >= 1 && m <= JAC_MAX_M, 1);
  PAMD_ARG_CHECK(n >= 1 && n <= m, 2);
  PAMD_ARG_CHECK(A != nullptr, 3);
  PAMD_ARG_CHECK(lda >= n, 4);
  PAMD_ARG_CHECK(U == nullptr || ldu >= n, 6);
  PAMD_ARG_CHECK(s != nullptr, 7);
  PAMD_ARG_CHECK(Vt == nullptr || ldvt >= n, 9);
  PAMD_ARG_CHECK(max_sweeps >= 1 && max_sweeps <= JAC_MAX_SWEEPS, 10);
  PAMD_ARG_CHECK(workspace != nullptr, 11);
  return jac_svd(m, n, A, lda, U, ldu, s, Vt, ldvt, max_sweeps, (double*)workspace, info, (hipStream_t)stream);
}

namespace {

// out = the lower triangle of A mirrored, plus shift * I (n x n)
__global__ void sym_shift_kernel(int64_t n, const double* __restrict__ A, int64_t lda, double shift,
                                 double* __restrict__ out, int64_t ldo) {
  const int64_t i = blockIdx.y;
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x) {
    double a = (i >= j) ? A[i * lda + j] : A[j * lda + i];
    if (i == j) a += shift;
    out[i * ldo + j] = a;
  }
}

}  // namespace

extern "C" int pamd_sym_shift_f64(int64_t n, const double* A, int64_t lda, double shift, double* out,
                                  int64_t ldo, void* stream) {
  PAMD_ARG_CHECK(n >= 0 && n < (int64_t)1 << 31, 1);
  PAMD_ARG_CHECK(A != nullptr || n == 0, 2);
  PAMD_ARG_CHECK(lda >= n && lda >= 1, 3);
  PAMD_ARG_CHECK(out != nullptr || n == 0, 5);
  PAMD_ARG_CHECK(ldo >= n && ldo >= 1, 6);
  if (n == 0) return PAMD_OK;
  dim3 grid((unsigned)imin64(pamd_cdiv(n, 256), 16), (unsigned)n);
  sym_shift_kernel<<<grid, 256, 0, (hipStream_t)stream>>>(n, A, lda, shift, out, ldo);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

extern "C" int pamd_eig_from_svd_f64(int64_t n, const double* U, int64_t ldu, const double* Vt, int64_t ldvt,
                                     const double* s, double shift, double* lamb, int* info, void* stream) {
  PAMD_ARG_CHECK(n >= 0 && n < (int64_t)1 << 31, 1);
  PAMD_ARG_CHECK(U != nullptr || n == 0, 2);
  PAMD_ARG_CHECK(ldu >= n && ldu >= 1, 3);
  PAMD_ARG_CHECK(Vt != nullptr || n == 0, 4);
  PAMD_ARG_CHECK(ldvt >= n && ldvt >= 1, 5);
  PAMD_ARG_CHECK(s != nullptr || n == 0, 6);
  PAMD_ARG_CHECK(lamb != nullptr || n == 0, 8);
  PAMD_ARG_CHECK(lamb != s || n == 0, 8);
  if (n == 0) return PAMD_OK;
  jac_eig_sign_kernel<<<(unsigned)n, 256, 0, (hipStream_t)stream>>>(n, U, ldu, Vt, ldvt, s, shift, lamb, info);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}
