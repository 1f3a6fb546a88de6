// Cholesky factorisation and right triangular solve for CholeskyQR.
//
// CholeskyQR2 orthonormalises a tall-skinny Y (m x k) with two rounds of
//   G = Y^T Y (MFMA GEMM),  G = R^T R (potrf),  Y <- Y R^{-1} (trsm_right),
// so the O(m k^2) work is GEMM-shaped and the only sequential parts act on
// the k x k Gram matrix.  It replaces the Householder QR inside the power
// iteration stabilizer (utils/linalg_wrappers.py:6-7) where Y is well enough
// conditioned (the caller falls back to Householder when potrf fails).
//
// potrf: one 512-thread workgroup with the triangle in registers
//   (potrf_reg.h), beyond 208 rows 128 of them at a time with chip-wide steps
//   between.  trtri: R^{-1} one column per workgroup, so that Y R^{-1} is a
//   plain MFMA GEMM.  trsm_right: the in-place alternative for callers that
//   cannot afford the k x k inverse; one workgroup per tile of rows, staged in
//   LDS, 16 lanes of one wavefront per row.
#include <utility>

#include "common.h"
#include "potrf_reg.h"
#include "trsm_dev.h"
#include "trsv_dev.h"

namespace {

constexpr int POTRF_MAX_N = 512;

__global__ void potrf_zero_info_kernel(int* info) { info[0] = 0; }

// The rows from j0 on that this step factors (pr_width).  info is written at
// j0 = 0; later steps leave a failure alone and report theirs offset by j0.
template <int SL>
__global__ __launch_bounds__(PR_THREADS) void potrf_reg_kernel(int n, int j0, double* __restrict__ A, int64_t lda,
                                                               int* __restrict__ info) {
  if (j0 && info[0]) return;
  potrf_reg<SL>(pr_width(n, j0), A + j0 * (lda + 1), lda, info, j0);
}

// n: rows of the matrix whose PR_LEAD leading ones (at A) are factored
__global__ __launch_bounds__(256) void potrf_row_kernel(int n, double* __restrict__ A, int64_t lda,
                                                        const int* __restrict__ info) {
  if (info[0]) return;
  pr_block_column(n, A, lda, PR_LEAD + PR_B * (int)blockIdx.x);
}

__global__ __launch_bounds__(64) void potrf_trailing_kernel(int n, double* __restrict__ A, int64_t lda,
                                                            const int* __restrict__ info) {
  if (info[0]) return;
  pr_trailing_tile(n, A, lda, (int)blockIdx.x);
}

// Batched: problem i = the n[i] x n[i] matrix at pool + off[i] (ld n[i]).  The
// same steps over all problems; workgroups leave where their problem has no
// such step.
template <int SL>
__global__ __launch_bounds__(PR_THREADS) void potrf_batched_kernel(const int64_t* __restrict__ nv,
                                                                   const int64_t* __restrict__ off, int j0,
                                                                   double* __restrict__ pool,
                                                                   int* __restrict__ info) {
  const int n = (int)nv[blockIdx.x];
  int* inf = info + blockIdx.x;
  const int w = pr_width(n, j0);
  if (w <= 0) {
    if (j0 == 0 && SL == PR_SMALL && threadIdx.x == 0) inf[0] = 0;
    return;
  }
  if (pr_small(w) != (SL == PR_SMALL) || (j0 && inf[0])) return;
  potrf_reg<SL>(w, pool + off[blockIdx.x] + j0 * ((int64_t)n + 1), n, inf, j0);
}

__global__ __launch_bounds__(256) void potrf_batched_row_kernel(const int64_t* __restrict__ nv,
                                                                const int64_t* __restrict__ off, int j0,
                                                                double* __restrict__ pool,
                                                                const int* __restrict__ info) {
  const int n = (int)nv[blockIdx.y], c0 = PR_LEAD + PR_B * (int)blockIdx.x;
  if (n - j0 <= PR_MAXN || c0 >= n - j0 || info[blockIdx.y]) return;
  pr_block_column(n - j0, pool + off[blockIdx.y] + j0 * ((int64_t)n + 1), n, c0);
}

__global__ __launch_bounds__(64) void potrf_batched_trailing_kernel(const int64_t* __restrict__ nv,
                                                                    const int64_t* __restrict__ off, int j0,
                                                                    double* __restrict__ pool,
                                                                    const int* __restrict__ info) {
  const int n = (int)nv[blockIdx.y];
  if (n - j0 <= PR_MAXN || info[blockIdx.y]) return;
  const int T = pr_trailing(n - j0);
  if ((int)blockIdx.x >= T * (T + 1) / 2) return;
  pr_trailing_tile(n - j0, pool + off[blockIdx.y] + j0 * ((int64_t)n + 1), n, (int)blockIdx.x);
}

// Rinv = R^{-1} (upper; zeros below): workgroup j solves R x = e_j on rows 0..j.
__global__ __launch_bounds__(256) void trtri_kernel(int64_t n, const double* __restrict__ R, int64_t ldr,
                                                    double* __restrict__ Ri, int64_t ldi) {
  extern __shared__ double smem[];
  const int64_t j = blockIdx.x;
  const int sz = (int)j + 1;
  double* xs = smem;
  for (int i = threadIdx.x; i < sz; i += blockDim.x) xs[i] = (i == sz - 1) ? 1.0 : 0.0;
  __syncthreads();
  trsv_upper_block<8>(0, sz, R, ldr, xs, smem + sz);
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) Ri[i * ldi + j] = (i <= j) ? xs[i] : 0.0;
}

// batched R^{-1}: grid (max n, problems); column j of problem i when j < n[i]
__global__ __launch_bounds__(256) void trtri_batched_kernel(const int64_t* __restrict__ nv,
                                                            const int64_t* __restrict__ off,
                                                            const double* __restrict__ Rp, double* __restrict__ Rip,
                                                            double* __restrict__ RiTp) {
  extern __shared__ double smem[];
  const int64_t n = nv[blockIdx.y];
  const int64_t j = blockIdx.x;
  if (j >= n) return;
  const double* R = Rp + off[blockIdx.y];
  double* Ri = Rip + off[blockIdx.y];
  const int sz = (int)j + 1;
  double* xs = smem;
  for (int i = threadIdx.x; i < sz; i += blockDim.x) xs[i] = (i == sz - 1) ? 1.0 : 0.0;
  __syncthreads();
  trsv_upper_block<8>(0, sz, R, n, xs, smem + sz);
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) Ri[i * n + j] = (i <= j) ? xs[i] : 0.0;
  if (RiTp != nullptr) {  // row j of the transpose: contiguous
    double* RiT = RiTp + off[blockIdx.y];
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) RiT[j * n + i] = (i <= j) ? xs[i] : 0.0;
  }
}

__global__ __launch_bounds__(64) void trsm_dinv_kernel(int k, const double* __restrict__ R, int64_t ldr,
                                                       double* __restrict__ Dinv) {
  trsm_dinv_body(blockIdx.x, k, R, ldr, Dinv);
}

__global__ __launch_bounds__(256) void trsm_strip_kernel(int64_t m, int k, const double* __restrict__ Y, int64_t ldy,
                                                         const double* __restrict__ R, int64_t ldr,
                                                         const double* __restrict__ Dinv, double* __restrict__ X,
                                                         int64_t ldx, const int* __restrict__ skip) {
  if (skip != nullptr && *skip != 0) return;
  trsm_strip_body(blockIdx.x, m, k, Y, ldy, R, ldr, Dinv, X, ldx);
}

// rows of B per workgroup: 16 lanes per row, tile of rows x n doubles <= 64 KiB
inline int trsm_rows(int64_t n) {
  int64_t r = 65536 / (8 * imax64(n, 1));
  r = imin64(64, r) / 4 * 4;
  return (int)imax64(4, r);
}

// B (m x n) <- B R^{-1}, R upper n x n.  LDS holds the `rows`-row tile of B.
__global__ __launch_bounds__(1024) void trsm_right_kernel(int64_t m, int64_t n, int rows,
                                                          const double* __restrict__ R, int64_t ldr,
                                                          double* __restrict__ B, int64_t ldb) {
  extern __shared__ double T[];  // rows x n
  const int64_t r0 = (int64_t)blockIdx.x * rows;
  const int nr = (int)imin64(rows, m - r0);
  for (int64_t e = threadIdx.x; e < (int64_t)rows * n; e += blockDim.x) {
    const int64_t rr = e / n, c = e % n;
    T[e] = (rr < nr) ? B[(r0 + rr) * ldb + c] : 0.0;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int sub = lane >> 4, q = lane & 15;  // 4 rows per wave, 16 lanes per row
  const int rr = wave * 4 + sub;
  double* row = T + (int64_t)rr * n;
  for (int64_t c = 0; c < n; ++c) {
    double s = 0.0;
    for (int64_t l = q; l < c; l += 16) s += row[l] * R[l * ldr + c];
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    s += __shfl_xor(s, 4, 64);
    s += __shfl_xor(s, 8, 64);
    const double v = (row[c] - s) / R[c * ldr + c];
    PAMD_WAVE_SYNC();
    if (q == 0) row[c] = v;
    PAMD_WAVE_SYNC();
  }
  __syncthreads();
  for (int64_t e = threadIdx.x; e < (int64_t)nr * n; e += blockDim.x) {
    const int64_t r = e / n, c = e % n;
    B[(r0 + r) * ldb + c] = T[r * n + c];
  }
}

// ---------------------------------------------------------------------------
// Small k x k helpers of CholeskyQR2, one workgroup each (k <= 512):
//   combine: out = A + alpha B + sigma I, or H(A + alpha B + sigma I) where H
//            keeps the upper triangle and halves the diagonal; optionally
//            ||A + alpha B + sigma I||_F (rows summed in order by each thread,
//            then the waves in order);
//   stats:   min |G_ii|, max |G_ii|, the norm above and the potrf info, packed
//            into four doubles for one read-back.
// ---------------------------------------------------------------------------
constexpr int SC_THREADS = 1024;

__global__ __launch_bounds__(SC_THREADS) void small_combine_kernel(int k, const double* __restrict__ A, int64_t lda,
                                                                  const double* __restrict__ B, int64_t ldb,
                                                                  double alpha, double sigma, int upper_half,
                                                                  double* __restrict__ out, int64_t ldo,
                                                                  double* __restrict__ nrm) {
  constexpr int U = 8;  // elements per thread whose loads are in flight together
  __shared__ double red[SC_THREADS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double ss = 0.0;
  const int total = k * k;  // k <= 512
  // thread tid takes the elements tid, tid + SC_THREADS, ... in that order
  for (int base = 0; base < total; base += SC_THREADS * U) {
    double va[U], vb[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = base + tid + SC_THREADS * u;
      const int i = e / k, j = e - (e / k) * k;
      va[u] = (e < total) ? A[(int64_t)i * lda + j] : 0.0;
      vb[u] = (e < total && B != nullptr) ? B[(int64_t)i * ldb + j] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = base + tid + SC_THREADS * u;
      if (e < total) {
        const int i = e / k, j = e - (e / k) * k;
        double v = va[u];
        if (B != nullptr) v += alpha * vb[u];
        if (i == j) v += sigma;
        ss += v * v;
        if (upper_half) v = (j > i) ? v : ((j == i) ? 0.5 * v : 0.0);
        out[(int64_t)i * ldo + j] = v;
      }
    }
  }
  if (nrm != nullptr) {
    ss = wave_sum(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    if (tid == 0) {
      double t = 0.0;
      for (int w = 0; w < SC_THREADS / 64; ++w) t += red[w];
      nrm[0] = sqrt(t);
    }
  }
}

// the same without the norm, over many workgroups: 8 elements per thread
constexpr int SCW_PER_BLOCK = 256 * 8;
__global__ __launch_bounds__(256) void small_combine_wide_kernel(int k, const double* __restrict__ A, int64_t lda,
                                                                 const double* __restrict__ B, int64_t ldb,
                                                                 double alpha, double sigma, int upper_half,
                                                                 double* __restrict__ out, int64_t ldo) {
  constexpr int U = SCW_PER_BLOCK / 256;
  const int total = k * k;  // k <= 512
  const int base = (int)blockIdx.x * SCW_PER_BLOCK + (int)threadIdx.x;
  double va[U], vb[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int e = base + 256 * u;
    const int i = e / k, j = e - (e / k) * k;
    va[u] = (e < total) ? A[(int64_t)i * lda + j] : 0.0;
    vb[u] = (e < total && B != nullptr) ? B[(int64_t)i * ldb + j] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int e = base + 256 * u;
    if (e < total) {
      const int i = e / k, j = e - (e / k) * k;
      double v = va[u];
      if (B != nullptr) v += alpha * vb[u];
      if (i == j) v += sigma;
      if (upper_half) v = (j > i) ? v : ((j == i) ? 0.5 * v : 0.0);
      out[(int64_t)i * ldo + j] = v;
    }
  }
}

__global__ __launch_bounds__(256) void cholqr_stats_kernel(int k, const double* __restrict__ G, int64_t ldg,
                                                          const int* __restrict__ info,
                                                          const double* __restrict__ enorm,
                                                          double* __restrict__ out) {
  __shared__ double smin[4], smax[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double mn = INFINITY, mx = 0.0;
  for (int i = tid; i < k; i += 256) {
    const double d = fabs(G[(int64_t)i * ldg + i]);
    mn = fmin(mn, d);
    mx = fmax(mx, d);
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
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 4; ++w) {
      mn = fmin(mn, smin[w]);
      mx = fmax(mx, smax[w]);
    }
    out[0] = mn;
    out[1] = mx;
    out[2] = (enorm != nullptr) ? enorm[0] : 0.0;
    out[3] = (double)info[0];
  }
}

}  // namespace

int pamd_potrf_run(int n, double* A, int64_t lda, int* info, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  if (n == 0) {
    potrf_zero_info_kernel<<<1, 1, 0, st>>>(info);
    PAMD_LAUNCH_CHECK();
    return PAMD_OK;
  }
  for (int j0 = 0; pr_width(n, j0) > 0; j0 += PR_LEAD) {
    if (pr_small(pr_width(n, j0)))
      potrf_reg_kernel<PR_SMALL><<<1, PR_THREADS, 0, st>>>(n, j0, A, lda, info);
    else
      potrf_reg_kernel<PR_LARGE><<<1, PR_THREADS, 0, st>>>(n, j0, A, lda, info);
    PAMD_LAUNCH_CHECK();
    const int r = n - j0;
    if (r <= PR_MAXN) break;
    double* Aj = A + j0 * (lda + 1);
    const int T = pr_trailing(r);
    potrf_row_kernel<<<(unsigned)T, 256, 0, st>>>(r, Aj, lda, info);
    PAMD_LAUNCH_CHECK();
    potrf_trailing_kernel<<<(unsigned)(T * (T + 1) / 2), 64, 0, st>>>(r, Aj, lda, info);
    PAMD_LAUNCH_CHECK();
  }
  return PAMD_OK;
}

extern "C" int pamd_potrf_upper_f64(int64_t n, double* A, int64_t lda, int* info, void* stream) {
  PAMD_ARG_CHECK(n >= 0 && n <= POTRF_MAX_N, 1);
  PAMD_ARG_CHECK(A != nullptr || n == 0, 2);
  PAMD_ARG_CHECK(lda >= n && lda >= 1, 3);
  PAMD_ARG_CHECK(info != nullptr, 4);
  return pamd_potrf_run((int)n, A, lda, info, stream);
}

#define PAMD_TRSM_MAX_N 2048

extern "C" int pamd_trsm_right_upper_f64(int64_t m, int64_t n, const double* R, int64_t ldr, double* B, int64_t ldb,
                                         void* stream) {
  PAMD_ARG_CHECK(m >= 0, 1);
  PAMD_ARG_CHECK(n >= 0 && n <= PAMD_TRSM_MAX_N, 2);
  PAMD_ARG_CHECK(R != nullptr || n == 0, 3);
  PAMD_ARG_CHECK(ldr >= n && ldr >= 1, 4);
  PAMD_ARG_CHECK(B != nullptr || m * n == 0, 5);
  PAMD_ARG_CHECK(ldb >= n && ldb >= 1, 6);
  if (m == 0 || n == 0) return PAMD_OK;
  const int rows = trsm_rows(n);
  const size_t shmem = (size_t)rows * n * sizeof(double);
  trsm_right_kernel<<<(unsigned)pamd_cdiv(m, rows), rows * 16, shmem, (hipStream_t)stream>>>(m, n, rows, R, ldr, B,
                                                                                             ldb);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

extern "C" int pamd_trtri_upper_f64(int64_t n, const double* R, int64_t ldr, double* Rinv, int64_t ldi,
                                    void* stream) {
  PAMD_ARG_CHECK(n >= 0 && n <= PAMD_TRSV_MAX_N, 1);
  PAMD_ARG_CHECK(R != nullptr || n == 0, 2);
  PAMD_ARG_CHECK(ldr >= n && ldr >= 1, 3);
  PAMD_ARG_CHECK(Rinv != nullptr || n == 0, 4);
  PAMD_ARG_CHECK(ldi >= n && ldi >= 1, 5);
  if (n == 0) return PAMD_OK;
  const size_t shmem = (size_t)(n + TRSV_SCRATCH_DOUBLES) * sizeof(double);
  trtri_kernel<<<(unsigned)n, 256, shmem, (hipStream_t)stream>>>(n, R, ldr, Rinv, ldi);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

// The steps that problems of up to nmax rows need.  Told the largest size, a
// batch of small problems is one launch, not the 14 of the largest allowed (us,
// 512 against the true size: 1 problem of 32 rows 34 / 5.4, 512 of 32 82 / 7.6,
// 64 of 200 78 / 55, 2000 of 40 287 / 43).
extern "C" int pamd_potrf_batched_nmax_f64(int64_t nprob, int64_t nmax, const int64_t* n, const int64_t* off,
                                           double* pool, int* info, void* stream) {
  PAMD_ARG_CHECK(nprob >= 0, 1);
  PAMD_ARG_CHECK(nmax >= 0 && nmax <= POTRF_MAX_N, 2);
  PAMD_ARG_CHECK(n != nullptr || nprob == 0, 3);
  PAMD_ARG_CHECK(off != nullptr || nprob == 0, 4);
  PAMD_ARG_CHECK(pool != nullptr || nprob == 0, 5);
  PAMD_ARG_CHECK(info != nullptr || nprob == 0, 6);
  if (nprob == 0) return PAMD_OK;
  hipStream_t st = (hipStream_t)stream;
  for (int j0 = 0;; j0 += PR_LEAD) {
    const int r = (int)nmax - j0;
    if (!pr_small(r)) {  // some problem's last rows may be more than the small instantiation takes
      potrf_batched_kernel<PR_LARGE><<<(unsigned)nprob, PR_THREADS, 0, st>>>(n, off, j0, pool, info);
      PAMD_LAUNCH_CHECK();
    }
    potrf_batched_kernel<PR_SMALL><<<(unsigned)nprob, PR_THREADS, 0, st>>>(n, off, j0, pool, info);
    PAMD_LAUNCH_CHECK();
    if (r <= PR_MAXN) break;
    const int T = pr_trailing(r);
    potrf_batched_row_kernel<<<dim3(T, (unsigned)nprob), 256, 0, st>>>(n, off, j0, pool, info);
    PAMD_LAUNCH_CHECK();
    potrf_batched_trailing_kernel<<<dim3(T * (T + 1) / 2, (unsigned)nprob), 64, 0, st>>>(n, off, j0, pool, info);
    PAMD_LAUNCH_CHECK();
  }
  return PAMD_OK;
}

extern "C" int pamd_potrf_batched_f64(int64_t nprob, const int64_t* n, const int64_t* off, double* pool, int* info,
                                      void* stream) {
  PAMD_ARG_CHECK(nprob >= 0, 1);
  PAMD_ARG_CHECK(n != nullptr || nprob == 0, 2);
  PAMD_ARG_CHECK(off != nullptr || nprob == 0, 3);
  PAMD_ARG_CHECK(pool != nullptr || nprob == 0, 4);
  PAMD_ARG_CHECK(info != nullptr || nprob == 0, 5);
  // the sizes are on the device: every step is launched for the largest one allowed
  return pamd_potrf_batched_nmax_f64(nprob, POTRF_MAX_N, n, off, pool, info, stream);
}

extern "C" int pamd_trtri_batched_f64(int64_t nprob, int64_t nmax, const int64_t* n, const int64_t* off,
                                      const double* R, double* Rinv, double* RinvT, void* stream) {
  PAMD_ARG_CHECK(nprob >= 0, 1);
  PAMD_ARG_CHECK(nmax >= 0 && nmax <= PAMD_TRSV_MAX_N, 2);
  PAMD_ARG_CHECK(n != nullptr || nprob == 0, 3);
  PAMD_ARG_CHECK(off != nullptr || nprob == 0, 4);
  PAMD_ARG_CHECK(R != nullptr || nprob == 0, 5);
  PAMD_ARG_CHECK(Rinv != nullptr || nprob == 0, 6);
  if (nprob == 0 || nmax == 0) return PAMD_OK;
  const size_t shmem = (size_t)(nmax + TRSV_SCRATCH_DOUBLES) * sizeof(double);
  dim3 grid((unsigned)nmax, (unsigned)nprob);
  trtri_batched_kernel<<<grid, 256, shmem, (hipStream_t)stream>>>(n, off, R, Rinv, RinvT);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

#define PAMD_TRSM_MFMA_MAX_K 512

int pamd_trsm_strip_run(int64_t m, int k, const double* R, int64_t ldr, const double* Y, int64_t ldy, double* X,
                        int64_t ldx, double* dinv, void* stream, const int* skip) {
  hipStream_t st = (hipStream_t)stream;
  trsm_dinv_kernel<<<(unsigned)pamd_cdiv(k, TS_B), 64, 0, st>>>(k, R, ldr, dinv);
  PAMD_LAUNCH_CHECK();
  trsm_strip_kernel<<<(unsigned)pamd_cdiv(m, TS_B), 256, trsm_strip_lds(k), st>>>(m, k, Y, ldy, R, ldr, dinv, X, ldx,
                                                                                         skip);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

extern "C" int pamd_trsm_mfma_workspace(int64_t k, int64_t* bytes) {
  PAMD_ARG_CHECK(k >= 0 && k <= PAMD_TRSM_MFMA_MAX_K, 1);
  PAMD_ARG_CHECK(bytes != nullptr, 2);
  *bytes = imax64(1, pamd_cdiv(k, TS_B)) * TS_B * TS_B * (int64_t)sizeof(double);
  return PAMD_OK;
}

extern "C" int pamd_trsm_right_upper_mfma_f64(int64_t m, int64_t k, const double* R, int64_t ldr, const double* Y,
                                              int64_t ldy, double* X, int64_t ldx, void* workspace, void* stream) {
  PAMD_ARG_CHECK(m >= 0, 1);
  PAMD_ARG_CHECK(k >= 0 && k <= PAMD_TRSM_MFMA_MAX_K, 2);
  PAMD_ARG_CHECK(R != nullptr || k == 0, 3);
  PAMD_ARG_CHECK(ldr >= k && ldr >= 1, 4);
  PAMD_ARG_CHECK(Y != nullptr || m * k == 0, 5);
  PAMD_ARG_CHECK(ldy >= k && ldy >= 1, 6);
  PAMD_ARG_CHECK(X != nullptr || m * k == 0, 7);
  PAMD_ARG_CHECK(ldx >= k && ldx >= 1, 8);
  PAMD_ARG_CHECK(workspace != nullptr || k == 0, 9);
  if (m == 0 || k == 0) return PAMD_OK;
  return pamd_trsm_strip_run(m, (int)k, R, ldr, Y, ldy, X, ldx, (double*)workspace, stream);
}

extern "C" int pamd_small_combine_f64(int64_t k, const double* A, int64_t lda, const double* B, int64_t ldb,
                                      double alpha, double sigma, int upper_half, double* out, int64_t ldo,
                                      double* nrm, void* stream) {
  PAMD_ARG_CHECK(k >= 0 && k <= 512, 1);
  PAMD_ARG_CHECK(A != nullptr || k == 0, 2);
  PAMD_ARG_CHECK(lda >= k && lda >= 1, 3);
  PAMD_ARG_CHECK(B == nullptr || ldb >= k, 5);
  PAMD_ARG_CHECK(upper_half == 0 || upper_half == 1, 8);
  PAMD_ARG_CHECK(out != nullptr || k == 0, 9);
  PAMD_ARG_CHECK(ldo >= k && ldo >= 1, 10);
  if (k == 0 && nrm == nullptr) return PAMD_OK;
  if (nrm == nullptr) {  // no reduction: spread over the chip
    small_combine_wide_kernel<<<(unsigned)pamd_cdiv(k * k, SCW_PER_BLOCK), 256, 0, (hipStream_t)stream>>>(
        (int)k, A, lda, B, ldb, alpha, sigma, upper_half, out, ldo);
  } else {
    small_combine_kernel<<<1, SC_THREADS, 0, (hipStream_t)stream>>>((int)k, A, lda, B, ldb, alpha, sigma, upper_half,
                                                                   out, ldo, nrm);
  }
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

extern "C" int pamd_cholqr_stats_f64(int64_t k, const double* G, int64_t ldg, const int* info, const double* enorm,
                                     double* out, void* stream) {
  PAMD_ARG_CHECK(k >= 1 && k <= 512, 1);
  PAMD_ARG_CHECK(G != nullptr, 2);
  PAMD_ARG_CHECK(ldg >= k, 3);
  PAMD_ARG_CHECK(info != nullptr, 4);
  PAMD_ARG_CHECK(out != nullptr, 6);
  cholqr_stats_kernel<<<1, 256, 0, (hipStream_t)stream>>>((int)k, G, ldg, info, enorm, out);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}
