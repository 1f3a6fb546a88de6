// Learned leverage-score sketch: the MLP surrogate's forward and backward
// kernels, its Adam step, and the row-sampling gather.
//
// Network: 16 -> 64 -> 64 -> 1, ReLU hidden layers, scalar output (the
// predicted log of the normalised leverage score).  The inputs pass through
// asinh first: pre-sketch features of coherent rows are orders of magnitude
// larger than the rest, and asinh keeps their scale logarithmic, which is
// the scale of the target.  Weights are BF16 (the
// optimiser keeps FP32 masters and rounds them to nearest-even after each
// step); every product and sum is FP32.  Parameter vector layout (FP32
// master, and the same order for gradients):
//   W1[16][64] | b1[64] | W2[64][64] | b2[64] | w3[64] | b3        (5313)
// Forward: one thread evaluates one row; the BF16 weights are widened once per
// workgroup into LDS and read there by same-address (broadcast) loads.
// Backward recomputes the forward pass (cheaper than storing activations) on
// the matrix units; workgroup partials are summed in a fixed order by a second
// kernel, so the gradients are deterministic.
#include "common.h"
#include "rng.h"

namespace {

constexpr int MLP_IN = 16, MLP_H = 64;
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + MLP_IN * MLP_H, OFF_W2 = OFF_B1 + MLP_H,
              OFF_B2 = OFF_W2 + MLP_H * MLP_H, OFF_W3 = OFF_B2 + MLP_H, OFF_B3 = OFF_W3 + MLP_H,
              MLP_NPARAM = OFF_B3 + 1;
constexpr int MLP_THREADS = 256;

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));  // inf/nan
  const uint32_t lsb = (u >> 16) & 1u;
  return (uint16_t)((u + 0x7fffu + lsb) >> 16);
}

struct MlpLds {
  float w1[MLP_IN][MLP_H];
  float b1[MLP_H];
  float w2[MLP_H][MLP_H];
  float b2[MLP_H];
  float w3[MLP_H];
  float b3;
};

__device__ inline void load_weights(MlpLds& s, const uint16_t* __restrict__ wb, const float* __restrict__ bias) {
  // wb: BF16 weights W1 | W2 | w3 (16*64 + 64*64 + 64); bias: FP32 b1 | b2 | b3
  for (int e = threadIdx.x; e < MLP_IN * MLP_H; e += blockDim.x) (&s.w1[0][0])[e] = bf16_to_f32(wb[e]);
  for (int e = threadIdx.x; e < MLP_H * MLP_H; e += blockDim.x)
    (&s.w2[0][0])[e] = bf16_to_f32(wb[MLP_IN * MLP_H + e]);
  for (int e = threadIdx.x; e < MLP_H; e += blockDim.x) {
    s.w3[e] = bf16_to_f32(wb[MLP_IN * MLP_H + MLP_H * MLP_H + e]);
    s.b1[e] = bias[e];
    s.b2[e] = bias[MLP_H + e];
  }
  if (threadIdx.x == 0) s.b3 = bias[2 * MLP_H];
}

// h1 = relu(W1^T x + b1) -> hrow (this thread's LDS row), h2 = relu(W2^T h1
// + b2) in registers, y = w3 . h2 + b3.  The second layer walks k through
// LDS (a register array may only be indexed with compile-time indices).
__device__ __forceinline__ float mlp_eval(const MlpLds& s, const float (&x)[MLP_IN], float* hrow,
                                          float (&h2)[MLP_H]) {
#pragma unroll
  for (int j = 0; j < MLP_H; ++j) {
    float a = s.b1[j];
#pragma unroll
    for (int k = 0; k < MLP_IN; ++k) a = fmaf(x[k], s.w1[k][j], a);
    hrow[j] = fmaxf(a, 0.f);
  }
#pragma unroll
  for (int j = 0; j < MLP_H; ++j) h2[j] = s.b2[j];
  for (int k = 0; k < MLP_H; ++k) {
    const float hk = hrow[k];
#pragma unroll
    for (int j = 0; j < MLP_H; ++j) h2[j] = fmaf(hk, s.w2[k][j], h2[j]);
  }
  float y = s.b3;
#pragma unroll
  for (int j = 0; j < MLP_H; ++j) {
    h2[j] = fmaxf(h2[j], 0.f);
    y = fmaf(h2[j], s.w3[j], y);
  }
  return y;
}

__global__ __launch_bounds__(MLP_THREADS) void mlp_fwd_kernel(int64_t rows, const float* __restrict__ X, int64_t ldx,
                                                               const uint16_t* __restrict__ wb,
                                                               const float* __restrict__ bias, float* __restrict__ y) {
  __shared__ MlpLds s;
  __shared__ float hrow[MLP_THREADS][MLP_H + 1];
  load_weights(s, wb, bias);
  __syncthreads();
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows) return;
  float x[MLP_IN], h2[MLP_H];
#pragma unroll
  for (int k = 0; k < MLP_IN; ++k) x[k] = asinhf(X[r * ldx + k]);
  y[r] = mlp_eval(s, x, hrow[threadIdx.x], h2);
}

// ---------------------------------------------------------------------------
// Backward.  Loss = (1 / rows_total) sum_r (y_r - t_r)^2 over this call's rows;
// partial gradients part[blockIdx.x][0 .. MLP_NPARAM) and the partial loss in
// part[blockIdx.x][MLP_NPARAM].
//
// Every product is v_mfma_f32_16x16x4f32 (FP32 products and sums), one
// wavefront per tile of 16 rows, so that an operand value read from LDS or
// held in a register serves sixteen products instead of one (one thread per
// row spent 118 us at 65536 rows on LDS reads of the weights and of the rows'
// activations; the arithmetic is 13 us at the matrix units' rate).  The result
// layout (lane l, item r: row 4 (l / 16) + r, column l % 16) is the A and B
// operand layout of a product whose k index runs over (4 (l / 16) + r), so with
// the k order chosen to match, results feed the next product from registers:
//   H1t (units x rows) = W1^T X^T   -> left operand of H2
//   H1  (rows x units) = X W1       -> left operand (transposed) of dW2, mask of dH1
//   H2  (rows x units) = H1 W2, dH2 -> right operand of dW2
//   dH1 (rows x units) = dH2 W2^T   -> right operand of dW1
// and only dH2 passes through LDS, to become dH1's left operand.  dW2, dW1 and
// the bias gradients stay in registers over the wavefront's tiles, with more
// than BW_TILES of them (LONG) over that many; then the eight wavefronts' are
// added and the workgroup goes on in FP64, so that no FP32 sum runs over more
// than 256 rows and eight terms however many rows there are (2^24 equal rows:
// the largest relative error of an entry 1.2e-4 without, 3.9e-6 with; LONG on
// every call would add 2 us to the 44 of 65536 rows).
// ---------------------------------------------------------------------------
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int BW_WAVES = 8;
constexpr int BW_THREADS = 64 * BW_WAVES;
constexpr int BW_MAX_GRID = 256;  // one workgroup per CU; further rows are looped over
constexpr int BW_TILES = 16;      // tiles of 16 rows per wavefront that are summed in FP32

inline int64_t bw_grid(int64_t rows) {
  return imax64(1, imin64(BW_MAX_GRID, pamd_cdiv(rows, 16 * BW_WAVES)));
}

struct BwLds {
  f4 w2[4][4][64];    // [i][j][lane]: W2[16 i + 4 g + r][16 j + c], g = lane / 16, c = lane % 16
  f4 w2t[4][4][64];   // [j][i][lane]: W2[16 i + c][16 j + 4 g + r]
  float dh2[BW_WAVES][16][MLP_H + 4];
};

__device__ __forceinline__ float row16_sum(float v) {
  v += dpp_f32<0xb1>(v);
  v += dpp_f32<0x4e>(v);
  v += dpp_f32<0x124>(v);
  return v + dpp_f32<0x128>(v);
}

template <bool LONG>
__global__ __launch_bounds__(BW_THREADS) void mlp_bwd_kernel(int64_t rows, double inv_total,
                                                             const float* __restrict__ X, int64_t ldx,
                                                             const float* __restrict__ t,
                                                             const uint16_t* __restrict__ wb,
                                                             const float* __restrict__ bias,
                                                             float* __restrict__ part) {
  __shared__ BwLds s;
  __shared__ float sum[MLP_NPARAM + 1];                // the wavefronts' sums over up to BW_TILES tiles each
  __shared__ double tot[LONG ? MLP_NPARAM + 1 : 1];    // the sums before those
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  // scalar where that saves a spilled register (13 -> 11; with LONG it costs eight more)
  const int wave = LONG ? tid >> 6 : __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint16_t* wb2 = wb + MLP_IN * MLP_H;
  for (int e = tid; e < 4 * 4 * 64; e += BW_THREADS) {
    const int hi = e >> 8, lo = (e >> 6) & 3, l = e & 63, lc = l & 15, lg = l >> 4;
    f4 u, v;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      u[r] = bf16_to_f32(wb2[(16 * hi + 4 * lg + r) * MLP_H + 16 * lo + lc]);
      v[r] = bf16_to_f32(wb2[(16 * lo + lc) * MLP_H + 16 * hi + 4 * lg + r]);
    }
    s.w2[hi][lo][l] = u;
    s.w2t[hi][lo][l] = v;
  }
  for (int e = tid; e <= MLP_NPARAM; e += BW_THREADS) {
    sum[e] = 0.f;
    if (LONG) tot[e] = 0.0;
  }
  // this lane's weights: W1[4 q + g][16 i + c], the biases by unit
  float w1[4][4], b1n[4], b2n[4], w3n[4];
  f4 b1t[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int q = 0; q < 4; ++q) w1[q][i] = bf16_to_f32(wb[(4 * q + g) * MLP_H + 16 * i + c]);
    b1n[i] = bias[16 * i + c];
    b2n[i] = bias[MLP_H + 16 * i + c];
    w3n[i] = bf16_to_f32(wb2[MLP_H * MLP_H + 16 * i + c]);
#pragma unroll
    for (int r = 0; r < 4; ++r) b1t[i][r] = bias[16 * i + 4 * g + r];
  }
  const float b3 = bias[2 * MLP_H], inv = (float)inv_total, inv2 = (float)(2.0 * inv_total);
  __syncthreads();

  f4 dw2[4][4], dw1[4];
  float db1[4], db2[4], dw3[4], db3, loss;
  auto clear = [&] {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j) dw2[i][j] = f4{0.f, 0.f, 0.f, 0.f};
      dw1[i] = f4{0.f, 0.f, 0.f, 0.f};
      db1[i] = db2[i] = dw3[i] = 0.f;
    }
    db3 = loss = 0.f;
  };
  // the registers of the workgroup's wavefronts to sum, wavefront after wavefront
  auto add_up = [&] {
    // the bias sums over the four row groups; db3 and the loss are the same in a row group's lanes
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      db1[i] += __shfl_xor(db1[i], 16, 64);
      db1[i] += __shfl_xor(db1[i], 32, 64);
      db2[i] += __shfl_xor(db2[i], 16, 64);
      db2[i] += __shfl_xor(db2[i], 32, 64);
      dw3[i] += __shfl_xor(dw3[i], 16, 64);
      dw3[i] += __shfl_xor(dw3[i], 32, 64);
    }
    db3 += __shfl_xor(db3, 16, 64);
    db3 += __shfl_xor(db3, 32, 64);
    loss += __shfl_xor(loss, 16, 64);
    loss += __shfl_xor(loss, 32, 64);
    for (int w = 0; w < BW_WAVES; ++w) {
      __syncthreads();
      if (w != wave) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
          for (int j = 0; j < 4; ++j) sum[OFF_W2 + (16 * i + 4 * g + r) * MLP_H + 16 * j + c] += dw2[i][j][r];
          sum[OFF_W1 + (4 * g + r) * MLP_H + 16 * i + c] += dw1[i][r];
        }
        if (g == 0) {
          sum[OFF_B1 + 16 * i + c] += db1[i];
          sum[OFF_B2 + 16 * i + c] += db2[i];
          sum[OFF_W3 + 16 * i + c] += dw3[i];
        }
      }
      if (lane == 0) {
        sum[OFF_B3] += db3;
        sum[MLP_NPARAM] += loss;
      }
    }
    __syncthreads();
  };
  clear();
  float(*T)[MLP_H + 4] = s.dh2[wave];
  const int64_t step = (int64_t)gridDim.x * BW_WAVES * 16;
  auto tile = [&](int64_t r0) {
    float x[4], xt[4], tr[4];  // X[c][4 q + g], X[4 g + r][c], t[4 g + r] (rows past the end: zero)
    const bool in = r0 + c < rows;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t rr = r0 + 4 * g + q;
      x[q] = in ? asinhf(X[(r0 + c) * ldx + 4 * q + g]) : 0.f;
      xt[q] = rr < rows ? asinhf(X[rr * ldx + c]) : 0.f;
      tr[q] = rr < rows ? t[rr] : 0.f;
    }
    f4 h1t[4], h1[4], h2[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      h1t[i] = b1t[i];
      h1[i] = f4{b1n[i], b1n[i], b1n[i], b1n[i]};
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        h1t[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[q][i], x[q], h1t[i], 0, 0, 0);
        h1[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[q], w1[q][i], h1[i], 0, 0, 0);
      }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        h1t[i][r] = fmaxf(h1t[i][r], 0.f);
        h1[i][r] = fmaxf(h1[i][r], 0.f);
      }
#pragma unroll
    for (int j = 0; j < 4; ++j) h2[j] = f4{b2n[j], b2n[j], b2n[j], b2n[j]};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f4 w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = s.w2[i][j][lane];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < 4; ++j) h2[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(h1t[i][r], w[j][r], h2[j], 0, 0, 0);
    }
    // y of rows 4 g + r, in every lane of the row group; h2 <- relu, then dH2
    float dy[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float y = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        h2[j][r] = fmaxf(h2[j][r], 0.f);
        y = fmaf(h2[j][r], w3n[j], y);
      }
      const float diff = (r0 + 4 * g + r < rows) ? row16_sum(y) + b3 - tr[r] : 0.f;
      dy[r] = inv2 * diff;
      db3 += dy[r];
      loss += inv * diff * diff;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        dw3[j] = fmaf(dy[r], h2[j][r], dw3[j]);
        h2[j][r] = h2[j][r] > 0.f ? dy[r] * w3n[j] : 0.f;
        db2[j] += h2[j][r];
        T[4 * g + r][16 * j + c] = h2[j][r];
      }
    // dW2[16 i ..][16 j ..] += H1^T dH2 (k: the rows 4 g + r)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          dw2[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(h1[i][r], h2[j][r], dw2[i][j], 0, 0, 0);
    PAMD_WAVE_SYNC();
    // dH1 = dH2 W2^T, k over the units 16 j + 4 g + r of row c
    f4 d1[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) d1[i] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f4 a = *reinterpret_cast<const f4*>(&T[c][16 * j + 4 * g]);
      f4 w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = s.w2t[j][i][lane];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) d1[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], w[i][r], d1[i], 0, 0, 0);
    }
    PAMD_WAVE_SYNC();  // T is written again by the next tile
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        d1[i][r] = h1[i][r] > 0.f ? d1[i][r] : 0.f;
        db1[i] += d1[i][r];
      }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) dw1[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(xt[r], d1[i][r], dw1[i], 0, 0, 0);
  };
  const int64_t first = ((int64_t)blockIdx.x * BW_WAVES + wave) * 16;
  if constexpr (LONG) {
    // as many rounds for every wavefront (some of the last one past the end), for the barriers of add_up
    const int rounds = (int)pamd_cdiv(imax64(0, rows - (int64_t)blockIdx.x * BW_WAVES * 16), step);
    for (int it = 0; it < rounds; ++it) {
      if (it && it % BW_TILES == 0) {
        add_up();
        clear();
        for (int e = tid; e <= MLP_NPARAM; e += BW_THREADS) {  // seen by the others after the next add_up's barrier
          tot[e] += (double)sum[e];
          sum[e] = 0.f;
        }
      }
      if (first + it * step < rows) tile(first + it * step);
    }
  } else {
    for (int64_t r0 = first; r0 < rows; r0 += step) tile(r0);
  }
  add_up();
  float* out = part + (int64_t)blockIdx.x * (MLP_NPARAM + 1);
  for (int e = tid; e <= MLP_NPARAM; e += BW_THREADS) out[e] = LONG ? (float)(tot[e] + (double)sum[e]) : sum[e];
}

// grad[e] = the workgroups' sums in FP64: 64 entries per workgroup, its four
// wavefronts take the partials g = w, w + 4, ... with eight in flight, and
// their sums are added in order (one thread per entry walking all 256
// partials took 62 us)
__global__ __launch_bounds__(256) void mlp_reduce_kernel(int nparts, const float* __restrict__ part,
                                                         float* __restrict__ grad) {
  constexpr int U = 8;
  __shared__ double red[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int e = (int)blockIdx.x * 64 + lane;
  double acc = 0.0;
  if (e <= MLP_NPARAM) {
    const float* p = part + e;
    int g = wave;
    for (; g + (U - 1) * 4 < nparts; g += 4 * U) {
      float v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = p[(int64_t)(g + 4 * u) * (MLP_NPARAM + 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) acc += (double)v[u];
    }
    for (; g < nparts; g += 4) acc += (double)p[(int64_t)g * (MLP_NPARAM + 1)];
  }
  red[wave][lane] = acc;
  __syncthreads();
  if (wave == 0 && e <= MLP_NPARAM)
    grad[e] = (float)((red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]));
}

// Adam on the FP32 masters; refresh the BF16 weights and FP32 biases.
__global__ void mlp_adam_kernel(float* __restrict__ w, float* __restrict__ m, float* __restrict__ v,
                                const float* __restrict__ g, float lr, float beta1, float beta2, float eps,
                                float bc1, float bc2, uint16_t* __restrict__ wb, float* __restrict__ bias) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= MLP_NPARAM) return;
  const float ge = g[e];
  const float me = beta1 * m[e] + (1.f - beta1) * ge;
  const float ve = beta2 * v[e] + (1.f - beta2) * ge * ge;
  m[e] = me;
  v[e] = ve;
  const float we = w[e] - lr * (me / bc1) / (sqrtf(ve / bc2) + eps);
  w[e] = we;
  // publish: BF16 weights W1 | W2 | w3, FP32 biases b1 | b2 | b3
  if (e < OFF_B1) {
    wb[e] = f32_to_bf16_rne(we);
  } else if (e < OFF_W2) {
    bias[e - OFF_B1] = we;
  } else if (e < OFF_B2) {
    wb[MLP_IN * MLP_H + (e - OFF_W2)] = f32_to_bf16_rne(we);
  } else if (e < OFF_W3) {
    bias[MLP_H + (e - OFF_B2)] = we;
  } else if (e < OFF_B3) {
    wb[MLP_IN * MLP_H + MLP_H * MLP_H + (e - OFF_W3)] = f32_to_bf16_rne(we);
  } else {
    bias[2 * MLP_H] = we;
  }
}

// out[r][:] = scale[r] * A[idx[r]][:]
__global__ void row_gather_kernel(int64_t d, int64_t n, const int64_t* __restrict__ idx,
                                  const double* __restrict__ scale, const double* __restrict__ A, int64_t lda,
                                  double* __restrict__ out, int64_t ldo) {
  const int64_t r = blockIdx.x;
  const double sc = scale ? scale[r] : 1.0;
  const double* src = A + idx[r] * lda;
  for (int64_t c = threadIdx.x; c < n; c += blockDim.x) out[r * ldo + c] = sc * src[c];
}

// out[idx[r], :] = A[r, :]: one workgroup per source row
__global__ void row_scatter_kernel(int64_t n, const int64_t* __restrict__ idx, const double* __restrict__ A,
                                   int64_t lda, double* __restrict__ out, int64_t ldo) {
  const int64_t r = blockIdx.x;
  double* dst = out + idx[r] * ldo;
  const double* src = A + r * lda;
  for (int64_t c = threadIdx.x; c < n; c += blockDim.x) dst[c] = src[c];
}

}  // namespace

extern "C" int pamd_mlp_nparams(void) { return MLP_NPARAM; }

extern "C" int pamd_mlp_fwd(int64_t rows, const float* X, int64_t ldx, const uint16_t* wb, const float* bias,
                            float* y, void* stream) {
  PAMD_ARG_CHECK(rows >= 0, 1);
  PAMD_ARG_CHECK(X != nullptr || rows == 0, 2);
  PAMD_ARG_CHECK(ldx >= MLP_IN, 3);
  PAMD_ARG_CHECK(wb != nullptr, 4);
  PAMD_ARG_CHECK(bias != nullptr, 5);
  PAMD_ARG_CHECK(y != nullptr || rows == 0, 6);
  if (rows == 0) return PAMD_OK;
  mlp_fwd_kernel<<<(unsigned)pamd_cdiv(rows, MLP_THREADS), MLP_THREADS, 0, (hipStream_t)stream>>>(rows, X, ldx, wb,
                                                                                                   bias, y);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

extern "C" int pamd_mlp_bwd_workspace(int64_t rows, int64_t* bytes) {
  PAMD_ARG_CHECK(rows >= 0, 1);
  PAMD_ARG_CHECK(bytes != nullptr, 2);
  *bytes = bw_grid(rows) * (MLP_NPARAM + 1) * (int64_t)sizeof(float);
  return PAMD_OK;
}

extern "C" int pamd_mlp_bwd(int64_t rows, int64_t rows_total, const float* X, int64_t ldx, const float* t,
                            const uint16_t* wb, const float* bias, float* grad, void* workspace, void* stream) {
  PAMD_ARG_CHECK(rows >= 1, 1);
  PAMD_ARG_CHECK(rows_total >= rows, 2);
  PAMD_ARG_CHECK(X != nullptr, 3);
  PAMD_ARG_CHECK(ldx >= MLP_IN, 4);
  PAMD_ARG_CHECK(t != nullptr, 5);
  PAMD_ARG_CHECK(wb != nullptr, 6);
  PAMD_ARG_CHECK(bias != nullptr, 7);
  PAMD_ARG_CHECK(grad != nullptr, 8);
  PAMD_ARG_CHECK(workspace != nullptr, 9);
  hipStream_t st = (hipStream_t)stream;
  const int64_t nblk = bw_grid(rows);
  float* part = (float*)workspace;
  const double inv = 1.0 / (double)rows_total;
  if (rows > nblk * BW_WAVES * 16 * BW_TILES)
    mlp_bwd_kernel<true><<<(unsigned)nblk, BW_THREADS, 0, st>>>(rows, inv, X, ldx, t, wb, bias, part);
  else
    mlp_bwd_kernel<false><<<(unsigned)nblk, BW_THREADS, 0, st>>>(rows, inv, X, ldx, t, wb, bias, part);
  PAMD_LAUNCH_CHECK();
  mlp_reduce_kernel<<<(unsigned)pamd_cdiv(MLP_NPARAM + 1, 64), 256, 0, st>>>((int)nblk, part, grad);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

extern "C" int pamd_mlp_adam(float* w, float* m, float* v, const float* grad, float lr, float beta1, float beta2,
                             float eps, int64_t step, uint16_t* wb, float* bias, void* stream) {
  PAMD_ARG_CHECK(w != nullptr, 1);
  PAMD_ARG_CHECK(m != nullptr, 2);
  PAMD_ARG_CHECK(v != nullptr, 3);
  PAMD_ARG_CHECK(grad != nullptr, 4);
  PAMD_ARG_CHECK(lr > 0.f, 5);
  PAMD_ARG_CHECK(step >= 1, 9);
  PAMD_ARG_CHECK(wb != nullptr, 10);
  PAMD_ARG_CHECK(bias != nullptr, 11);
  const float bc1 = 1.f - powf(beta1, (float)step), bc2 = 1.f - powf(beta2, (float)step);
  mlp_adam_kernel<<<(unsigned)pamd_cdiv(MLP_NPARAM, 256), 256, 0, (hipStream_t)stream>>>(w, m, v, grad, lr, beta1,
                                                                                         beta2, eps, bc1, bc2, wb,
                                                                                         bias);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

extern "C" int pamd_row_gather_f64(int64_t d, int64_t m, int64_t n, const int64_t* idx, const double* scale,
                                   const double* A, int64_t lda, double* out, int64_t ldo, void* stream) {
  PAMD_ARG_CHECK(d >= 0, 1);
  PAMD_ARG_CHECK(m >= 1, 2);
  PAMD_ARG_CHECK(n >= 0, 3);
  PAMD_ARG_CHECK(idx != nullptr || d == 0, 4);
  PAMD_ARG_CHECK(A != nullptr, 6);
  PAMD_ARG_CHECK(lda >= n, 7);
  PAMD_ARG_CHECK(out != nullptr || d == 0, 8);
  PAMD_ARG_CHECK(ldo >= n, 9);
  if (d == 0 || n == 0) return PAMD_OK;
  row_gather_kernel<<<(unsigned)d, 256, 0, (hipStream_t)stream>>>(d, n, idx, scale, A, lda, out, ldo);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

extern "C" int pamd_row_scatter_f64(int64_t d, int64_t m, int64_t n, const int64_t* idx, const double* A,
                                    int64_t lda, double* out, int64_t ldo, void* stream) {
  PAMD_ARG_CHECK(d >= 0, 1);
  PAMD_ARG_CHECK(m >= d, 2);
  PAMD_ARG_CHECK(n >= 0, 3);
  PAMD_ARG_CHECK(idx != nullptr || d == 0, 4);
  PAMD_ARG_CHECK(A != nullptr || d == 0, 5);
  PAMD_ARG_CHECK(lda >= n, 6);
  PAMD_ARG_CHECK(out != nullptr || d == 0, 7);
  PAMD_ARG_CHECK(ldo >= n, 8);
  if (d == 0 || n == 0) return PAMD_OK;
  row_scatter_kernel<<<(unsigned)d, 256, 0, (hipStream_t)stream>>>(n, idx, A, lda, out, ldo);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}

namespace {

// Inclusive prefix sums of the m row weights p in one 1024-thread workgroup:
// thread t sums its contiguous chunk in order, thread 0 scans the 1024 chunk
// totals in order, then each thread writes its chunk's running sums.  A fixed
// summation order, so the CDF is run-to-run identical.
__global__ __launch_bounds__(1024) void weights_cdf_kernel(int64_t m, const double* __restrict__ p,
                                                           double* __restrict__ cdf) {
  __shared__ double tot[1024];
  const int t = threadIdx.x;
  const int64_t chunk = pamd_cdiv(m, 1024);
  const int64_t i0 = imin64(m, (int64_t)t * chunk), i1 = imin64(m, i0 + chunk);
  // the chunk's weights eight at a time (loads issued together, added in order)
  double s = 0.0;
  for (int64_t i = i0; i < i1; i += 8) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = (i + u < i1) ? p[i + u] : 0.0;
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i + u < i1) s += v[u];
  }
  tot[t] = s;
  __syncthreads();
  if (t == 0) {
    double run = 0.0;
    for (int k = 0; k < 1024; k += 8) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = tot[k + u];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        tot[k + u] = run;
        run += v[u];
      }
    }
  }
  __syncthreads();
  double run = tot[t];
  for (int64_t i = i0; i < i1; i += 8) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = (i + u < i1) ? p[i + u] : 0.0;
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i + u < i1) {
        run += v[u];
        cdf[i + u] = run;
      }
  }
}

// Draw i: u in (0, 1] from Philox-4x32-10 at counter i, the row j with
// cdf[j - 1] < u * total <= cdf[j] (binary search; a row of weight 0 is never
// chosen since u > 0), and the scale 1 / sqrt(d p_j / total) of a sampling
// sketch with replacement.
__global__ void sample_rows_kernel(int64_t m, int64_t d, uint64_t seed, const double* __restrict__ p,
                                   const double* __restrict__ cdf, int64_t* __restrict__ idx,
                                   double* __restrict__ scale) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d) return;
  const U4 r = philox4x32_10(U4{(uint32_t)i, (uint32_t)(i >> 32), 0x3C6EF372u, 0x510E527Fu}, (uint32_t)seed,
                             (uint32_t)(seed >> 32));
  const double total = cdf[m - 1];
  const double target = u53_open0(r.x, r.y) * total;
  int64_t lo = 0, hi = m - 1;
  while (lo < hi) {
    const int64_t mid = lo + (hi - lo) / 2;
    if (cdf[mid] >= target)
      hi = mid;
    else
      lo = mid + 1;
  }
  idx[i] = lo;
  scale[i] = 1.0 / sqrt((double)d * p[lo] / total);
}

}  // namespace

extern "C" int pamd_sample_rows_workspace(int64_t m, int64_t* bytes) {
  PAMD_ARG_CHECK(m >= 1, 1);
  PAMD_ARG_CHECK(bytes != nullptr, 2);
  *bytes = m * (int64_t)sizeof(double);
  return PAMD_OK;
}

extern "C" int pamd_sample_rows_f64(int64_t m, const double* p, int64_t d, uint64_t seed, int64_t* idx,
                                    double* scale, void* workspace, void* stream) {
  PAMD_ARG_CHECK(m >= 1, 1);
  PAMD_ARG_CHECK(p != nullptr, 2);
  PAMD_ARG_CHECK(d >= 0, 3);
  PAMD_ARG_CHECK(idx != nullptr || d == 0, 5);
  PAMD_ARG_CHECK(scale != nullptr || d == 0, 6);
  PAMD_ARG_CHECK(workspace != nullptr, 7);
  if (d == 0) return PAMD_OK;
  hipStream_t st = (hipStream_t)stream;
  double* cdf = (double*)workspace;
  weights_cdf_kernel<<<1, 1024, 0, st>>>(m, p, cdf);
  PAMD_LAUNCH_CHECK();
  sample_rows_kernel<<<(unsigned)pamd_cdiv(d, 256), 256, 0, st>>>(m, d, seed, p, cdf, idx, scale);
  PAMD_LAUNCH_CHECK();
  return PAMD_OK;
}
