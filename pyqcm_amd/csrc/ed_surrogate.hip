// ed_surrogate.hip -- kernels of the learned surrogate (gfx950).
//
// The MLP's layers are GEMMs on the matrix cores: bf16 operands staged in LDS,
// v_mfma_f32_16x16x32_bf16 with fp32 accumulation, and the bias / GELU /
// GELU-derivative work fused into the GEMM epilogue.  Master weights, Adam
// moments, pre-activations and gradients are fp32; activations and the
// GEMM-side gradients are bf16.  Every reduction has a fixed order.
#include <algorithm>
#include <cmath>

#include "ed_surrogate.hpp"

namespace ed {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kBM = 64, kBN = 64, kBK = 32;
constexpr int kLdsPitch = kBK + 8;  // bf16 per LDS row: 80 B, keeps the 16-byte fragment reads aligned

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float z) {
  return 0.5f * (1.f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// One 64 x 64 tile of C per block of 4 waves (2 x 2); each wave owns 32 x 32 =
// 2 x 2 MFMA tiles of 16 x 16, accumulated over k in steps of 32.
// Fragment layout of v_mfma_f32_16x16x32_bf16 (wave64): lane l supplies row
// l % 16 of A and column l % 16 of B, each with the 8 consecutive k values
// 8 * (l / 16) .. + 7; it receives D rows 4 * (l / 16) .. + 3 of column l % 16.
template <int EPI, bool AKC, bool BKC>
__global__ __launch_bounds__(256) void k_gemm(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) bf16_t As[kBM * kLdsPitch];
  __shared__ __attribute__((aligned(16))) bf16_t Bs[kBN * kLdsPitch];
  const int t = threadIdx.x, l = t & 63, w = t >> 6, wm = w >> 1, wn = w & 1;
  const int m0 = blockIdx.x * kBM, n0 = blockIdx.y * kBN;
  const int nkt = (g.K + kBK - 1) / kBK;
  const int per = (nkt + g.ksplit - 1) / g.ksplit;
  const int kt0 = blockIdx.z * per, kt1 = min(nkt, kt0 + per);
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bf16x8 zero8 = {};
  for (int kt = kt0; kt < kt1; ++kt) {
    const int k0 = kt * kBK;
    // stage A (64 x 32) and B (32 x 64): 256 chunks of 8 bf16 each
    if (AKC) {
      const int r = t >> 2, kc = (t & 3) * 8, m = m0 + r, k = k0 + kc;
      bf16x8 v = zero8;
      if (m < g.M && k < g.Kpad) v = *(const bf16x8 *)(g.A + (long)m * g.sam + k);
      *(bf16x8 *)&As[r * kLdsPitch + kc] = v;
    } else {
      const int kk = t >> 3, mc = (t & 7) * 8, k = k0 + kk, m = m0 + mc;
      bf16x8 v = zero8;
      if (k < g.K && m < g.Mpad) v = *(const bf16x8 *)(g.A + (long)k * g.sak + m);
#pragma unroll
      for (int j = 0; j < 8; ++j) As[(mc + j) * kLdsPitch + kk] = v[j];
    }
    if (BKC) {
      const int r = t >> 2, kc = (t & 3) * 8, n = n0 + r, k = k0 + kc;
      bf16x8 v = zero8;
      if (n < g.N && k < g.Kpad) v = *(const bf16x8 *)(g.B + (long)n * g.sbn + k);
      *(bf16x8 *)&Bs[r * kLdsPitch + kc] = v;
    } else {
      const int kk = t >> 3, nc = (t & 7) * 8, k = k0 + kk, n = n0 + nc;
      bf16x8 v = zero8;
      if (k < g.K && n < g.Npad) v = *(const bf16x8 *)(g.B + (long)k * g.sbk + n);
#pragma unroll
      for (int j = 0; j < 8; ++j) Bs[(nc + j) * kLdsPitch + kk] = v[j];
    }
    __syncthreads();
    bf16x8 a[2], b[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) a[i] = *(const bf16x8 *)&As[(wm * 32 + i * 16 + (l & 15)) * kLdsPitch + 8 * (l >> 4)];
#pragma unroll
    for (int j = 0; j < 2; ++j) b[j] = *(const bf16x8 *)&Bs[(wn * 32 + j * 16 + (l & 15)) * kLdsPitch + 8 * (l >> 4)];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    __syncthreads();
  }
  float *Cf = g.Cf;
  if (EPI == EPI_STORE) Cf += (long)blockIdx.z * g.split_stride;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = n0 + wn * 32 + j * 16 + (l & 15);
      if (n >= g.N) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm * 32 + i * 16 + 4 * (l >> 4) + r;
        if (m >= g.M) continue;
        const float v = acc[i][j][r];
        if (EPI == EPI_BIAS_GELU) {
          const float zv = v + g.bias[n];
          Cf[(long)m * g.ldc + n] = zv;
          g.Cb[(long)m * g.ldcb + n] = (bf16_t)gelu(zv);
        } else if (EPI == EPI_BIAS) {
          Cf[(long)m * g.ldc + n] = v + g.bias[n];
        } else if (EPI == EPI_GELU_GRAD) {
          g.Cb[(long)m * g.ldcb + n] = (bf16_t)(v * gelu_grad(g.Z[(long)m * g.ldz + n]));
        } else {
          Cf[(long)m * g.ldc + n] = v;
        }
      }
    }
}

__device__ __forceinline__ float wave_sum_f(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__global__ __launch_bounds__(256) void k_to_bf16(size_t n, const float *in, bf16_t *out) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) out[i] = (bf16_t)in[i];
}

__global__ __launch_bounds__(256) void k_loss_grad(int B, int n_out, int ld, const float *y, const float *t,
                                                   const float *w, bf16_t *dy, float *part) {
  __shared__ float red[4];
  float s = 0.f;
  const size_t n = (size_t)B * ld;
  const float scale = 2.f / (float)B;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const int o = (int)(i % ld);
    float d = 0.f;
    if (o < n_out) {
      const float r = y[i] - t[i];
      s += w[o] * r * r;
      d = scale * w[o] * r;
    }
    dy[i] = (bf16_t)d;
  }
  s = wave_sum_f(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// column sums in two fixed-order stages: block (x, r) sums rows [r rc, (r+1) rc)
// of 64 columns (4 row groups) into part[r N + n]; k_colsum_fold adds the R
// row chunks in order
__global__ __launch_bounds__(256) void k_colsum(int M, int N, int ld, int rc, const bf16_t *dz, float *part) {
  __shared__ float red[4][64];
  const int c = threadIdx.x & 63, rg = threadIdx.x >> 6, n = blockIdx.x * 64 + c;
  const int m0 = blockIdx.y * rc, m1 = min(M, m0 + rc);
  float s = 0.f;
  if (n < N)
    for (int m = m0 + rg; m < m1; m += 4) s += (float)dz[(long)m * ld + n];
  red[rg][c] = s;
  __syncthreads();
  if (rg == 0 && n < N) part[(long)blockIdx.y * N + n] = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
}
// 64 columns per workgroup, 4 row groups over the R chunks, fixed order
__global__ __launch_bounds__(256) void k_colsum_fold(int R, int N, const float *part, float *db) {
  __shared__ float red[4][64];
  const int c = threadIdx.x & 63, rg = threadIdx.x >> 6, n = blockIdx.x * 64 + c;
  float s = 0.f;
  if (n < N)
    for (int r = rg; r < R; r += 4) s += part[(long)r * N + n];
  red[rg][c] = s;
  __syncthreads();
  if (rg == 0 && n < N) db[n] = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
}

// only the R x C logical entries are written: the padding of out keeps its zeros
__global__ __launch_bounds__(256) void k_split_reduce(int S, int R, int C, int ld, long stride, const float *part,
                                                      float *out) {
  const size_t n = (size_t)R * C;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const size_t e = (i / C) * ld + i % C;
    float s = 0.f;
    for (int z = 0; z < S; ++z) s += part[(long)z * stride + e];
    out[e] = s;
  }
}

__global__ __launch_bounds__(256) void k_adam(size_t n, float *p, const float *g, float *m, float *v, bf16_t *pb,
                                              float lr, float b1, float b2, float eps, float c1, float c2) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    if (pb) pb[i] = (bf16_t)pi;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_gather(int n, int ld, const int *idx, const T *src, T *dst) {
  const size_t tot = (size_t)n * ld;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < tot; i += (size_t)gridDim.x * 256) {
    const size_t r = i / ld, c = i % ld;
    dst[i] = src[(size_t)idx[r] * ld + c];
  }
}

// ---------------------------------------------------------------------------
// Row-block kernels (widths 64, 128, 256).  A layer at a batch of 2 048 is 0.3
// GFLOP, a fraction of a microsecond of matrix-core time, so separate GEMM,
// loss, column-sum and optimizer launches were all launch and load latency (42
// launches, 290 us a step).  Rows of the batch are independent through the
// forward pass, the loss and the input gradients: k_mlp_rows takes 16 of them
// through all layers and back with activations, pre-activations (fp32) and
// gradients in LDS, and reads the weights as MFMA fragments straight from
// L2 (16 bytes a lane, from W forward and from a transposed copy backward).  It
// leaves activations and gradients feature-major, so that k_mlp_wgrad reads
// both operands of dW = dZ^T A as fragments too, all layers in one launch; k_mlp_update
// folds the batch splits and applies Adam.  A step of 12 -> 256 x 4 -> 641 at
// 2 048 rows: 290 us -> 73 (rows 48, bound by the instructions of 128
// workgroups' GELUs and by load latency; weight gradients 17; update 8); a
// forward pass of 1 000 rows 26 us.
// ---------------------------------------------------------------------------
constexpr int kRows = 16, kRowThreads = 1024, kRowWaves = kRowThreads / 64;

// KS k-steps of one weight row per lane (w: the lane's row at its 8-element
// offset).  No lane is masked, a masked load is a branch: rows are clamped by
// the caller, and steps past a row's end read on (the copies are allocated
// with a layer width to spare) and are used in no product.
template <int KS>
__device__ __forceinline__ void mlp_load(bf16x8 (&x)[KS], const bf16_t *w) {
#pragma unroll
  for (int i = 0; i < KS; ++i) x[i] = *(const bf16x8 *)(w + 32 * i);
}
// c += A(16 x 32 KS) x^T, a: the lane's LDS row at its 8-element offset
template <int KS>
__device__ __forceinline__ void mlp_mma(const bf16_t *a, const bf16x8 (&x)[KS], f32x4 &c) {
#pragma unroll
  for (int i = 0; i < KS; ++i)
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8 *)(a + 32 * i), x[i], c, 0, 0, 0);
}
template <int KS>
__device__ __forceinline__ void mlp_take(bf16x8 (&x)[KS], const bf16x8 (&y)[KS]) {
#pragma unroll
  for (int i = 0; i < KS; ++i) x[i] = y[i];
}

// columns f < nf of a 16-row LDS matrix to feature-major memory (row pitch
// Bp), and their sums over the rows to db (when not null)
__device__ __forceinline__ void mlp_store_t(const bf16_t *buf, int pitch, int nf, bf16_t *dst, long Bp, int b0,
                                            float *db) {
  for (int t = threadIdx.x; t < 2 * nf; t += kRowThreads) {
    const int f = t >> 1, h = t & 1;
    bf16x8 v;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[i] = buf[(8 * h + i) * pitch + f];
      s += (float)v[i];
    }
    *(bf16x8 *)(dst + (long)f * Bp + b0 + 8 * h) = v;
    if (db) {
      s += __shfl_xor(s, 1, 64);
      if (h == 0) db[f] = s;
    }
  }
}

template <int KS, bool TRAIN>
__global__ __launch_bounds__(kRowThreads) void k_mlp_rows(MlpRows P) {
  constexpr int WD = 32 * KS, PA = WD + 8, ZP = WD + 4, NT = WD / 16;
  extern __shared__ __attribute__((aligned(16))) char sm[];
  __shared__ float red[kRowWaves];
  bf16_t *a0 = (bf16_t *)sm, *a1 = a0 + kRows * PA;
  float *gg = (float *)(a1 + kRows * PA);                    // gelu'(Z): depth x 16 x ZP (TRAIN)
  const int PO = P.out32 + 8, nbias = P.depth * WD + P.n_out;
  // biases, and (TRAIN) loss weights and the output gradients, 16 x PO
  float *sb = TRAIN ? gg + (long)P.depth * kRows * ZP : gg, *slw = sb + nbias;
  bf16_t *dy = (bf16_t *)(slw + (P.n_out + nbias + 7) / 8 * 8 - nbias);
  const int b0 = blockIdx.x * kRows;
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6, lc = l & 15, lk = 8 * (l >> 4);
  // wave w owns 16 columns of a hidden layer (waves beyond NT idle there);
  // the weights of the next product are loaded before the current one is used
  const bool own = w < NT;
  const int n = 16 * w + lc, nh = 16 * (w % NT) + lc;
  bf16x8 x[KS], nx[KS] = {};
  // (past the inputs a row would read on into other neurons' weights, of which an
  // infinite one times a zero of A is not zero: these lanes read the zeros behind
  // the last row.  Zeroing the registers instead cost 1 to 2 of a forward pass's
  // 26 us, a copy of the weights in rows of a layer width 2.5)
  const bf16_t *w0 = P.W[0] + (long)nh * P.in_pad + lk, *none = P.W[0] + (long)WD * P.in_pad;
#pragma unroll
  for (int i = 0; i < KS; ++i) x[i] = *(const bf16x8 *)(lk + 32 * i < P.in_pad ? w0 + 32 * i : none);
  // the sample of each of this lane's four output rows (the last row repeated
  // past the batch; its results are dropped), and everything else a wave will
  // want from memory one value at a time: each would be a full latency later
  long sample[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int b = min(b0 + 4 * (l >> 4) + r, P.B - 1);
    sample[r] = P.idx ? P.idx[b] : b;
  }
  float tv[4] = {};
  if (TRAIN)
#pragma unroll
    for (int r = 0; r < 4; ++r) tv[r] = P.T[sample[r] * P.out_pad + min(n, P.n_out - 1)];
  for (int y = 0; y <= P.depth; ++y)
    for (int e = threadIdx.x; e < (y < P.depth ? WD : P.n_out); e += kRowThreads) sb[y * WD + e] = P.bias[y][e];
  if (TRAIN)
    for (int e = threadIdx.x; e < P.n_out; e += kRowThreads) slw[e] = P.lw[e];
  for (int e = threadIdx.x; e < kRows * PA; e += kRowThreads) {
    const int r = e / PA, c = e - r * PA, b = b0 + r;
    bf16_t v = (bf16_t)0.f;
    if (b < P.B && c < P.in_pad) v = P.X[(long)(P.idx ? P.idx[b] : b) * P.in_pad + c];
    a0[e] = v;
  }
  if (TRAIN)
    for (int e = threadIdx.x; e < kRows * PO; e += kRowThreads) dy[e] = (bf16_t)0.f;
  __syncthreads();
  if (TRAIN) mlp_store_t(a0, PA, P.n_in, P.actT, P.Bp, b0, nullptr);
  for (int y = 0; y < P.depth; ++y) {
    const bf16_t *src = y & 1 ? a1 : a0;
    bf16_t *dst = y & 1 ? a0 : a1;
    const bool hid = y + 1 < P.depth;  // else the first output tile of the wave follows
    mlp_load(nx, P.W[y + 1] + (long)(hid ? nh : min(n, P.n_out - 1)) * WD + lk);
    if (own) {
      f32x4 c = {0.f, 0.f, 0.f, 0.f};
      mlp_mma(src + lc * PA + lk, x, c);
      const float bias = sb[y * WD + n];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * (l >> 4) + r;
        const float z = c[r] + bias, h = 0.5f * (1.f + erff(z * 0.70710678118654752f));
        dst[row * PA + n] = (bf16_t)(z * h);
        if (TRAIN) gg[((long)y * kRows + row) * ZP + n] = h + z * 0.39894228040143268f * expf(-0.5f * z * z);
      }
    }
    mlp_take(x, nx);
    __syncthreads();
    if (TRAIN) mlp_store_t(dst, PA, WD, P.actT + (long)(P.n_in + y * WD) * P.Bp, P.Bp, b0, nullptr);
  }
  // output layer: tiles w, w + kRowWaves, ...
  float loss = 0.f;
  {
    const bf16_t *a = (P.depth & 1 ? a1 : a0) + lc * PA + lk;
    for (int m = n; m - lc < P.n_out; m += 16 * kRowWaves) {
      const int m2 = m + 16 * kRowWaves, mc = min(m, P.n_out - 1);
      mlp_load(nx, P.W[P.depth] + (long)min(m2, P.n_out - 1) * WD + lk);
      float tn[4] = {};
      if (TRAIN)
#pragma unroll
        for (int r = 0; r < 4; ++r) tn[r] = P.T[sample[r] * P.out_pad + min(m2, P.n_out - 1)];
      f32x4 c = {0.f, 0.f, 0.f, 0.f};
      mlp_mma(a, x, c);
      mlp_take(x, nx);
      const float bias = sb[P.depth * WD + mc], wo = TRAIN ? slw[mc] : 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * (l >> 4) + r, b = b0 + row;
        const bool in = b < P.B && m < P.n_out;
        const float yv = c[r] + bias;
        if (!TRAIN) {
          if (in) P.y[(long)b * P.out_pad + m] = yv;
        } else {
          const float rr = in ? yv - tv[r] : 0.f;
          loss += wo * rr * rr;
          if (m < P.n_out) dy[row * PO + m] = (bf16_t)(P.scale * wo * rr);
          tv[r] = tn[r];
        }
      }
    }
  }
  if (!TRAIN) return;
  const int ko = P.out32;  // row pitch of the transposed output weights
  mlp_load(x, P.Wt[P.depth] + (long)nh * ko + lk);
  loss = wave_sum_f(loss);
  if (l == 0) red[w] = loss;
  __syncthreads();
  if (threadIdx.x == 0) {
    float sum = 0.f;
    for (int i = 0; i < kRowWaves; ++i) sum += red[i];
    P.loss[b0 / kRows] = sum;
  }
  float *db = P.db + (long)(b0 / kRows) * (P.depth * WD + P.n_out);
  mlp_store_t(dy, PO, P.n_out, P.dzT + (long)P.depth * WD * P.Bp, P.Bp, b0, db + P.depth * WD);
  // dZ_{y-1} = (dZ_y W_y) gelu'(Z_{y-1}); the activation buffers are free again
  const bf16_t *src = dy;
  int spitch = PO;
  for (int y = P.depth; y >= 1; --y) {
    bf16_t *dst = (P.depth - y) & 1 ? a1 : a0;
    const bf16_t *a = src + lc * spitch + lk;
    f32x4 c = {0.f, 0.f, 0.f, 0.f};
    if (y == P.depth) {
      // the output layer's k range in groups of KS steps (steps past its end
      // meet zero weights; their LDS reads stay inside the row)
      for (int k = WD; k < ko; k += WD) {
        mlp_load(nx, P.Wt[y] + (long)nh * ko + lk + k);
        mlp_mma(a + k - WD, x, c);
        mlp_take(x, nx);
      }
      const int kl = (ko - 1) / WD * WD;
      if (y > 1) mlp_load(nx, P.Wt[y - 1] + (long)nh * WD + lk);
#pragma unroll
      for (int i = 0; i < KS; ++i)
        if (kl + 32 * i < ko)
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8 *)(a + kl + 32 * i), x[i], c, 0, 0, 0);
    } else {
      if (y > 1) mlp_load(nx, P.Wt[y - 1] + (long)nh * WD + lk);
      mlp_mma(a, x, c);
    }
    mlp_take(x, nx);
    if (own) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * (l >> 4) + r;
        dst[row * PA + n] = (bf16_t)(c[r] * gg[((long)(y - 1) * kRows + row) * ZP + n]);
      }
    }
    __syncthreads();
    mlp_store_t(dst, PA, WD, P.dzT + (long)(y - 1) * WD * P.Bp, P.Bp, b0, db + (y - 1) * WD);
    src = dst;
    spitch = PA;
  }
}

// dW of every layer, one 32 x 64 tile and one split of the batch per wave;
// both operands are read feature-major (K, the batch, contiguous)
__global__ __launch_bounds__(256) void k_mlp_wgrad(MlpShape S, int ntile, int nsplit, int nk, long Bp,
                                                   const bf16_t *__restrict__ actT, const bf16_t *__restrict__ dzT,
                                                   float *__restrict__ part) {
  const int l = threadIdx.x & 63, lc = l & 15, lk = 8 * (l >> 4);
  const int tile = (int)(blockIdx.x / nsplit) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sp = (int)(blockIdx.x % nsplit);
  if (tile >= ntile) return;
  int y = 0;
  while (tile >= S.t0[y + 1]) ++y;
  const int in = S.in[y], out = S.out[y], ntn = (in + 63) / 64, q = tile - S.t0[y];
  const int m0 = 32 * (q / ntn), n0 = 64 * (q % ntn);
  const int per = (nk + nsplit - 1) / nsplit, k0 = sp * per, k1 = min(nk, k0 + per);
  const bf16_t *A[2], *Bv[4];
  bool ma[2], nb[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = m0 + 16 * i + lc;
    ma[i] = m < out;
    A[i] = dzT + (S.zoff[y] + (ma[i] ? m : 0)) * Bp + lk;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + 16 * j + lc;
    nb[j] = n < in;
    Bv[j] = actT + (S.aoff[y] + (nb[j] ? n : 0)) * Bp + lk;
  }
  f32x4 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // four k-steps' fragments are loaded together, 24 loads in flight a wave: a
  // round takes ~3 us (sixteen rows a load, written by other XCDs)
  constexpr int KB = 4;
  for (int k = k0; k < k1; k += KB) {
    bf16x8 a[KB][2], b[KB][4];
#pragma unroll
    for (int q = 0; q < KB; ++q) {
      const long at = 32L * min(k + q, k1 - 1);
#pragma unroll
      for (int i = 0; i < 2; ++i) a[q][i] = *(const bf16x8 *)(A[i] + at);
#pragma unroll
      for (int j = 0; j < 4; ++j) b[q][j] = *(const bf16x8 *)(Bv[j] + at);
    }
#pragma unroll
    for (int q = 0; q < KB; ++q)
      if (k + q < k1)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q][i], b[q][j], acc[i][j], 0, 0, 0);
  }
  // (rows and columns past the layer read row 0 and are not stored)
  float *C = part + (long)sp * S.nw + S.poff[y];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + 16 * j + lc;
      if (n >= in) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + 16 * i + 4 * (l >> 4) + r;
        if (m < out) C[(long)m * in + n] = acc[i][j][r];
      }
    }
}

__device__ __forceinline__ float adam_one(float p, float g, float &m, float &v, const MlpAdam &h) {
  m = h.b1 * m + (1.f - h.b1) * g;
  v = h.b2 * v + (1.f - h.b2) * g * g;
  return p - h.lr * (m / h.c1) / (sqrtf(v / h.c2) + h.eps);
}

// gradients folded over the batch splits (weights) and row blocks (biases, one
// wave each), both in a fixed order, then one Adam step on the fp32 masters
// and the two bf16 copies (ADAM), or the gradients stored
// (grid y: the layer, uniform, so that the tables are scalar loads)
template <bool ADAM>
__global__ __launch_bounds__(256) void k_mlp_update(MlpShape S, MlpParams Q, MlpAdam h, int nsplit, int nrow,
                                                    const float *part, const float *db) {
  const int y = blockIdx.y, in = S.in[y], out = S.out[y], wblk = (out * in + 255) / 256;
  if ((int)blockIdx.x < wblk) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= out * in) return;
    const int o = e / in, i = e - o * in;
    float g = 0.f;
    for (int z = 0; z < nsplit; ++z) g += part[(long)z * S.nw + S.poff[y] + e];
    const long at = (long)o * Q.in_pad[y] + i;
    if (!ADAM) {
      Q.gW[y][at] = g;
      return;
    }
    float m = Q.mW[y][at], v = Q.vW[y][at];
    const float x = adam_one(Q.W[y][at], g, m, v, h);
    Q.mW[y][at] = m;
    Q.vW[y][at] = v;
    Q.W[y][at] = x;
    Q.Wb[y][at] = (bf16_t)x;
    Q.Wt[y][(long)i * Q.out32[y] + o] = (bf16_t)x;
    return;
  }
  const int o = ((int)blockIdx.x - wblk) * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63;
  if (o >= out) return;
  const long nbias = S.zoff[S.nl];
  float g = 0.f;
  for (int r = l; r < nrow; r += 64) g += db[r * nbias + S.zoff[y] + o];
  g = wave_sum_f(g);
  if (l) return;
  if (!ADAM) {
    Q.gb[y][o] = g;
    return;
  }
  float m = Q.mb[y][o], v = Q.vb[y][o];
  Q.b[y][o] = adam_one(Q.b[y][o], g, m, v, h);
  Q.mb[y][o] = m;
  Q.vb[y][o] = v;
}

// the bf16 copies of one layer's weights: row-major, and transposed with a
// pitch of 32-element groups (padding zero from the allocation)
__global__ __launch_bounds__(256) void k_mlp_copies(int out, int in, int in_pad, int out32, const float *W, bf16_t *Wb,
                                                    bf16_t *Wt) {
  const size_t n = (size_t)out * in;
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (size_t)gridDim.x * 256) {
    const int o = (int)(e / in), i = (int)(e - (size_t)o * in);
    const bf16_t v = (bf16_t)W[(size_t)o * in_pad + i];
    Wb[(size_t)o * in_pad + i] = v;
    Wt[(size_t)i * out32 + o] = v;
  }
}

int grid1(size_t n) { return (int)std::max<size_t>(1, std::min<size_t>((n + 255) / 256, 4096)); }

}  // namespace

void mlp_gemm(const GemmArgs &g, int epi, hipStream_t s) {
  if (g.M <= 0 || g.N <= 0) return;
  const bool akc = g.sak == 1, bkc = g.sbk == 1;
  if (!akc && g.sam != 1) fail(ED_ERR_INTERNAL, "mlp_gemm: A has no contiguous axis");
  if (!bkc && g.sbn != 1) fail(ED_ERR_INTERNAL, "mlp_gemm: B has no contiguous axis");
  if (g.Kpad % 8 || (!akc && g.Mpad % 8) || (!bkc && g.Npad % 8) || g.Kpad < g.K)
    fail(ED_ERR_INTERNAL, "mlp_gemm: padded extents must be multiples of 8");
  if ((akc && g.sam % 8) || (!akc && g.sak % 8) || (bkc && g.sbn % 8) || (!bkc && g.sbk % 8) ||
      (reinterpret_cast<uintptr_t>(g.A) & 15) || (reinterpret_cast<uintptr_t>(g.B) & 15))
    fail(ED_ERR_INTERNAL, "mlp_gemm: operands must be 16-byte aligned rows");
  if (epi != EPI_STORE && g.ksplit != 1) fail(ED_ERR_INTERNAL, "mlp_gemm: split k only for plain stores");
  const dim3 grid((g.M + kBM - 1) / kBM, (g.N + kBN - 1) / kBN, std::max(1, g.ksplit));
#define ED_GEMM(E)                                                                                      \
  do {                                                                                                  \
    if (akc && bkc) hipLaunchKernelGGL((k_gemm<E, true, true>), grid, dim3(256), 0, s, g);              \
    else if (akc) hipLaunchKernelGGL((k_gemm<E, true, false>), grid, dim3(256), 0, s, g);               \
    else if (bkc) hipLaunchKernelGGL((k_gemm<E, false, true>), grid, dim3(256), 0, s, g);               \
    else hipLaunchKernelGGL((k_gemm<E, false, false>), grid, dim3(256), 0, s, g);                       \
  } while (0)
  switch (epi) {
    case EPI_BIAS_GELU: ED_GEMM(EPI_BIAS_GELU); break;
    case EPI_BIAS: ED_GEMM(EPI_BIAS); break;
    case EPI_GELU_GRAD: ED_GEMM(EPI_GELU_GRAD); break;
    default: ED_GEMM(EPI_STORE); break;
  }
#undef ED_GEMM
  ED_HIP(hipGetLastError());
}

void mlp_to_bf16(size_t n, const float *in, bf16_t *out, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_to_bf16, dim3(grid1(n)), dim3(256), 0, s, n, in, out);
  ED_HIP(hipGetLastError());
}

int mlp_loss_grad(int B, int n_out, int ld, const float *y, const float *t, const float *w, bf16_t *dy,
                  float *partials, hipStream_t s) {
  const int g = std::min(grid1((size_t)B * ld), 1024);
  hipLaunchKernelGGL(k_loss_grad, dim3(g), dim3(256), 0, s, B, n_out, ld, y, t, w, dy, partials);
  ED_HIP(hipGetLastError());
  return g;
}

int mlp_colsum_chunks(int M) { return std::max(1, std::min(64, (M + 63) / 64)); }

void mlp_colsum(int M, int N, int ld, const bf16_t *dz, float *db, float *part, hipStream_t s) {
  if (N <= 0) return;
  const int R = mlp_colsum_chunks(M);
  const int rc = (M + R - 1) / R;
  hipLaunchKernelGGL(k_colsum, dim3((N + 63) / 64, R), dim3(256), 0, s, M, N, ld, rc, dz, part);
  ED_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_colsum_fold, dim3((N + 63) / 64), dim3(256), 0, s, R, N, (const float *)part, db);
  ED_HIP(hipGetLastError());
}

void mlp_split_reduce(int S, int R, int C, int ld, long stride, const float *part, float *out, hipStream_t s) {
  if (R <= 0 || C <= 0) return;
  hipLaunchKernelGGL(k_split_reduce, dim3(grid1((size_t)R * C)), dim3(256), 0, s, S, R, C, ld, stride, part, out);
  ED_HIP(hipGetLastError());
}

void mlp_adam(size_t n, float *p, const float *g, float *m, float *v, bf16_t *pb, float lr, float b1, float b2,
              float eps, float c1, float c2, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_adam, dim3(grid1(n)), dim3(256), 0, s, n, p, g, m, v, pb, lr, b1, b2, eps, c1, c2);
  ED_HIP(hipGetLastError());
}

void mlp_gather_bf16(int n, int ld, const int *idx, const bf16_t *src, bf16_t *dst, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_gather<bf16_t>, dim3(grid1((size_t)n * ld)), dim3(256), 0, s, n, ld, idx, src, dst);
  ED_HIP(hipGetLastError());
}

void mlp_gather_f32(int n, int ld, const int *idx, const float *src, float *dst, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_gather<float>, dim3(grid1((size_t)n * ld)), dim3(256), 0, s, n, ld, idx, src, dst);
  ED_HIP(hipGetLastError());
}

size_t mlp_rows_lds(int width, int depth, int n_out, bool train) {
  const size_t act = 2 * (size_t)kRows * (width + 8) * sizeof(bf16_t), nbias = (size_t)depth * width + n_out;
  const int out32 = (n_out + 31) / 32 * 32;
  if (!train) return act + (nbias + 8) * sizeof(float);
  return act + (size_t)depth * kRows * (width + 4) * sizeof(float) + (n_out + nbias + 7) / 8 * 8 * sizeof(float) +
         (size_t)kRows * (out32 + 8) * sizeof(bf16_t);
}

int mlp_rows(const MlpRows &P, int width, bool train, hipStream_t s) {
  if (P.B <= 0) return 0;
  const size_t lds = mlp_rows_lds(width, P.depth, P.n_out, train);
  if (lds > kMlpRowsLds || P.depth > kMlpLayers - 1 || P.in_pad > width || P.Bp % 32 || P.Bp < P.B ||
      (P.in_pad % 8) || (reinterpret_cast<uintptr_t>(P.actT) & 15) || (reinterpret_cast<uintptr_t>(P.dzT) & 15))
    fail(ED_ERR_INTERNAL, "mlp_rows: network outside the row-block kernel's range");
  // a training step's blocks cover the padded batch: the padding of the
  // feature-major matrices is written too (gradients zero)
  const int nb = train ? (P.B + 31) / 32 * 2 : (P.B + kRows - 1) / kRows;
#define ED_ROWS(KS)                                                                                          \
  do {                                                                                                       \
    auto kern = train ? k_mlp_rows<KS, true> : k_mlp_rows<KS, false>;                                        \
    if (lds > 64 * 1024)                                                                                     \
      ED_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),                                       \
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));                     \
    hipLaunchKernelGGL(kern, dim3(nb), dim3(kRowThreads), lds, s, P);                                        \
  } while (0)
  if (width == 64) ED_ROWS(2);
  else if (width == 128) ED_ROWS(4);
  else if (width == 256) ED_ROWS(8);
  else fail(ED_ERR_INTERNAL, "mlp_rows: width");
#undef ED_ROWS
  ED_HIP(hipGetLastError());
  return nb;
}

void mlp_wgrad(const MlpShape &S, int nsplit, int nk, long Bp, const bf16_t *actT, const bf16_t *dzT, float *part,
               hipStream_t s) {
  const int nt = S.t0[S.nl];
  hipLaunchKernelGGL(k_mlp_wgrad, dim3((nt + 3) / 4 * nsplit), dim3(256), 0, s, S, nt, nsplit, nk, Bp, actT, dzT, part);
  ED_HIP(hipGetLastError());
}

void mlp_update(const MlpShape &S, const MlpParams &Q, const MlpAdam *h, int nsplit, int nrow, const float *part,
                const float *db, hipStream_t s) {
  int nx = 1;
  for (int y = 0; y < S.nl; ++y) nx = std::max(nx, (S.out[y] * S.in[y] + 255) / 256 + (S.out[y] + 3) / 4);
  const dim3 grid((unsigned)nx, (unsigned)S.nl);
  if (h)
    hipLaunchKernelGGL((k_mlp_update<true>), grid, dim3(256), 0, s, S, Q, *h, nsplit, nrow, part, db);
  else
    hipLaunchKernelGGL((k_mlp_update<false>), grid, dim3(256), 0, s, S, Q, MlpAdam(), nsplit, nrow, part, db);
  ED_HIP(hipGetLastError());
}

void mlp_copies(int out, int in, int in_pad, int out32, const float *W, bf16_t *Wb, bf16_t *Wt, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_copies, dim3(grid1((size_t)out * in)), dim3(256), 0, s, out, in, in_pad, out32, W, Wb, Wt);
  ED_HIP(hipGetLastError());
}

double mlp_fold(const float *partials, int n) {
  std::vector<double> w(partials, partials + std::max(n, 0));
  size_t k = w.size();
  while (k > 1) {
    const size_t half = (k + 1) / 2;
    for (size_t i = 0; i + half < k; ++i) w[i] += w[i + half];
    k = half;
  }
  return k ? w[0] : 0.0;
}

}  // namespace ed
