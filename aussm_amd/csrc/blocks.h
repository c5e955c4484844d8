// Kernels of the blocks around the scans: depthwise causal convolution on channel rows, and the root-mean-square norm.
//
// Inside a block every activation is kept as channel rows (b, d, l), the scans' layout: the input projection writes it
// (gemm.h takes (b, l, d) rows on one side and channel rows on the other), the output projection reads it, and no
// tensor is transposed on the way.
#pragma once
#include "block_args.h"
#include "scan_common.h"

namespace aussm {

// ---- y[b,i,l] = bias[i] + sum_k w[i,k] x[b,i,l - (K-1) + k]   (x = 0 before the sequence), ai-modules/wavesAI/model/
// aussm.py:762, :863, along rows of L elements.  Thread = four consecutive steps of one row; the previous K - 1
// elements come from the cache.  Memory bound: 8 bytes per element (12 with the second output silu(y)).
template <int K>
__global__ __launch_bounds__(256) void conv_rows_fwd_kernel(const ConvRowsArgs p) {
  const int nq = (p.L + 3) / 4;
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t row = idx / nq;
  if (row >= (size_t)p.B * p.D) return;
  const int l0 = 4 * (int)(idx - row * nq), i = (int)(row % p.D), b = (int)(row / p.D);
  const float* __restrict__ x = p.x + (size_t)b * p.xs_b + (size_t)i * p.L;
  const int kk = K ? K : p.K;
  const float* __restrict__ w = p.w + (size_t)i * kk;
  float acc[4];
#pragma unroll
  for (int a = 0; a < 4; ++a) acc[a] = p.bias ? p.bias[i] : 0.0f;
#pragma unroll
  for (int k = 0; k < (K ? K : 8); ++k) {
    if (K == 0 && k >= kk) break;
    const float wk = w[k];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int l = l0 + a - (kk - 1) + k;
      const float v = (l >= 0 && l < p.L) ? x[l] : 0.0f;
      acc[a] = fmaf(wk, v, acc[a]);
    }
  }
  const size_t o = row * p.L + l0;
  const int left = p.L - l0;
  const bool vec = left >= 4 && (p.L & 3) == 0;           // (rows of y start on 16 bytes)
  store4(p.y, o, acc, vec, left);
}

// dx[b,i,l] = sum_k w[i,k] dy[b,i,l + (K-1) - k];  dw[i,k] += sum dy[l] x[l - (K-1) + k];  dbias[i] += sum dy.
// One wavefront per (row, piece of CONV_PIECE steps): dx and the weight sums in one pass over dy and x.
template <int K>
__global__ __launch_bounds__(256) void conv_rows_bwd_kernel(const ConvRowsArgs p) {
  const int lane = threadIdx.x & 63;
  const size_t row = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= (size_t)p.B * p.D) return;                   // (whole wavefronts)
  const int i = (int)(row % p.D), b = (int)(row / p.D);
  const float* __restrict__ x = p.x + (size_t)b * p.xs_b + (size_t)i * p.L;
  const float* __restrict__ dy = p.dy + row * p.L;
  float* __restrict__ dx = p.dx + (size_t)b * p.dxs_b + (size_t)i * p.L;
  const int kk = K ? K : p.K;
  float w[K ? K : 8], acc[K ? K : 8], accb = 0.0f;
#pragma unroll
  for (int k = 0; k < (K ? K : 8); ++k) { w[k] = k < kk ? p.w[(size_t)i * kk + k] : 0.0f; acc[k] = 0.0f; }
  const int lb = blockIdx.y * CONV_PIECE, le = lb + CONV_PIECE < p.L ? lb + CONV_PIECE : p.L;
  for (int l = lb + lane; l < le; l += 64) {
    const float g0 = dy[l];
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < (K ? K : 8); ++k) {
      if (K == 0 && k >= kk) break;
      const int lt = l + (kk - 1) - k, ls = l - (kk - 1) + k;
      const float g = lt < p.L ? dy[lt] : 0.0f;
      s = fmaf(w[k], g, s);
      acc[k] = fmaf(g0, ls >= 0 ? x[ls] : 0.0f, acc[k]);
    }
    accb += g0;
    dx[l] = s;
  }
#pragma unroll
  for (int k = 0; k < (K ? K : 8); ++k) {
    float v = acc[k];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane == 0 && k < kk) atomicAdd(p.dw + (size_t)i * kk + k, v);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) accb += __shfl_xor(accb, o, 64);
  if (lane == 0 && p.dbias) atomicAdd(p.dbias + i, accb);
}

// ---- RMSNorm over rows of d elements: y = x rstd w, rstd = rsqrt(mean(x^2) + eps)  (aussm.py:905-916).
// One wavefront per row; NJ: elements per lane (d <= 64 NJ).
template <int NJ>
__global__ __launch_bounds__(256) void rms_norm_fwd_kernel(const NormArgs p) {
  const int lane = threadIdx.x & 63;
  const size_t row = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= p.rows) return;
  const float* __restrict__ x = p.x + row * p.d;
  float v[NJ], s = 0.0f;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    v[j] = lane + 64 * j < p.d ? x[lane + 64 * j] : 0.0f;
    s = fmaf(v[j], v[j], s);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
  const float r = rsqrtf(s / (float)p.d + p.eps);
  float* __restrict__ y = p.y + row * p.d;
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    if (lane + 64 * j < p.d) y[lane + 64 * j] = v[j] * r * p.w[lane + 64 * j];
  if (lane == 0 && p.rstd) p.rstd[row] = r;
}

// g = dy w, xh = x rstd:  dx = rstd (g - xh mean(g xh)) (+ res),  dw += sum over rows dy xh.
// A workgroup of four wavefronts walks NORM_ROWS rows, a row per wavefront and turn; the sums for dw stay in registers
// until the end, meet in LDS and leave as one atomic per column and workgroup.
template <int NJ>
__global__ __launch_bounds__(256) void rms_norm_bwd_kernel(const NormArgs p) {
  __shared__ float s_w[4][NJ * 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t r0 = (size_t)blockIdx.x * NORM_ROWS;
  float wv[NJ], dwv[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) { wv[j] = lane + 64 * j < p.d ? p.w[lane + 64 * j] : 0.0f; dwv[j] = 0.0f; }
  for (int t = wave; t < NORM_ROWS; t += 4) {
    const size_t row = r0 + t;
    if (row >= p.rows) break;
    const float rs = p.rstd[row];
    float xh[NJ], g[NJ], s = 0.0f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const bool ok = lane + 64 * j < p.d;
      const float dy = ok ? p.dy[row * p.d + lane + 64 * j] : 0.0f;
      xh[j] = ok ? p.x[row * p.d + lane + 64 * j] * rs : 0.0f;
      g[j] = dy * wv[j];
      dwv[j] = fmaf(dy, xh[j], dwv[j]);
      s = fmaf(g[j], xh[j], s);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    s /= (float)p.d;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      if (lane + 64 * j < p.d) {
        const size_t o = row * p.d + lane + 64 * j;
        const float v = rs * fmaf(-xh[j], s, g[j]);
        p.dx[o] = p.res ? v + p.res[o] : v;
      }
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) s_w[wave][lane + 64 * j] = dwv[j];
  __syncthreads();
  for (int c = threadIdx.x; c < p.d; c += 256) atomicAdd(p.dw + c, s_w[0][c] + s_w[1][c] + s_w[2][c] + s_w[3][c]);
}

// ---- column sums: out[c] += scale sum over rows x[row, c] (bias gradients of linear layers on (rows, d) tensors)
__global__ __launch_bounds__(256) void col_sum_kernel(const float* __restrict__ x, float* __restrict__ out, size_t rows, int d, float scale) {
  __shared__ float s_red[4][64];
  const int dl = threadIdx.x & 63, wave = threadIdx.x >> 6, c = blockIdx.x * 64 + dl;
  const size_t r0 = (size_t)blockIdx.y * COLSUM_ROWS;
  float s = 0.0f;
  if (c < d)
    for (int t = wave; t < COLSUM_ROWS && r0 + t < rows; t += 4) s += x[(r0 + t) * d + c];
  s_red[wave][dl] = s;
  __syncthreads();
  if (wave == 0 && c < d) atomicAdd(out + c, scale * (s_red[0][dl] + s_red[1][dl] + s_red[2][dl] + s_red[3][dl]));
}

// ---- row sums: out[row % d] += scale sum_l x[row, l] (bias gradients on channel rows), one wavefront per row
__global__ __launch_bounds__(256) void row_sum_kernel(const float* __restrict__ x, float* __restrict__ out, size_t rows, int d, int L, float scale) {
  const int lane = threadIdx.x & 63;
  const size_t row = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  float s = 0.0f;
  for (int l = lane; l < L; l += 64) s += x[row * L + l];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
  if (lane == 0) atomicAdd(out + row % d, scale * s);
}

// ---- A = -exp(A_log), and on the way back dA_log = dA A
__global__ __launch_bounds__(256) void neg_exp_kernel(const float* __restrict__ a_log, const float* __restrict__ dA, float* __restrict__ out, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float A = -expf(a_log[i]);
  out[i] = dA ? dA[i] * A : A;
}

}  // namespace aussm
