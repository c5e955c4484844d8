// Kernels of the blocks around the scans: depthwise causal convolution on channel rows, and the root-mean-square norm.
//
// Inside a block every activation is kept as channel rows (b, d, l), the scans' layout: the input projection writes it
// (gemm.h takes (b, l, d) rows on one side and channel rows on the other), the output projection reads it, and no
// tensor is transposed on the way.
#pragma once
#include "block_args.h"
#include "scan_common.h"

namespace aussm {

// quotient and remainder in 32 bits where they suffice (a 64-bit division is a hundred instructions)
__device__ __forceinline__ void divide(size_t a, unsigned d, size_t* q, unsigned* r) {
  if (a <= 0xffffffffu) {
    const unsigned v = (unsigned)a;
    *q = v / d;
    *r = v % d;
  } else {
    *q = a / d;
    *r = (unsigned)(a % d);
  }
}

// ---- y[b,i,l] = bias[i] + sum_k w[i,k] x[b,i,l - (K-1) + k]   (x = 0 before the sequence), ai-modules/wavesAI/model/
// aussm.py:762, :863, along rows of L elements.  Thread = four consecutive steps of one row.  Memory bound: 8 bytes per
// element.
// V4: K = 4, rows of whole, aligned groups of four: the four steps and the four before them are two 16-byte loads
// (32 x 256 and 32 x 512 rows of 720 steps, mean 37 -> 14 us; one load per tap and step and 64-bit divisions took the time).
template <int K, bool V4>
__global__ __launch_bounds__(256) void conv_rows_fwd_kernel(const ConvRowsArgs p) {
  const int nq = (p.L + 3) / 4;
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  size_t row, bq;
  unsigned lq, ii;
  divide(idx, (unsigned)nq, &row, &lq);
  if (row >= (size_t)p.B * p.D) return;
  divide(row, (unsigned)p.D, &bq, &ii);
  const int l0 = 4 * (int)lq, i = (int)ii;
  const float* __restrict__ x = p.x + bq * p.xs_b + (size_t)i * p.L;
  const int kk = K ? K : p.K;
  const float* __restrict__ w = p.w + (size_t)i * kk;
  float acc[4];
#pragma unroll
  for (int a = 0; a < 4; ++a) acc[a] = p.bias ? p.bias[i] : 0.0f;
  if constexpr (V4) {
    static_assert(K == 4, "three steps before the first one");
    const float4 c = *reinterpret_cast<const float4*>(x + l0);
    const float4 h = l0 ? *reinterpret_cast<const float4*>(x + l0 - 4) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float v[7] = {h.y, h.z, h.w, c.x, c.y, c.z, c.w};
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int a = 0; a < 4; ++a) acc[a] = fmaf(w[k], v[a + k], acc[a]);
  } else {
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
  }
  const size_t o = row * p.L + l0;
  const int left = p.L - l0;
  const bool vec = left >= 4 && (p.L & 3) == 0;           // (rows of y start on 16 bytes)
  store4(p.y, o, acc, vec, left);
}

// dx[b,i,l] = sum_k w[i,k] dy[b,i,l + (K-1) - k];  dw[i,k] += sum dy[l] x[l - (K-1) + k];  dbias[i] += sum dy.
// One wavefront per (row, piece of CONV_PIECE steps): dx and the weight sums in one pass over dy and x.
// V4: as in the forward kernel, four steps per lane and turn from four 16-byte loads (the same rows, mean 35 -> 27 us).
template <int K, bool V4>
__global__ __launch_bounds__(256) void conv_rows_bwd_kernel(const ConvRowsArgs p) {
  const int lane = threadIdx.x & 63;
  const size_t row = (size_t)blockIdx.x * 4 + wave_index();
  if (row >= (size_t)p.B * p.D) return;                   // (whole wavefronts)
  size_t bq;
  unsigned ii;
  divide(row, (unsigned)p.D, &bq, &ii);
  const int i = (int)ii;
  const float* __restrict__ x = p.x + bq * p.xs_b + (size_t)i * p.L;
  const float* __restrict__ dy = p.dy + row * p.L;
  float* __restrict__ dx = p.dx + bq * p.dxs_b + (size_t)i * p.L;
  const int kk = K ? K : p.K;
  float w[K ? K : 8], acc[K ? K : 8], accb = 0.0f;
#pragma unroll
  for (int k = 0; k < (K ? K : 8); ++k) { w[k] = k < kk ? p.w[(size_t)i * kk + k] : 0.0f; acc[k] = 0.0f; }
  const int lb = blockIdx.y * CONV_PIECE, le = lb + CONV_PIECE < p.L ? lb + CONV_PIECE : p.L;
  if constexpr (V4) {
    static_assert(K == 4, "three steps around");
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int l = lb + 4 * lane; l < le; l += 256) {
      const float4 g0 = *reinterpret_cast<const float4*>(dy + l);
      const float4 g1 = l + 4 < p.L ? *reinterpret_cast<const float4*>(dy + l + 4) : zero;
      const float4 x1 = *reinterpret_cast<const float4*>(x + l);
      const float4 x0 = l ? *reinterpret_cast<const float4*>(x + l - 4) : zero;
      const float g[7] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z}, v[7] = {x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
      float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          s[a] = fmaf(w[k], g[a + 3 - k], s[a]);
          acc[k] = fmaf(g[a], v[a + k], acc[k]);
        }
      accb += (g[0] + g[1]) + (g[2] + g[3]);
      *reinterpret_cast<float4*>(dx + l) = make_float4(s[0], s[1], s[2], s[3]);
    }
  } else {
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

// sum over the 64 lanes, in every lane
__device__ __forceinline__ float lanes_sum(float v) {
  v += dpp_perm<0x128>(v);    // row_ror:8
  v += dpp_perm<0x124>(v);
  v += dpp_perm<0x122>(v);
  v += dpp_perm<0x121>(v);
  return rows_sum(v);
}

// g = dy w, xh = x rstd:  dx = rstd (g - xh mean(g xh)) (+ res),  dw += sum over rows dy xh.
// A workgroup of four wavefronts walks NORM_ROWS rows, R rows per wavefront and turn, all their loads in flight together; the
// sums for dw stay in registers until the end, meet in LDS and leave as one atomic per column and workgroup.
// V4: rows of whole, aligned groups of four; lane = four neighbouring columns of every 256.
// Memory bound: 12 bytes per element (16 with the residual).  23040 rows of 256 with the residual: 27 us; 61 us with one
// row at a time and 4-byte loads.
template <int NJ, bool V4>
__global__ __launch_bounds__(256) void rms_norm_bwd_kernel(const NormArgs p) {
  static_assert(!V4 || NJ % 4 == 0, "four columns per lane");
  constexpr int R = NJ <= 4 ? 4 : NJ <= 8 ? 2 : 1;
  __shared__ float s_w[4][NJ * 64];
  const int lane = threadIdx.x & 63, wave = wave_index();
  const size_t r0 = (size_t)blockIdx.x * NORM_ROWS;
  auto col = [&](int j) { return V4 ? 256 * (j >> 2) + 4 * lane + (j & 3) : lane + 64 * j; };
  // a row's elements of this lane; columns past the end read as zero
  auto load = [&](const float* __restrict__ src, float (&v)[NJ]) {
    if constexpr (V4) {
#pragma unroll
      for (int j = 0; j < NJ; j += 4) {
        const float4 t = col(j) < p.d ? *reinterpret_cast<const float4*>(src + col(j)) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        v[j] = t.x; v[j + 1] = t.y; v[j + 2] = t.z; v[j + 3] = t.w;
      }
    } else {
#pragma unroll
      for (int j = 0; j < NJ; ++j) v[j] = col(j) < p.d ? src[col(j)] : 0.0f;
    }
  };
  float wv[NJ], dwv[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) { wv[j] = col(j) < p.d ? p.w[col(j)] : 0.0f; dwv[j] = 0.0f; }
  for (int t = wave * R; t < NORM_ROWS; t += 4 * R) {
    if (r0 + t >= p.rows) break;
    float dy[R][NJ], x[R][NJ], res[R][NJ], rs[R], s[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      // (rows past the last one repeat it and leave neither results nor sums)
      const size_t row = r0 + t + q < p.rows ? r0 + t + q : p.rows - 1;
      load(p.dy + row * p.d, dy[q]);
      load(p.x + row * p.d, x[q]);
      if (p.res) load(p.res + row * p.d, res[q]);
      rs[q] = p.rstd[row];
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const bool ok = r0 + t + q < p.rows;                // uniform
      s[q] = 0.0f;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        x[q][j] *= rs[q];
        const float g = dy[q][j] * wv[j];
        if (ok) dwv[j] = fmaf(dy[q][j], x[q][j], dwv[j]);
        dy[q][j] = g;
        s[q] = fmaf(g, x[q][j], s[q]);
      }
      s[q] = lanes_sum(s[q]) / (float)p.d;
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      if (r0 + t + q >= p.rows) break;
      float* __restrict__ dx = p.dx + (r0 + t + q) * p.d;
      float v[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        v[j] = rs[q] * fmaf(-x[q][j], s[q], dy[q][j]);
        if (p.res) v[j] += res[q][j];
      }
      if constexpr (V4) {
#pragma unroll
        for (int j = 0; j < NJ; j += 4)
          if (col(j) < p.d) *reinterpret_cast<float4*>(dx + col(j)) = make_float4(v[j], v[j + 1], v[j + 2], v[j + 3]);
      } else {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          if (col(j) < p.d) dx[col(j)] = v[j];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) s_w[wave][col(j)] = dwv[j];
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
