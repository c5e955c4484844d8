// Argument blocks of the block kernels (blocks.h), shared with the host side.
#pragma once
#include <stddef.h>

namespace aussm {

constexpr int CONV_PIECE = 2048;   // steps of a row per wavefront of the backward kernel
constexpr int NORM_ROWS = 32;      // rows per workgroup of the norm's backward kernel
constexpr int NORM_MAX_D = 1024;
constexpr int COLSUM_ROWS = 256;

struct ConvRowsArgs {
  const float* x;      // row (b, i) at x + b xs_b + i L
  const float* w;      // [D, K], K <= 8
  const float* bias;   // [D] or null
  float* y;            // [B, D, L] (forward)
  const float* dy;     // [B, D, L] (backward)
  float* dx;           // row (b, i) at dx + b dxs_b + i L
  float* dw;           // [D, K], accumulated into
  float* dbias;        // [D] or null, accumulated into
  long xs_b, dxs_b;
  int B, D, L, K;
};

struct NormArgs {
  const float* x;      // [rows, d]
  const float* w;      // [d]
  float* y;            // forward
  float* rstd;         // [rows]
  const float* dy;     // backward
  const float* res;    // [rows, d] added to dx, or null
  float* dx;
  float* dw;           // [d], accumulated into
  size_t rows;
  int d;
  float eps;
};

}  // namespace aussm
