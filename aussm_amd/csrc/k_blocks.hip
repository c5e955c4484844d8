// Translation unit of the block kernels (blocks.h).
#include "blocks.h"
#include "launch.h"

#include <initializer_list>

namespace aussm {

// 16-byte accesses to whole groups of four
static bool quads(std::initializer_list<const void*> ps, std::initializer_list<long> strides) {
  for (const void* q : ps)
    if (reinterpret_cast<uintptr_t>(q) & 15) return false;
  for (long t : strides)
    if (t & 3) return false;
  return true;
}

int run_conv_rows_fwd(const ConvRowsArgs& a, hipStream_t s) {
  const size_t n = (size_t)a.B * a.D * ((a.L + 3) / 4);
  if ((n + 255) / 256 > 0x7fffffffULL) return -2;
  const dim3 grid((unsigned)((n + 255) / 256));
  if (a.K == 4 && quads({a.x}, {a.L, a.xs_b})) hipLaunchKernelGGL((conv_rows_fwd_kernel<4, true>), grid, dim3(256), 0, s, a);
  else if (a.K == 4) hipLaunchKernelGGL((conv_rows_fwd_kernel<4, false>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((conv_rows_fwd_kernel<0, false>), grid, dim3(256), 0, s, a);
  return launch_status();
}

int run_conv_rows_bwd(const ConvRowsArgs& a, hipStream_t s) {
  const size_t rows = (size_t)a.B * a.D;
  const dim3 grid((unsigned)((rows + 3) / 4), (unsigned)((a.L + CONV_PIECE - 1) / CONV_PIECE));
  if ((rows + 3) / 4 > 0x7fffffffULL || grid.y > 65535) return -2;
  if (a.K == 4 && quads({a.x, a.dy, a.dx}, {a.L, a.xs_b, a.dxs_b})) hipLaunchKernelGGL((conv_rows_bwd_kernel<4, true>), grid, dim3(256), 0, s, a);
  else if (a.K == 4) hipLaunchKernelGGL((conv_rows_bwd_kernel<4, false>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((conv_rows_bwd_kernel<0, false>), grid, dim3(256), 0, s, a);
  return launch_status();
}

#define NORM_DISPATCH(KERNEL, grid)                                                                    \
  if (a.d <= 64) hipLaunchKernelGGL(KERNEL<1>, grid, dim3(256), 0, s, a);                              \
  else if (a.d <= 128) hipLaunchKernelGGL(KERNEL<2>, grid, dim3(256), 0, s, a);                        \
  else if (a.d <= 256) hipLaunchKernelGGL(KERNEL<4>, grid, dim3(256), 0, s, a);                        \
  else if (a.d <= 512) hipLaunchKernelGGL(KERNEL<8>, grid, dim3(256), 0, s, a);                        \
  else hipLaunchKernelGGL(KERNEL<16>, grid, dim3(256), 0, s, a);

int run_norm_fwd(const NormArgs& a, hipStream_t s) {
  if (a.d > NORM_MAX_D || (a.rows + 3) / 4 > 0x7fffffffULL) return -2;
  NORM_DISPATCH(rms_norm_fwd_kernel, dim3((unsigned)((a.rows + 3) / 4)))
  return launch_status();
}

int run_norm_bwd(const NormArgs& a, hipStream_t s) {
  if (a.d > NORM_MAX_D || (a.rows + NORM_ROWS - 1) / NORM_ROWS > 0x7fffffffULL) return -2;
  const dim3 grid((unsigned)((a.rows + NORM_ROWS - 1) / NORM_ROWS));
  const bool v4 = a.d > 128 && quads({a.dy, a.x, a.res, a.dx}, {a.d});
#define NB(NJ_, V4_) hipLaunchKernelGGL((rms_norm_bwd_kernel<NJ_, V4_>), grid, dim3(256), 0, s, a)
  if (a.d <= 64) NB(1, false);
  else if (a.d <= 128) NB(2, false);
  else if (a.d <= 256) { if (v4) NB(4, true); else NB(4, false); }
  else if (a.d <= 512) { if (v4) NB(8, true); else NB(8, false); }
  else { if (v4) NB(16, true); else NB(16, false); }
#undef NB
  return launch_status();
}

int run_col_sum(const float* x, float* out, size_t rows, int d, float scale, hipStream_t s) {
  const dim3 grid((unsigned)((d + 63) / 64), (unsigned)((rows + COLSUM_ROWS - 1) / COLSUM_ROWS));
  if ((rows + COLSUM_ROWS - 1) / COLSUM_ROWS > 65535) return -2;
  hipLaunchKernelGGL(col_sum_kernel, grid, dim3(256), 0, s, x, out, rows, d, scale);
  return launch_status();
}

int run_row_sum(const float* x, float* out, size_t rows, int d, int L, float scale, hipStream_t s) {
  if ((rows + 3) / 4 > 0x7fffffffULL) return -2;
  hipLaunchKernelGGL(row_sum_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, x, out, rows, d, L, scale);
  return launch_status();
}

int run_neg_exp(const float* a_log, const float* dA, float* out, int n, hipStream_t s) {
  hipLaunchKernelGGL(neg_exp_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a_log, dA, out, n);
  return launch_status();
}

}  // namespace aussm
