// Launch functions of the library's translation units (one unit per kernel family, so that they
// compile side by side).  Each enqueues on the given stream and returns AUSSM_OK or the launch's
// hipError_t; argument checking is done by the callers in scan_api.hip.
#pragma once
#include <hip/hip_runtime.h>

#include "scan_args.h"
#include "block_args.h"
#include "dropin_args.h"
#include "gemm_args.h"

namespace aussm {

inline int launch_status() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

// A workgroup of nt threads (nt / 64 wavefronts) of unitary_bwd_kernel owns 64 channels; each wavefront owns nw states.
struct Cfg { int nw, nt; };

// ---- k_oct_fwd.hip, k_oct_bwd.hip, k_ubwd.hip: vector-ALU scans; k_generic.hip: convolution, layout swap.  in_dtype: 0 float, 1 bf16
int run_oct_fwd(int variant, const FwdArgs& a, int in_dtype, hipStream_t s);
int run_oct_adj(int variant, const AdjSegArgs& a, int in_dtype, unsigned grid, hipStream_t s);   // adjoint entering every segment
int run_oct_bwd(int variant, const RecBwdArgs& a, int in_dtype, hipStream_t s);
int run_oct_ubwd(const UniBwdArgs& a, int in_dtype, hipStream_t s);   // N <= 32 where du leaves in bf16
int run_unitary_bwd_generic(const UniBwdArgs& a, Cfg c, hipStream_t s);   // N > 32, bf16 inputs, du and ddelta in bf16
int run_aux_invalidate(float* tag, bool fill_tag, bool images_tag, hipStream_t s);   // clears tag(s) in the buffer's pad
int run_hbm_probe(const float* a, const float* b, const float* c, float* o1, float* o2, int rows, int L, int pattern,
                  int write, hipStream_t s);
int run_conv_fwd(const ConvArgs& a, hipStream_t s);
int run_conv_bwd(const ConvArgs& a, hipStream_t s);
int run_swap_last2(const SwapArgs& a, int B, hipStream_t s);
// dz null: out = ypre silu(z); else out = dy silu(z), dz = dy ypre silu'(z)
int run_gate(const float* dy, const float* ypre, const float* z, float* out, float* dz, size_t n, hipStream_t s);

// ---- k_xdl.hip: matrix-core unitary scans that prepare their operands themselves, and the
// kernels of the split along L.  mode: operand pieces (2, 3; backward also 5 = three everywhere).
int run_xdl_fwd(int mode, const FwdArgs& a, int in_dtype, hipStream_t s);
int run_xdl_bwd(int mode, const UniBwdArgs& a, int in_dtype, hipStream_t s);
int run_seg_state(bool adjoint, const SegArgs& a, int in_dtype, unsigned grid, hipStream_t s);

// ---- k_px.hip: matrix-core unitary scans on operands prepared by a pre-pass
int run_px_prep(const PrepArgs& a, int B, int in_dtype, hipStream_t s);
int run_prep_seg(const PrepArgs& a, int B, const SegArgs& sa, unsigned nseg, int in_dtype, hipStream_t s);   // both in one launch
int run_px_fwd(const FwdArgs& a, const u4* img, const ImgNote& note, int in_dtype, hipStream_t s);
int run_px_bwd(const UniBwdArgs& a, const u4* img, int in_dtype, hipStream_t s);

// ---- k_dropin.hip: the reference's 12-input operator as fused kernels
int dropin_channels_per_workgroup(int ks);
int dropin_compiled_ks(int ks);
size_t dropin_records(int ks, int steps);
int run_dropin_prep(DropinPrepArgs a, int bg, bool rows, const FillArgs& f, hipStream_t s);   // rows: the records of x too
int run_dropin_fwd(const DropinArgs& a, hipStream_t s);
int run_dropin_seg(const DropinBwdArgs& a, hipStream_t s);   // maps of the segments (nseg > 1): backward with sega, else forward
int run_dropin_bwd(const DropinBwdArgs& a, hipStream_t s);
int run_fill(const FillArgs& a, hipStream_t s);   // several buffers set (zero or a copy) in one launch

// ---- k_blocks.hip: what the blocks do around the scans, on channel rows (b, d, l)
int run_conv_rows_fwd(const ConvRowsArgs& a, hipStream_t s);
int run_conv_rows_bwd(const ConvRowsArgs& a, hipStream_t s);
int run_norm_fwd(const NormArgs& a, hipStream_t s);
int run_norm_bwd(const NormArgs& a, hipStream_t s);
int run_col_sum(const float* x, float* out, size_t rows, int d, float scale, hipStream_t s);
int run_row_sum(const float* x, float* out, size_t rows, int d, int L, float scale, hipStream_t s);
int run_neg_exp(const float* a_log, const float* dA, float* out, int n, hipStream_t s);

// ---- k_gemm.hip: fp32-accurate matrix products on the bf16 matrix cores
int run_xgemm(XGemmArgs a, hipStream_t s);

}  // namespace aussm
