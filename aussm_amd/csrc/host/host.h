// Entry points of the native host path, bound to Python in module.cpp.
#pragma once
#include "common.h"

namespace aussm_host {

int unitary_ck(int b, int d, int n, int l);
std::pair<Tensor, Tensor> unitary_scan(const Tensor& u, const Tensor& delta, const Tensor& theta, const Tensor& Bc, const Tensor& Cc,
                                       const OptTensor& D, const OptTensor& z, const OptTensor& h0, bool want_state);
std::pair<Tensor, Tensor> complex_scan(const Tensor& u, const Tensor& delta, const Tensor& rho, const Tensor& theta, const Tensor& Bc,
                                       const Tensor& Cc, const OptTensor& D, const OptTensor& z, const OptTensor& h0, bool want_state);
std::pair<Tensor, Tensor> selective_scan(const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B, const Tensor& C,
                                         const OptTensor& D, const OptTensor& z, const OptTensor& delta_bias, bool delta_softplus,
                                         bool want_state, const OptTensor& h0);

bool operator_supported(int64_t b, int64_t d, int64_t n, int64_t l);
Tensor adaptive_operator(const Tensor& u, const Tensor& dt, const Tensor& x, const Tensor& x_bias, const Tensor& B, const Tensor& C,
                         const Tensor& D, const Tensor& z);

// The blocks and linear layers answer nothing where they do not take the tensors (another type or device, sizes
// beyond the kernels): the caller then composes the layer from separate operators.
// (the AUSSM block also returns what it handed to its operator, outside the graph: u, dt, the rows whose second half is z, and,
// one after the other in one buffer, the projection's weight and bias as the operator's x and x_bias)
struct AussmBlockResult { Tensor out, u, dt, xz, x_and_bias; };
std::optional<AussmBlockResult> aussm_block(const Tensor& x, const OptTensor& norm_w, double eps, bool residual, const Tensor& W_in, const OptTensor& b_in,
                      const Tensor& conv_w, const OptTensor& conv_b, const Tensor& W_xp, const Tensor& W_dt, const Tensor& b_dt, const Tensor& xA_w,
                      const Tensor& xA_b, const Tensor& B, const Tensor& C, const Tensor& D, const Tensor& W_out, const OptTensor& b_out, double scale);
OptTensor mamba_block(const Tensor& x, const OptTensor& norm_w, double eps, bool residual, const Tensor& W_in, const OptTensor& b_in,
                      const Tensor& conv_w, const OptTensor& conv_b, const Tensor& W_xp, const Tensor& W_dt, const Tensor& b_dt, const Tensor& A_log,
                      const Tensor& D, const Tensor& W_out, const OptTensor& b_out);
OptTensor norm_linear(const Tensor& x, const OptTensor& norm_w, double eps, const Tensor& W, const OptTensor& b);

}  // namespace aussm_host
