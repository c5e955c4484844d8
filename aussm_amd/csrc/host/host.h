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

}  // namespace aussm_host
