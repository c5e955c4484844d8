// Argument block of the fp32-accurate GEMM (gemm.h), shared with the host side.
#pragma once

namespace aussm {

//     C(m, n) = act( alpha sum_k A(m, k) B(k, n) + bias_scale bias[m] + add(m, n) )
// Column n lies in batch n / nper, at position n % nper of it: B and C move by sbb / scb per batch and by sbn / scn
// per position, so that a batch of products with one A is a single product over all columns.
//     reduce over z:  C(m, n) = alpha sum_z sum_k A_z(m, k) B_z(k, n)      (saz, sbz)
// Strides are in elements; one of sam / sak, one of sbk / sbn and one of scm / scn is 1.
struct XGemmArgs {
  const float* A;
  const float* B;
  float* C;
  const float* bias;      // [M] or null
  const float* add;       // laid out as C (may be C), or null
  float alpha, bias_scale;
  int act;                // 1: softplus
  long sam, sak, saz;
  long sbk, sbn, sbb, sbz;
  long scm, scn, scb;
  int M, N, K, Z, nper;
  int slices;             // set by the launch: the (z, step) pairs are cut into that many slices, summed with atomics
  int reduce;             // C holds the addend of the sum (zero for a plain product): slices may be more than one
};

}  // namespace aussm
