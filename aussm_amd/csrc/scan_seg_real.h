// Splitting the complex and the real (S6) scans along the sequence.  With few (batch, channel group)
// pairs a launch of the scan kernels leaves most of the chip idle, so the sequence is cut into ns
// segments and the scan runs over (batch, segment) pairs:
//   forward   1. oct_fwd_kernel over the pairs from a zero state, outputs off: end state Z_k of every
//                segment and the product q_k of its a_l (FwdArgs::ptot),
//             2. the chain  h <- q_k h + Z_k  over the segments of each (batch, channel, state)
//                (seg_carry_kernel for complex states, seg_carry_real_kernel here),
//             3. oct_fwd_kernel over the pairs, each from the state that enters it;
//   backward  1. oct_adj_kernel: adjoint Y_k of the state entering every segment from a zero adjoint
//                at its end (the reverse recurrence alone - no states are needed for it), and q_k,
//             2. the chain  g <- conj(q_k) g + Y_k, last segment first,
//             3. oct_bwd_kernel over the pairs, each from the adjoint that enters it at its end.
// The unitary scan on the vector-ALU kernels (more than 16 states, a length that is not a multiple of 4, ...)
// splits the same way: oct_fwd_kernel<VAR_UNITARY> for 1. and 3., oct_adj_kernel, the complex chains, and unitary_bwd_kernel
// over the pairs, which takes the state at the end of each segment from the forward pass's checkpoints.
// Reference semantics: the loops of extension-cpp/extension_cpp/ops.py:215-223 (unitary), :270-291 (complex)
// and :349-356 (real) are associative in exactly this way; the reference itself does not split.
#pragma once
#include "scan_common.h"

namespace aussm {

// Chain of the segments of one (batch, channel, state) of the real scan, q_k = exp(A[d,n] * sum of the
// segment's step sizes).  Forward (ADJ false): on entry seg[k] holds the end state of segment k from a
// zero start, on return the state that enters it; the state after the last segment goes to `last`.
// ADJ: on entry the adjoint at the start of segment k from a zero adjoint at its end, on return the
// adjoint that enters it at its end, walking from the last segment; the adjoint of the initial state
// goes to `last`.  `first`: state before the first segment / adjoint after the last one (or null).
template <bool ADJ>
__global__ void seg_carry_real_kernel(float* __restrict__ seg, const float* __restrict__ ptot,
                                      const float* __restrict__ A, const float* __restrict__ first,
                                      float* __restrict__ last, int B, int D, int N, int ns) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)B * D * N) return;
  const int n = (int)(idx % N);
  const int d = (int)((idx / N) % D);
  const int b = (int)(idx / ((size_t)N * D));
  const float a2 = A[(size_t)d * N + n] * LOG2E;
  float h = first ? first[idx] : 0.0f;
  for (int j = 0; j < ns; ++j) {
    const int k = ADJ ? ns - 1 - j : j;
    const size_t v = ((size_t)b * ns + k) * D + d;
    const float z = seg[v * N + n];
    const float q = __builtin_amdgcn_exp2f(ptot[v * 2] * a2);
    seg[v * N + n] = h;
    h = fmaf(q, h, z);
  }
  if (last) last[idx] = h;
}

}  // namespace aussm
