// Translation unit of the vector-ALU forward scans and of the adjoints of a call that is split along L (scan_oct.h).
#include "launch.h"
#include "scan_oct.h"

namespace aussm {

// groups of eight states: S = 1 .. 4 (N <= 32), 6 or 8
template <int VAR, typename Tin>
static int oct_fwd_t(const FwdArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)(a.B * a.ncg)), block(512);
  const bool lean = a.ptot != nullptr;
  auto go = [&](auto sc) {
    constexpr int S = decltype(sc)::value;
    if (lean) {
      hipLaunchKernelGGL((oct_fwd_kernel<VAR, S, false, Tin, Tin, true>), grid, block, 0, s, a);
      return;
    }
    if constexpr (S <= 2) {
      if (a.N == 8 * S) {
        hipLaunchKernelGGL((oct_fwd_kernel<VAR, S, true, Tin, Tin, false>), grid, block, 0, s, a);
        return;
      }
    }
    hipLaunchKernelGGL((oct_fwd_kernel<VAR, S, false, Tin, Tin, false>), grid, block, 0, s, a);
  };
  const int S = (a.N + 7) / 8;
  if (S == 1) go(std::integral_constant<int, 1>{});
  else if (S == 2) go(std::integral_constant<int, 2>{});
  else if (S == 3) go(std::integral_constant<int, 3>{});
  else if (S == 4) go(std::integral_constant<int, 4>{});
  else if (S <= 6) go(std::integral_constant<int, 6>{});
  else if (S <= 8) go(std::integral_constant<int, 8>{});
  else return -2;
  return launch_status();
}

int run_oct_fwd(int variant, const FwdArgs& a, int in_dtype, hipStream_t s) {
  if (variant == VAR_UNITARY) return in_dtype ? oct_fwd_t<VAR_UNITARY, bf16_t>(a, s) : oct_fwd_t<VAR_UNITARY, float>(a, s);
  if (variant == VAR_COMPLEX) return in_dtype ? oct_fwd_t<VAR_COMPLEX, bf16_t>(a, s) : oct_fwd_t<VAR_COMPLEX, float>(a, s);
  return in_dtype ? oct_fwd_t<VAR_REAL, bf16_t>(a, s) : oct_fwd_t<VAR_REAL, float>(a, s);
}

template <int VAR, typename Tin>
static int oct_adj_t(const AdjSegArgs& a, unsigned grid, hipStream_t s) {
  auto go = [&](auto sc) {
    constexpr int S = decltype(sc)::value;
    hipLaunchKernelGGL((oct_adj_kernel<VAR, S, false, Tin, Tin>), dim3(grid), dim3(512), 0, s, a);
  };
  const int S = (a.N + 7) / 8;
  if (S == 1) go(std::integral_constant<int, 1>{});
  else if (S == 2) go(std::integral_constant<int, 2>{});
  else if (S == 3) go(std::integral_constant<int, 3>{});
  else if (S == 4) go(std::integral_constant<int, 4>{});
  else if (S <= 6) go(std::integral_constant<int, 6>{});
  else if (S <= 8) go(std::integral_constant<int, 8>{});
  else return -2;
  return launch_status();
}

int run_oct_adj(int variant, const AdjSegArgs& a, int in_dtype, unsigned grid, hipStream_t s) {
  if (variant == VAR_UNITARY) return in_dtype ? oct_adj_t<VAR_UNITARY, bf16_t>(a, grid, s) : oct_adj_t<VAR_UNITARY, float>(a, grid, s);
  if (variant == VAR_COMPLEX) return in_dtype ? oct_adj_t<VAR_COMPLEX, bf16_t>(a, grid, s) : oct_adj_t<VAR_COMPLEX, float>(a, grid, s);
  return in_dtype ? oct_adj_t<VAR_REAL, bf16_t>(a, grid, s) : oct_adj_t<VAR_REAL, float>(a, grid, s);
}

}  // namespace aussm
