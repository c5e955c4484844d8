// Translation unit of the vector-ALU forward scans (scan_fwd.h).
#include "launch.h"
#include "scan_fwd.h"

namespace aussm {

#define AUSSM_FWD_CASE(NW_, NT_)                                                                     \
  if (c.nw == NW_ && c.nt == NT_) {                                                                  \
    hipLaunchKernelGGL((core_fwd_kernel<VAR, NW_, NT_, Tin, Tbc>), grid, dim3(NT_), 0, s, a);        \
    return launch_status();                                                                          \
  }

template <int VAR, typename Tin, typename Tbc>
static int core_fwd_t(const FwdArgs& a, Cfg c, hipStream_t s) {
  const dim3 grid((unsigned)(a.B * a.ncg));
  // (the complex scan's instance without bounds came out slower: 410 -> 650 us at B32 D512 N16 L2048)
  if constexpr (VAR == VAR_REAL) {
    const void* const ps[] = {a.u, a.delta, a.y};
    bool plain = c.nw == 2 && c.nt == 512 && a.N == 16 && a.D % CH == 0 && a.ld % T == 0 && a.L % T == 0 && a.y && !a.z && !a.u_act &&
                 !a.delta_softplus && !a.delta_bias && !a.ptot;
    for (const void* q : ps) plain = plain && (reinterpret_cast<uintptr_t>(q) & 15) == 0;
    if (plain) {
      hipLaunchKernelGGL((core_fwd_kernel<VAR, 2, 512, Tin, Tbc, true>), grid, dim3(512), 0, s, a);
      return launch_status();
    }
  }
  AUSSM_FWD_CASE(1, 256) AUSSM_FWD_CASE(2, 256) AUSSM_FWD_CASE(4, 256) AUSSM_FWD_CASE(8, 256)
  AUSSM_FWD_CASE(16, 256) AUSSM_FWD_CASE(1, 512) AUSSM_FWD_CASE(2, 512) AUSSM_FWD_CASE(4, 512)
  AUSSM_FWD_CASE(8, 512)
  return -2;
}

template <int VAR>
static int core_fwd_v(const FwdArgs& a, int in_dtype, Cfg c, hipStream_t s) {
  if (in_dtype == 0) return core_fwd_t<VAR, float, float>(a, c, s);
  if constexpr (VAR == VAR_UNITARY) {
    if (in_dtype == 1) return core_fwd_t<VAR, bf16_t, bf16_t>(a, c, s);
  } else {
    if (in_dtype == IN_BF16_BC32) return core_fwd_t<VAR, bf16_t, float>(a, c, s);
  }
  return -2;
}

int run_core_fwd(int variant, const FwdArgs& a, int in_dtype, Cfg c, hipStream_t s) {
  if (variant == VAR_UNITARY) return core_fwd_v<VAR_UNITARY>(a, in_dtype, c, s);
  if (variant == VAR_COMPLEX) return core_fwd_v<VAR_COMPLEX>(a, in_dtype, c, s);
  return core_fwd_v<VAR_REAL>(a, in_dtype, c, s);
}

}  // namespace aussm
