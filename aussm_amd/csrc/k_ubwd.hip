// Translation unit of the unitary reverse scan on the vector ALU (scan_bwd_unitary.h).
#include "launch.h"
#include "scan_bwd_unitary.h"

namespace aussm {

// The backward workgroup keeps a (dw, dtheta) slab per wavefront in LDS: four wavefronts afford
// 32-step tiles, eight wavefronts 16-step tiles.
#define AUSSM_UBWD_CASE(NW_, NT_, TT_)                                                               \
  if (c.nw == NW_ && c.nt == NT_) {                                                                  \
    hipLaunchKernelGGL((unitary_bwd_kernel<NW_, NT_, TT_, Tin>), grid, dim3(NT_), 0, s, a);          \
    return launch_status();                                                                          \
  }

template <typename Tin>
static int unitary_bwd_t(const UniBwdArgs& a, Cfg c, hipStream_t s) {
  const dim3 grid((unsigned)(a.B * a.ncg));
  AUSSM_UBWD_CASE(1, 256, 32) AUSSM_UBWD_CASE(2, 256, 32) AUSSM_UBWD_CASE(4, 256, 32)
  AUSSM_UBWD_CASE(8, 256, 32) AUSSM_UBWD_CASE(16, 256, 32)
  AUSSM_UBWD_CASE(1, 512, 16) AUSSM_UBWD_CASE(2, 512, 16) AUSSM_UBWD_CASE(4, 512, 16)
  AUSSM_UBWD_CASE(8, 512, 16)
  return -2;
}

int run_unitary_bwd_generic(const UniBwdArgs& a, int in_dtype, Cfg c, hipStream_t s) {
  return in_dtype == 1 ? unitary_bwd_t<bf16_t>(a, c, s) : unitary_bwd_t<float>(a, c, s);
}

}  // namespace aussm
