// Translation unit of the unitary reverse scan of 33 to 64 states that leaves du and ddelta in bf16 (scan_bwd_unitary.h).
#include "launch.h"
#include "scan_bwd_unitary.h"

namespace aussm {

// The backward workgroup keeps a (dw, dtheta) slab per wavefront in LDS: four wavefronts afford
// 32-step tiles, eight wavefronts 16-step tiles.
int run_unitary_bwd_generic(const UniBwdArgs& a, Cfg c, hipStream_t s) {
  const dim3 grid((unsigned)(a.B * a.ncg)), block((unsigned)c.nt);
  if (c.nw == 8 && c.nt == 512) hipLaunchKernelGGL((unitary_bwd_kernel<8, 512, 16, bf16_t>), grid, block, 0, s, a);
  else if (c.nw == 16 && c.nt == 256) hipLaunchKernelGGL((unitary_bwd_kernel<16, 256, 32, bf16_t>), grid, block, 0, s, a);
  else return -2;
  return launch_status();
}

}  // namespace aussm
