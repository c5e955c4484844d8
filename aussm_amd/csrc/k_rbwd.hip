// Translation unit of the recomputing reverse scans, complex and real (scan_bwd_recompute.h).
#include "launch.h"
#include "scan_bwd_recompute.h"

namespace aussm {

#define AUSSM_RBWD_CASE(NW_)                                                                         \
  if (nw == NW_) {                                                                                   \
    hipLaunchKernelGGL((recompute_bwd_kernel<VAR, NW_, 256, Tin, float>), grid, dim3(256), 0, s, a); \
    done = true;                                                                                     \
  }

template <int VAR, typename Tin>
static int rec_bwd_t(const RecBwdArgs& args, hipStream_t s) {
  const dim3 grid((unsigned)(args.B * args.ncg));
  // one launch per block of 16 states (stream order makes the later blocks' additions safe)
  for (int nbase = 0; nbase < args.N; nbase += 16) {
    RecBwdArgs a = args;
    a.nbase = nbase;
    a.accum = nbase > 0;
    const int left = args.N - nbase;
    const int nw = left <= 4 ? 1 : (left <= 8 ? 2 : 4);
    bool done = false;
#ifndef AUSSM_REC_NARROW
    // a full block of 16 states: eight wavefronts of two states, two wavefronts per SIMD (the complex scan with a
    // gate gradient to return keeps a fourth partial sum per wavefront)
    if (left > 8) {
      const bool plain = !a.z && !a.dz && !a.u_act && !a.delta_softplus && !a.delta_bias && !a.dbias && !a.accum;
      // (a launch that is split along the sequence has segments of whole tiles, the last one may end earlier)
      const bool whole = left >= 16 && a.D % CH == 0 && a.ld % RT == 0 && a.L % RT == 0;
      auto go = [&](auto whole_tag) {
        constexpr bool W = decltype(whole_tag)::value;
        if (plain) {
          hipLaunchKernelGGL((recompute_bwd_kernel<VAR, 2, 512, Tin, float, false, true, W>), grid, dim3(512), 0, s, a);
        } else if constexpr (VAR == VAR_COMPLEX) {
          if (a.dz) hipLaunchKernelGGL((recompute_bwd_kernel<VAR, 2, 512, Tin, float, true, false, W>), grid, dim3(512), 0, s, a);
          else hipLaunchKernelGGL((recompute_bwd_kernel<VAR, 2, 512, Tin, float, false, false, W>), grid, dim3(512), 0, s, a);
        } else {
          hipLaunchKernelGGL((recompute_bwd_kernel<VAR, 2, 512, Tin, float, false, false, W>), grid, dim3(512), 0, s, a);
        }
      };
      if (whole) go(std::true_type{});
      else go(std::false_type{});
      done = true;
    }
#endif
    if (!done) { AUSSM_RBWD_CASE(1) AUSSM_RBWD_CASE(2) AUSSM_RBWD_CASE(4) }
    if (!done) return -2;
    if (int e = launch_status()) return e;
  }
  return 0;
}

int run_rec_bwd(int variant, const RecBwdArgs& a, int in_dtype, hipStream_t s) {
  if (in_dtype != 0 && in_dtype != IN_BF16_BC32) return -2;      // B_t / C_t are float in every instance
  if (variant == VAR_COMPLEX)
    return in_dtype ? rec_bwd_t<VAR_COMPLEX, bf16_t>(a, s) : rec_bwd_t<VAR_COMPLEX, float>(a, s);
  return in_dtype ? rec_bwd_t<VAR_REAL, bf16_t>(a, s) : rec_bwd_t<VAR_REAL, float>(a, s);
}

}  // namespace aussm
