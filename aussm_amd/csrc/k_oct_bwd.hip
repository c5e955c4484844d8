// Translation unit of the recomputing reverse scans, complex and real (scan_oct.h).
#include "launch.h"
#include "scan_oct.h"

namespace aussm {

// One launch per block of states (stream order makes the later blocks' additions safe): as many groups of eight as the
// registers for the recomputed states and the slabs in LDS hold - complex 16 states, real 24.
template <int VAR, typename Tin>
static int oct_bwd_t(const RecBwdArgs& args, hipStream_t s) {
  const dim3 grid((unsigned)(args.B * args.ncg)), block(512);
  constexpr int BLOCK = VAR == VAR_REAL ? 24 : 16;
  for (int nbase = 0; nbase < args.N; nbase += BLOCK) {
    RecBwdArgs a = args;
    a.nbase = nbase;
    a.accum = nbase > 0;
    const int left = a.N - nbase, S = left >= BLOCK ? BLOCK / 8 : (left + 7) / 8;
    auto launch = [&](auto sc, auto full, auto ragged) {
      constexpr int S_ = decltype(sc)::value;
      constexpr bool F = decltype(full)::value, R = decltype(ragged)::value;
      if (a.z) hipLaunchKernelGGL((oct_bwd_kernel<VAR, S_, F, R, Tin, Tin, true>), grid, block, 0, s, a);
      else hipLaunchKernelGGL((oct_bwd_kernel<VAR, S_, F, R, Tin, Tin, false>), grid, block, 0, s, a);
    };
    auto go = [&](auto sc, auto full) {
      if constexpr (VAR == VAR_REAL) {
        if (a.ld % 16 == 0) return launch(sc, full, std::false_type{});
      }
      launch(sc, full, std::true_type{});
    };
    using std::integral_constant;
    if (S == 1) go(integral_constant<int, 1>{}, std::false_type{});
    else if (S == 2) {
      if (left >= 16) go(integral_constant<int, 2>{}, std::true_type{});
      else go(integral_constant<int, 2>{}, std::false_type{});
    } else {
      if constexpr (VAR == VAR_REAL) {
        go(integral_constant<int, 3>{}, std::false_type{});
      }
    }
    if (int e = launch_status()) return e;
  }
  return 0;
}

int run_oct_bwd(int variant, const RecBwdArgs& a, int in_dtype, hipStream_t s) {
  if (variant == VAR_COMPLEX) return in_dtype ? oct_bwd_t<VAR_COMPLEX, bf16_t>(a, s) : oct_bwd_t<VAR_COMPLEX, float>(a, s);
  return in_dtype ? oct_bwd_t<VAR_REAL, bf16_t>(a, s) : oct_bwd_t<VAR_REAL, float>(a, s);
}

// The unitary scan's, blocks of 32 states.
template <typename Tin>
static int oct_ubwd_t(const RecBwdArgs& args, hipStream_t s) {
  const dim3 grid((unsigned)(args.B * args.ncg)), block(512);
  for (int nbase = 0; nbase < args.N; nbase += 32) {
    RecBwdArgs a = args;
    a.nbase = nbase;
    a.accum = nbase > 0;
    auto go = [&](auto sc, auto full) {
      constexpr int S = decltype(sc)::value;
      constexpr bool F = decltype(full)::value;
      if (a.ld % 16 == 0) hipLaunchKernelGGL((oct_bwd_kernel<VAR_UNITARY, S, F, false, Tin, Tin, false>), grid, block, 0, s, a);
      else hipLaunchKernelGGL((oct_bwd_kernel<VAR_UNITARY, S, F, true, Tin, Tin, false>), grid, block, 0, s, a);
    };
    using std::integral_constant;
    const int left = a.N - nbase, S = (left + 7) / 8;
    if (S == 1) go(integral_constant<int, 1>{}, std::false_type{});
    else if (S == 2 && left == 16) go(integral_constant<int, 2>{}, std::true_type{});
    else if (S == 2) go(integral_constant<int, 2>{}, std::false_type{});
    else if (S == 3) go(integral_constant<int, 3>{}, std::false_type{});
    else go(integral_constant<int, 4>{}, std::false_type{});
    if (int e = launch_status()) return e;
  }
  return 0;
}

int run_oct_ubwd(const UniBwdArgs& u, int in_dtype, hipStream_t s) {
  RecBwdArgs a{};
  a.dy = u.dy; a.dhL = u.dhL; a.u = u.u; a.delta = u.delta; a.theta = u.theta; a.Bm = u.Bm; a.Cm = u.Cm; a.Dskip = u.Dskip; a.hck = u.hck;
  a.du = u.du; a.ddelta = u.ddelta; a.dtheta = u.dtheta; a.dB = u.dB; a.dC = u.dC; a.dD = u.dD; a.dh0 = u.dh0;
  a.B = u.B; a.D = u.D; a.N = u.N; a.L = u.L; a.ck = u.ck; a.nck = u.nck; a.ncg = u.ncg; a.ld = u.ld; a.ns = u.ns; a.seg = u.seg; a.segq = u.segq;
  a.urep = u.urep; a.g16 = u.g16;
  return in_dtype ? oct_ubwd_t<bf16_t>(a, s) : oct_ubwd_t<float>(a, s);
}

}  // namespace aussm
