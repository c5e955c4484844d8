// Translation unit of the fp32-accurate GEMM (gemm.h).
#include "gemm.h"
#include "launch.h"

namespace aussm {

template <int TNH, bool QUAD>
static int launch_xgemm(const XGemmArgs& a, unsigned grid, hipStream_t s) {
  const bool ak1 = a.sak == 1, bk1 = a.sbk == 1, tr = a.scm == 1 && a.scn != 1;
#define XG(A_, B_, T_)                                                                       \
  if (ak1 == A_ && bk1 == B_ && tr == T_) {                                                  \
    hipLaunchKernelGGL((xgemm_kernel<A_, B_, T_, TNH, QUAD>), dim3(grid), dim3(256), 0, s, a);     \
    return launch_status();                                                                  \
  }
  XG(false, false, false) XG(false, false, true) XG(false, true, false) XG(false, true, true)
  XG(true, false, false) XG(true, false, true) XG(true, true, false) XG(true, true, true)
#undef XG
  return -2;
}

// Slices: a sum over many steps with few tiles is cut into as many workgroups as run at once (two per compute unit;
// more would start a second round: 540 workgroups 140 us, 450 workgroups 91 us for the product with 90 tiles and
// 128 steps), at least four steps of 32 per slice (shorter ones would spend their time on the atomics of the tile).
int run_xgemm(XGemmArgs a, hipStream_t s) {
  if (a.M < 1 || a.N < 1 || a.K < 1 || a.Z < 1 || a.nper < 1) return -2;
  if (a.reduce && a.scm == 1 && a.scn != 1 && a.nper < a.N) return -2;
  const int tnh = a.N <= 64 ? 1 : 2;
  const long tiles = (long)((a.M + XG_TM - 1) / XG_TM) * ((a.N + 64 * tnh - 1) / (64 * tnh));
  const long steps = (long)((a.K + 31) / 32) * a.Z;
  long sl = 1;
  if (a.reduce && !a.bias && !a.add && !a.act) {
    sl = 512 / tiles;
    if (sl > steps / 4) sl = steps / 4;
    if (sl < 1) sl = 1;
    const long per = (steps + sl - 1) / sl;
    sl = (steps + per - 1) / per;
  }
  if (steps > 0x7fffffffL || tiles * sl > 0x7fffffffL) return -2;
  a.slices = (int)sl;
  // (offsets inside a tile of C are 32-bit)
  if (a.scm < 0 || a.scn < 0 || a.scm >= (1l << 24) || a.scn >= (1l << 24)) return -2;
  const unsigned grid = (unsigned)(tiles * sl);
  if (a.K % 4 == 0) return tnh == 1 ? launch_xgemm<1, true>(a, grid, s) : launch_xgemm<2, true>(a, grid, s);
  return tnh == 1 ? launch_xgemm<1, false>(a, grid, s) : launch_xgemm<2, false>(a, grid, s);
}

}  // namespace aussm
