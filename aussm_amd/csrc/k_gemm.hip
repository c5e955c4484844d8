// Translation unit of the fp32-accurate GEMM (gemm.h).
#include "gemm.h"
#include "launch.h"

namespace aussm {

template <int EN, bool QUAD, bool WIDE>
static int launch_xgemm(const XGemmArgs& a, unsigned grid, hipStream_t s) {
  const bool ak1 = a.sak == 1, bk1 = a.sbk == 1, tr = a.scm == 1 && a.scn != 1;
#define XG(A_, B_, T_)                                                                       \
  if (ak1 == A_ && bk1 == B_ && tr == T_) {                                                  \
    hipLaunchKernelGGL((xgemm_kernel<A_, B_, T_, EN, QUAD, WIDE>), dim3(grid), dim3(WIDE ? 512 : 256), 0, s, a);     \
    return launch_status();                                                                  \
  }
  XG(false, false, false) XG(false, false, true) XG(false, true, false) XG(false, true, true)
  XG(true, false, false) XG(true, false, true) XG(true, true, false) XG(true, true, true)
#undef XG
  return -2;
}

// Tile: the wide ones for more rows than the narrow one has, by the rounds that the tiles make on the chip (256 compute
// units, one wide or two narrow workgroups each) times what a round takes: 1 for 256 x 128, 0.88 for 256 x 96, 1.2 for two of
// 128 x 128, 0.72 for one.  23040 columns, us narrow / 96 / 128: 256 rows, K = 1024 93 / 70 / 78; 512 rows, K = 256 46 / 43 /
// 50; 1024 rows, K = 256 77 / 80 / 73; 512 rows, K = 16 17.1 / 17.1 / 19.2.
//
// Slices: a sum over many steps with few tiles is cut into as many workgroups as run at once (more would start a second
// round: 540 workgroups 140 us, 450 workgroups 91 us for the product with 90 tiles and 128 steps), at least four steps of
// 32 per slice (shorter ones would spend their time on the atomics of the tile).  The wide tile from 32 steps a slice on:
// 4096 x 256, sums of 23040, 281 -> 248 us; 512 x 256 (12 steps) 56 against 58 us.
int run_xgemm(XGemmArgs a, hipStream_t s) {
  if (a.M < 1 || a.N < 1 || a.K < 1 || a.Z < 1 || a.nper < 1) return -2;
  if (a.reduce && a.scm == 1 && a.scn != 1 && a.nper < a.N) return -2;
  const long steps = (long)((a.K + 31) / 32) * a.Z;
  const bool sliced = a.reduce && !a.bias && !a.add && !a.act;
  auto tiles_of = [&](int tm, int tn) { return (long)((a.M + tm - 1) / tm) * ((a.N + tn - 1) / tn); };
  bool wide = false;
  int en = a.N <= 64 ? 2 : 4;
  if (a.M > XG_TM && a.N > 64) {
    if (sliced) {
      const long t = tiles_of(XG_TM_WIDE, 128);
      wide = steps >= 32 * (t < 256 ? 256 / t : 1);
    } else {
      auto rounds = [](long t, long slots) { return (double)((t + slots - 1) / slots); };
      const double w4 = rounds(tiles_of(XG_TM_WIDE, 128), 256), w3 = 0.88 * rounds(tiles_of(XG_TM_WIDE, 96), 256);
      const long t = tiles_of(XG_TM, 128);
      const double narrow = 1.2 * (double)(t / 512) + (t % 512 > 256 ? 1.2 : t % 512 ? 0.72 : 0.0);
      wide = w3 < narrow || w4 < narrow;
      if (wide && w3 < w4) en = 3;
    }
  }
  const int tm = wide ? XG_TM_WIDE : XG_TM;
  const long tiles = tiles_of(tm, 32 * en);
  long sl = 1;
  if (sliced) {
    sl = (wide ? 256 : 512) / tiles;
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
  if (a.K % 4 == 0) {
    if (wide) return en == 3 ? launch_xgemm<3, true, true>(a, grid, s) : launch_xgemm<4, true, true>(a, grid, s);
    return en == 2 ? launch_xgemm<2, true, false>(a, grid, s) : launch_xgemm<4, true, false>(a, grid, s);
  }
  if (wide) return en == 3 ? launch_xgemm<3, false, true>(a, grid, s) : launch_xgemm<4, false, true>(a, grid, s);
  return en == 2 ? launch_xgemm<2, false, false>(a, grid, s) : launch_xgemm<4, false, false>(a, grid, s);
}

}  // namespace aussm
