// Translation unit of the fp32-accurate GEMM (gemm.h).
#include "gemm.h"
#include "launch.h"

namespace aussm {

template <int WM, int EM, int EN, bool QUAD>
static int launch_tile(const XGemmArgs& a, unsigned grid, hipStream_t s) {
  constexpr bool WIDE = WM == 4;
  const bool ak1 = a.sak == 1, bk1 = a.sbk == 1, tr = a.scm == 1 && a.scn != 1;
#define XG(A_, B_, T_)                                                                       \
  if (ak1 == A_ && bk1 == B_ && tr == T_) {                                                  \
    hipLaunchKernelGGL((xgemm_kernel<A_, B_, T_, WM, EM, EN, QUAD, WIDE>), dim3(grid), dim3(WIDE ? 512 : 256), 0, s, a);     \
    return launch_status();                                                                  \
  }
  XG(false, false, false) XG(false, false, true) XG(false, true, false) XG(false, true, true)
  XG(true, false, false) XG(true, false, true) XG(true, true, false) XG(true, true, true)
#undef XG
  return -2;
}

struct Tile { int wm, em, en; };        // wavefronts along the rows; 16-wide row and column tiles per wavefront
constexpr int rows_of(const Tile& t) { return 16 * t.em * t.wm; }
constexpr int cols_of(const Tile& t) { return 16 * t.en * (t.wm == 4 ? 2 : 4 / t.wm); }
constexpr Tile NARROW{2, 4, 4}, COLS64{2, 4, 2}, COLS32{2, 4, 1}, ROWS64{1, 4, 2}, ROWS32{1, 2, 2}, WIDE128{4, 4, 4}, WIDE96{4, 4, 3};

template <bool QUAD>
static int launch_xgemm(const Tile& t, const XGemmArgs& a, unsigned grid, hipStream_t s) {
#define XT(T_) if (t.wm == T_.wm && t.em == T_.em && t.en == T_.en) return launch_tile<T_.wm, T_.em, T_.en, QUAD>(a, grid, s);
  XT(NARROW) XT(COLS64) XT(COLS32) XT(ROWS64) XT(ROWS32) XT(WIDE128) XT(WIDE96)
#undef XT
  return -2;
}

// Tiles of few rows or few columns where the product has no more: the matrix instructions and the staging of a 128-row
// tile would mostly work on repeated rows.  (Columns 23040, K = 512: 48 rows 39 -> 30 us, 16 rows 42 -> 27 us; 32 rows,
// 11264 columns, K = 2048 in slices 44 -> 28 us; 2048 x 32, sums of 11264, 28 -> 23 us.)
// Else the wide ones for more rows than the narrow one has, by the rounds that the tiles make on the chip (256 compute
// units, one wide or two narrow workgroups each) times what a round takes: 1 for 256 x 128, 0.88 for 256 x 96, 1.2 for two of
// 128 x 128, 0.72 for one.  23040 columns, us narrow / 96 / 128: 256 rows, K = 1024 93 / 70 / 78; 512 rows, K = 256 46 / 43 /
// 50; 1024 rows, K = 256 77 / 80 / 73; 512 rows, K = 16 17.1 / 17.1 / 19.2.
//
// Slices: a sum over many steps with few tiles is cut into as many workgroups as run at once (more would start a second
// round: 540 workgroups 140 us, 450 workgroups 91 us for the product with 90 tiles and 128 steps), at least four steps of
// 32 per slice (shorter ones would spend their time on the atomics of the tile).  The wide tile from 24 steps a slice on:
// 4096 x 256, sums of 23040, 281 -> 248 us; 256 x 5760, K = 4096 93 -> 81 us; 512 x 256 (12 steps) 56 against 58 us.
int run_xgemm(XGemmArgs a, hipStream_t s) {
  if (a.M < 1 || a.N < 1 || a.K < 1 || a.Z < 1 || a.nper < 1) return -2;
  if (a.reduce && a.scm == 1 && a.scn != 1 && a.nper < a.N) return -2;
  const long steps = (long)((a.K + 31) / 32) * a.Z;
  const bool sliced = a.reduce && !a.bias && !a.add && !a.act;
  auto tiles_of = [&](const Tile& t) { return (long)((a.M + rows_of(t) - 1) / rows_of(t)) * ((a.N + cols_of(t) - 1) / cols_of(t)); };
  Tile tile = a.N <= 32 ? COLS32 : a.N <= 64 ? COLS64 : a.M <= 32 ? ROWS32 : a.M <= 64 ? ROWS64 : NARROW;
  if (a.M > rows_of(NARROW) && a.N > 64) {
    if (sliced) {
      const long t = tiles_of(WIDE128);
      if (steps >= 24 * (t < 256 ? 256 / t : 1)) tile = WIDE128;
    } else {
      auto rounds = [](long t, long slots) { return (double)((t + slots - 1) / slots); };
      const double w4 = rounds(tiles_of(WIDE128), 256), w3 = 0.88 * rounds(tiles_of(WIDE96), 256);
      const long t = tiles_of(NARROW);
      const double narrow = 1.2 * (double)(t / 512) + (t % 512 > 256 ? 1.2 : t % 512 ? 0.72 : 0.0);
      if (w3 < narrow || w4 < narrow) tile = w3 < w4 ? WIDE96 : WIDE128;
    }
  }
  const long tiles = tiles_of(tile);
  long sl = 1;
  if (sliced) {
    sl = (tile.wm == 4 ? 256 : 512) / tiles;
    if (sl > steps / 4) sl = steps / 4;
    if (sl < 1) sl = 1;
    const long per = (steps + sl - 1) / sl;
    sl = (steps + per - 1) / per;
  }
  if (steps > 0x7fffffffL || tiles * sl > 0x7fffffffL) return -2;
  a.slices = (int)sl;
  if (a.scm < 0 || a.scn < 0) return -2;
  const unsigned grid = (unsigned)(tiles * sl);
  return a.K % 4 == 0 ? launch_xgemm<true>(tile, a, grid, s) : launch_xgemm<false>(tile, a, grid, s);
}

}  // namespace aussm
