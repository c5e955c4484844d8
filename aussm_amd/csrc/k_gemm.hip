// Translation unit of the fp32-accurate GEMM (gemm.h).
#include "gemm.h"
#include "launch.h"

namespace aussm {

template <int NW, int WM, int EM, int EN, bool QUAD, bool HALF>
static int launch_tile(const XGemmArgs& a, unsigned grid, hipStream_t s) {
  const bool ak1 = a.sak == 1, bk1 = a.sbk == 1, tr = a.scm == 1 && a.scn != 1;
#define XG(A_, B_, T_)                                                                       \
  if (ak1 == A_ && bk1 == B_ && tr == T_) {                                                  \
    hipLaunchKernelGGL((xgemm_kernel<A_, B_, T_, NW, WM, EM, EN, QUAD, HALF>), dim3(grid), dim3(64 * NW), 0, s, a);     \
    return launch_status();                                                                  \
  }
  XG(false, false, false) XG(false, false, true) XG(false, true, false) XG(false, true, true)
  XG(true, false, false) XG(true, false, true) XG(true, true, false) XG(true, true, true)
#undef XG
  return -2;
}

struct Tile { int nw, wm, em, en; };    // wavefronts, of them along the rows; 16-wide row and column tiles per wavefront
constexpr int rows_of(const Tile& t) { return 16 * t.em * t.wm; }
constexpr int cols_of(const Tile& t) { return 16 * t.en * (t.nw / t.wm); }
constexpr Tile NARROW{4, 2, 4, 4}, COLS64{4, 2, 4, 2}, COLS32{4, 2, 4, 1}, ROWS32{4, 1, 2, 2}, WIDE128{8, 4, 4, 4}, WIDE96{8, 4, 4, 3};
constexpr Tile T64{4, 2, 2, 2}, R32C64{4, 1, 2, 1}, R64C32{4, 2, 2, 1}, T32{4, 2, 1, 1};       // 64 x 64, 32 x 64, 64 x 32, 32 x 32

template <bool QUAD, bool HALF>
static int launch_xgemm(const Tile& t, const XGemmArgs& a, unsigned grid, hipStream_t s) {
#define XT(T_) if (t.nw == T_.nw && t.wm == T_.wm && t.em == T_.em && t.en == T_.en) return launch_tile<T_.nw, T_.wm, T_.em, T_.en, QUAD, HALF>(a, grid, s);
  XT(NARROW) XT(COLS64) XT(COLS32) XT(ROWS32) XT(T64) XT(R32C64) XT(R64C32) XT(T32)
  if constexpr (HALF) { XT(WIDE128) XT(WIDE96) }
#undef XT
  return -2;
}

// f16 pieces: offsets of 32 bits inside a tile, whatever its position, and along k (XgHalfOperand)
static bool near(const XGemmArgs& a) {
  constexpr long most = 1l << 28, rows = 256;              // elements; a tile's rows or columns, at most
  auto fits = [](long n, long stride) { return stride >= 0 && (stride == 0 || n < most / stride); };
  return fits(rows, a.sam) && fits(a.K, a.sak) && fits(a.K, a.sbk) && fits(a.nper < a.N ? a.nper : rows, a.sbn) &&
         (a.nper >= a.N || fits(rows / a.nper + 2, a.sbb));
}

// Small tiles where a product has few of them.  What a step of 32 costs a workgroup is mostly waiting - for the values, for the
// other wavefronts -, 2.3 us with 128 x 128, 1.4 with 64 x 64, 0.95 with 32 x 32, so a product that leaves the chip
// part empty is done sooner in many small ones: the smallest tile of which there are at most 256, else 64 x 64 up to 1024 of
// them.  us, 128-wide tile / the one taken: 256 x 5760, K = 1024 74 / 45; 1000 x 1000, K = 250 31 / 16; 137 x 1008, K = 548
// 51 / 20; 384 x 954, K = 96 23 / 7.4; 54 x 1320, K = 27 11 / 5.1; 48 x 23040, K = 512 30 / 24; 16 x 131072, K = 32 9.3 with 32 x 64, 8.0
// with 32 x 128; 512 x 8192, K = 256 (1024 tiles of 64 x 64) 23.9 / 23.2, 1024 x 8192 (2048) 27.4 with the wide tile against 34.8.  Sums over z alike, by the work there is:
// 64 x 64 up to 18000 tile steps, past 8000 in twice the slices (512 x 128, 512 steps 56 / 27; 96 x 192, 30 steps 20 / 6.8;
// 142 x 3960, 71 steps, 13206 of them: 42 / 39, 53 in half the slices; 200 x 3000, 100 steps, 18800: 51 / 50), where rows of K that do
// not start on 16 bytes cost the small tile's loads more to 6000 (2272 x 142, 50 steps of 791, 5400: 41 / 38; 75 steps, 8100: 48 / 54), for 32 columns or rows up to 4500 (512 x 16, 736 steps, 5900:
// 13.7 against 15.0; 256 x 16 11.8 / 10.0).  Past that few rows take 32 x 128 (32 x 32768, sums of 2048: 62, 128 x 128 111), or 64 x 64
// and twice the slices (64 x 23040, 1024: 34.7, with 64 x 128 42.6; 64 x 32768, 4096: 156, 151).
//
// Else the wide ones for more rows than the narrow one has, by the rounds that the tiles make on the chip (256 compute
// units, one wide or two narrow workgroups each) times what a round takes: 1 for 256 x 128, 0.9 for 256 x 96, 1.2 for two of
// 128 x 128, 0.72 for one.  23040 columns, us narrow / 96 / 128: 256 rows, K = 1024 66 / 57 / 59; K = 512 41 / 34 / 38; 512 rows, K = 256
// 39 / 39 / 42; 1024 rows, K = 256 68 / 77 / 65.
//
// Slices: a sum over many steps with few tiles is cut into as many workgroups as run at once (more would start a second
// round: 540 workgroups 140 us, 450 workgroups 91 us for the product with 90 tiles and 128 steps), at least four steps of
// 32 per slice (shorter ones would spend their time on the atomics of the tile), of small tiles two unless four leave 200
// workgroups (548 x 137, 36 steps: 10.2 against 11.7 us; 96 x 192, 30 steps: 9.6 against 6.8).  The wide tile from 24 steps a
// slice on: 4096 x 256, sums of 23040, 281 -> 248 us; 256 x 5760, K = 4096 93 -> 81 us; 512 x 256 (12 steps) 56 against 58 us.
//
// f16 pieces from six steps a workgroup on, from eight in the tiles of 32 x 32 to 64 x 32: finding the scales costs 1 to 2 us.  us bf16 / f16:
// 256 x 256 in tiles of 32 x 32, K = 128 5.2 / 6.0, 192 6.5 / 6.8, 256 7.9 / 7.7, 512 13.3 / 11.0; 512 x 2048 in tiles of 64 x 64, K = 128 7.8 / 8.4,
// 192 9.7 / 9.6, 512 20.0 / 15.9; 256 x 23040, K = 1024 77 / 57; 256 x 5760, K = 4096 91 / 70; 4096 x 256, sums of 5760 84 / 67.
// Sums of up to 64 terms, which are more exact on three bf16 pieces, never get there.
int run_xgemm(XGemmArgs a, hipStream_t s) {
  if (a.M < 1 || a.N < 1 || a.K < 1 || a.Z < 1 || a.nper < 1) return -2;
  if (a.reduce && a.scm == 1 && a.scn != 1 && a.nper < a.N) return -2;
  const long steps = (long)((a.K + 31) / 32) * a.Z;
  const bool can_half = near(a);
  const bool sliced = a.reduce && !a.bias && !a.add && !a.act;
  auto tiles_of = [&](const Tile& t) { return (long)((a.M + rows_of(t) - 1) / rows_of(t)) * ((a.N + cols_of(t) - 1) / cols_of(t)); };
  Tile tile = a.N <= 32 ? COLS32 : a.N <= 64 ? COLS64 : NARROW;
  bool small = true;
  int slots = 512;
  const Tile pair = tiles_of(R64C32) < tiles_of(R32C64) ? R64C32 : R32C64;
  if (sliced) {
    if (a.M <= 32 && a.N <= 32) tile = T32;
    else if ((a.M <= 32 || a.N <= 32) && tiles_of(pair) * steps <= 4500) tile = pair;
    else if (a.M > 32 && a.N > 32 && tiles_of(T64) * steps <= (a.K % 4 ? 6000 : 18000)) {
      tile = T64;
      if (tiles_of(T64) * steps > 8000) slots = 1024;
    }
    else if (a.M <= 32 && a.N > 64) tile = ROWS32;
    else if (a.M <= 64 && a.N > 64) tile = T64, slots = 1024;
    else small = false;
  } else {
    if (tiles_of(T32) <= 256) tile = T32;
    else if (tiles_of(pair) <= 256) tile = pair;
    else if (a.M <= 32) tile = tiles_of(pair) <= 512 ? pair : ROWS32;
    else if (tiles_of(T64) <= 1024 || a.M <= 64) tile = T64;
    else small = false;
  }
  if (can_half && steps >= 6 && !small && a.M > rows_of(NARROW) && a.N > 64) {
    if (sliced) {
      const long t = tiles_of(WIDE128);
      if (steps >= 24 * (t < 256 ? 256 / t : 1)) tile = WIDE128;
    } else {
      auto rounds = [](long t, long slots) { return (double)((t + slots - 1) / slots); };
      const double w4 = rounds(tiles_of(WIDE128), 256), w3 = 0.9 * rounds(tiles_of(WIDE96), 256);
      const long t = tiles_of(NARROW);
      const double narrow = 1.2 * (double)(t / 512) + (t % 512 > 256 ? 1.2 : t % 512 ? 0.72 : 0.0);
      if (w3 < narrow || w4 < narrow) tile = w3 < w4 ? WIDE96 : WIDE128;
    }
  }
  const long tiles = tiles_of(tile);
  long sl = 1, per = steps;
  if (sliced) {
    sl = (tile.nw == 8 ? 256 : slots) / tiles;
    const long least = small && tiles * (steps / 4) < 200 ? 2 : 4;
    if (sl > steps / least) sl = steps / least;
    if (sl < 1) sl = 1;
    per = (steps + sl - 1) / sl;
    sl = (steps + per - 1) / per;
  }
  const bool half = can_half && per >= (tile.em * tile.en <= 2 ? 8 : 6);
  if (steps > 0x7fffffffL || tiles * sl > 0x7fffffffL) return -2;
  a.slices = (int)sl;
  if (a.scm < 0 || a.scn < 0) return -2;
  const unsigned grid = (unsigned)(tiles * sl);
  if (half) return a.K % 4 == 0 ? launch_xgemm<true, true>(tile, a, grid, s) : launch_xgemm<false, true>(tile, a, grid, s);
  return a.K % 4 == 0 ? launch_xgemm<true, false>(tile, a, grid, s) : launch_xgemm<false, false>(tile, a, grid, s);
}

}  // namespace aussm
