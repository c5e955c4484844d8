// Argument blocks of the fused operator kernels (dropin.h), shared with the host side.
#pragma once
#include "scan_args.h"

namespace aussm {

constexpr int DT = 16;            // timesteps per tile
constexpr int D_MAXKS = 16;       // 32-wide steps of the contraction over r held in registers: d <= 512
constexpr int PHASE_HALF_KS = 3;  // from so many of them on the phase product takes two f16 pieces instead of three bf16 ones
constexpr int D_MAXN = 64;        // states per channel: up to four blocks of 16, one block per wavefront

struct DropinArgs {
  const float* u;        // [b, d, L]
  const float* dt;       // [b, d, L]
  const float* z;        // [b, d, L]
  const float* x_bias;   // [d, n]: element (i, j) at i xsi + j xsj
  const float* B_r;      // [n], consecutive states bcs elements apart
  const float* B_th;
  const float* C_r;
  const float* C_th;
  const float* Dp;       // [d]
  const float* h_re;     // [b, d, n] state before tile t0, or null: zero
  const float* h_im;
  float* y;              // [b, d, L] or null (states only)
  float* nh_re;          // [b, d, n] or null: state after tile t1 - 1 (may be the same buffer as h_*)
  float* nh_im;
  const u4* xp;          // rows of x as matrix operands: [d nb][ks][piece][64 lanes] (f16 pieces: 16 exponents behind each [ks])
  const u4* up;          // tiles of u, prefix-summed along the tile, as matrix operands: [b][tile - up_t0][KS][piece][64 lanes] (likewise)
  int up_b0, up_t0, up_nt;   // up holds the batch elements from up_b0 on and the tiles up_t0 .. up_t0 + up_nt - 1
  int b, d, n, L, ks;    // b: batch elements of this launch; ks = ceil(d / 32)
  int nb;                // blocks of 16 states per channel: 1, 2 or 4 (>= ceil(n / 16))
  int b0;                // first batch element of this launch (tensors are indexed by b0 + ...)
  int t0, t1;            // tiles of 16 timesteps of this launch (forward kernel; the backward kernel has its own)
  int xsi, xsj;          // row of (channel i, state j) in x, x_bias and the phase adjoints: i xsi + j xsj (n, 1 or 1, d)
  int bcs, raw;          // stride of the four polar parameters; raw: the radii are given before their softplus
  long zs;               // elements between the batch elements of z (d L for a tensor of its own)
  int nseg, sl;          // segments of sl tiles that the launch works on side by side (nseg 0 or 1: none, one sweep)
  f4* seg;               // [nseg][b][d][n] what a segment makes of the state: (E, F), h -> E h + F; backward (M, N), h -> M h + N towards the front
};

struct DropinBwdArgs {
  DropinArgs f;            // inputs (y, nh_* unused)
  const float* gy;         // [b, d, L]
  float* hc_re;            // [b, d, n] in: state after tile t1 - 1; out: state before tile t0
  float* hc_im;
  float* dth;              // workspace [bg][d n][lc]: phase adjoints of the launch
  float* du;               // [b, d, L] direct part (the product with x is added afterwards)
  float* ddt;
  float* dz;               // (batch elements f.zs apart)
  float* dxb;              // [d, n]   accumulated with atomics (zeroed by the host)
  float* dB_r;             // [n] each, accumulated with atomics
  float* dB_th;
  float* dC_r;
  float* dC_th;
  float* dD;               // [d]      (atomics)
  float* dh_re;            // [b, d, n] in: adjoint of the state after tile t1 - 1; out: of the state before tile t0
  float* dh_im;
  int b0, bg;              // batch elements b0 .. b0 + bg - 1 ...
  int t0, t1;              // ... and tiles of 16 timesteps t0 .. t1 - 1 (in reverse) are this launch's
  int lc;                  // row length of dth (>= 16 (t1 - t0))
  int dt_act;              // dt = softplus(pre): ddt is the gradient of pre, and ddtb [d] (or null) sums it (atomics)
  float* ddtb;
  float ddtb_scale;
  float2* sega;            // [nseg][bg][d][n] with nseg > 1: A of the adjoint, which becomes M hat h + A
  f4* ent;                 // [bg][d][n] ... and the state and the adjoint after tile t1 - 1 (hc_*, dh_* are written by the first segment)
};

// The pre-pass of a call: records of x (xblocks workgroups, 0: none) and the tiles t0 .. t0 + nt - 1 of u (ublocks)
struct DropinPrepArgs {
  const float* x;          // rows of d, (channel i, state j) at row i xsi + j xsj
  const float* x_bias;
  const float* u;          // [b, d, L]
  u4* xp;
  u4* up;
  float* x_out;            // scale x, and x_bias, in the operator's own order, or null
  float* xb_out;
  int d, n, L, ks, KS, nb, xsi, xsj;   // ks = ceil(d / 32), KS: compiled steps of the contraction
  int b0, t0, nt;
  float scale;
  unsigned xblocks, ublocks;
};

// Up to FILL_MAX buffers set in one launch: dst[i] = src ? src[i] : 0 for i < n.
constexpr int FILL_MAX = 16;
constexpr int FILL_BLOCK = 4096;    // floats per workgroup
struct FillArgs {
  float* dst[FILL_MAX];
  const float* src[FILL_MAX];
  unsigned long long n[FILL_MAX];
  int count;
};

}  // namespace aussm
