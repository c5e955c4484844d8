// Translation unit of the fused operator kernels (dropin.h).
#include "launch.h"
#include "dropin.h"

namespace aussm {

int run_fill(const FillArgs& a, hipStream_t s) {
  size_t most = 0;
  for (int i = 0; i < a.count; ++i) most = a.n[i] > most ? a.n[i] : most;
  const size_t blocks = (most + FILL_BLOCK - 1) / FILL_BLOCK;
  if (blocks > 0x7fffffffULL) return -2;
  if (!blocks) return 0;
  hipLaunchKernelGGL(fill_kernel, dim3((unsigned)blocks, (unsigned)a.count), dim3(256), 0, s, a);
  return launch_status();
}

#ifndef DROPIN_NW_
#define DROPIN_NW_ 8
#endif
constexpr int DROPIN_NW = DROPIN_NW_;     // channels (wavefronts) per workgroup

// (d > 256: the rows of x take up to 128 registers, in workgroups of four)
template <int KS, int NW>
static void launch_fwd_nw(const DropinArgs& a, hipStream_t s) {
  const unsigned grid = (unsigned)((a.nseg > 1 ? a.nseg : 1) * a.b * ((a.d * a.nb + NW - 1) / NW));
  hipLaunchKernelGGL((dropin_fwd_kernel<KS, NW>), dim3(grid), dim3(NW * 64), 0, s, a);
}
// Past two wavefronts on every SIMD 128 < d takes workgroups of four, four to a compute unit (dropin.h); up to there they
// would only read the tiles twice (8 x 250 x 16, 720 steps: 86 us in eights, 90 in fours; past it 20 x 256: 233, 174).
template <int KS>
static void launch_fwd(const DropinArgs& a, hipStream_t s) {
  if constexpr (KS > 8) {
    launch_fwd_nw<KS, 4>(a, s);
  } else if constexpr (KS > 4) {
    if ((a.nseg > 1 ? a.nseg : 1l) * a.b * a.d * a.nb > 256l * DROPIN_NW) launch_fwd_nw<KS, 4>(a, s);
    else launch_fwd_nw<KS, DROPIN_NW>(a, s);
  } else {
    launch_fwd_nw<KS, DROPIN_NW>(a, s);
  }
}
template <int KS>
static void launch_bwd(const DropinBwdArgs& a, hipStream_t s) {
  constexpr int NW = KS > 8 ? 4 : DROPIN_NW;
  const unsigned grid = (unsigned)((a.f.nseg > 1 ? a.f.nseg : 1) * a.bg * ((a.f.d * a.f.nb + NW - 1) / NW));
  hipLaunchKernelGGL((dropin_bwd_kernel<KS, NW>), dim3(grid), dim3(NW * 64), 0, s, a);
}
template <int KS>
static void launch_seg(const DropinBwdArgs& a, hipStream_t s) {
  constexpr int NW = KS > 8 ? 4 : DROPIN_NW;
  const unsigned grid = (unsigned)((a.f.nseg - 1) * a.bg * ((a.f.d * a.f.nb + NW - 1) / NW));
  if (a.sega) hipLaunchKernelGGL((dropin_seg_kernel<KS, NW, true>), dim3(grid), dim3(NW * 64), 0, s, a);
  else hipLaunchKernelGGL((dropin_seg_kernel<KS, NW, false>), dim3(grid), dim3(NW * 64), 0, s, a);
}

int dropin_channels_per_workgroup(int ks) { return ks > 8 ? 4 : DROPIN_NW; }

// the compiled size of the contraction (steps of 32) that serves ceil(d / 32) = ks
int dropin_compiled_ks(int ks) { return ks <= 4 ? (ks < 1 ? 1 : ks) : ks <= 6 ? 6 : ks <= 8 ? 8 : ks <= 12 ? 12 : 16; }

// 16-byte records of `steps` steps of 16 rows or columns (Phase in dropin.h), by the compiled size of the contraction
size_t dropin_records(int ks, int steps) {
  return dropin_compiled_ks(ks) >= PHASE_HALF_KS ? (size_t)steps * 2 * 64 + 4 : (size_t)steps * 3 * 64;
}

int run_dropin_prep(DropinPrepArgs a, int bg, bool rows, const FillArgs& f, hipStream_t s) {
  const size_t xb = rows ? (size_t)a.d * a.nb : 0, ub = (size_t)bg * a.nt;
  size_t total = xb + ub;
  for (int i = 0; i < f.count; ++i) total += (f.n[i] + FILL_BLOCK - 1) / FILL_BLOCK;
  if (total > 0x7fffffffULL) return -2;
  a.KS = dropin_compiled_ks(a.ks); a.xblocks = (unsigned)xb; a.ublocks = (unsigned)ub;
  hipLaunchKernelGGL(dropin_prep_kernel, dim3((unsigned)total), dim3(256), 0, s, a, f);
  return launch_status();
}

// compiled sizes of the contraction over r, in steps of 32: the smallest one >= ceil(d / 32) runs
#define DROPIN_KS_DISPATCH(LAUNCH, ks)          \
  if (ks <= 1) LAUNCH<1>(a, s);                 \
  else if (ks <= 2) LAUNCH<2>(a, s);            \
  else if (ks <= 3) LAUNCH<3>(a, s);            \
  else if (ks <= 4) LAUNCH<4>(a, s);            \
  else if (ks <= 6) LAUNCH<6>(a, s);            \
  else if (ks <= 8) LAUNCH<8>(a, s);            \
  else if (ks <= 12) LAUNCH<12>(a, s);          \
  else LAUNCH<16>(a, s);

int run_dropin_fwd(const DropinArgs& a, hipStream_t s) {
  DROPIN_KS_DISPATCH(launch_fwd, a.ks)
  return launch_status();
}

int run_dropin_seg(const DropinBwdArgs& a, hipStream_t s) {
  DROPIN_KS_DISPATCH(launch_seg, a.f.ks)
  return launch_status();
}

int run_dropin_bwd(const DropinBwdArgs& a, hipStream_t s) {
  DROPIN_KS_DISPATCH(launch_bwd, a.f.ks)
  return launch_status();
}

}  // namespace aussm
