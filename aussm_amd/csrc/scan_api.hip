// C ABI of libaussm_hip.so: argument checks, kernel selection and launches.
// Declarations and tensor layouts: include/aussm_hip.h.
#include "../../include/aussm_hip.h"

#include <hip/hip_runtime.h>
#include <atomic>

#include "launch.h"
#include "scan_args.h"

using namespace aussm;

namespace {

// Process-wide options (aussm_set_option): kernel selection for comparisons and tuning.  They are
// plain atomics read once per call; -1 means "let the launcher decide".
std::atomic<int> g_opt[AUSSM_OPT_COUNT] = {{-1}, {-1}, {-1}, {-1}, {-1}, {-1}};
static_assert(AUSSM_OPT_COUNT == 6, "one initialiser per option");
inline int opt(int key) { return g_opt[key].load(std::memory_order_relaxed); }

// ---- configuration of unitary_bwd_kernel (33 to 64 states): eight wavefronts of eight states, unless the options force the four
// of sixteen (two wavefronts on a SIMD hide each other's scalar loads: 64 states 10 % faster)
inline Cfg pick_cfg() {
  return opt(AUSSM_OPT_GENERIC_NW) == 16 && opt(AUSSM_OPT_GENERIC_NT) == 256 ? Cfg{16, 256} : Cfg{8, 512};
}

// flags that the backward entry points take beside the input type
inline int take_flag(int& in_dtype, int flag) {
  const int f = in_dtype & flag;
  in_dtype &= ~flag;
  return f != 0;
}

inline int check_common(int B, int D, int N, int L, int ck, int in_dtype) {
  if (B < 1 || D < 1 || N < 1 || L < 1) return AUSSM_E_SHAPE;
  if (N > AUSSM_MAX_STATE) return AUSSM_E_SHAPE;
  if ((long long)B * ((D + CH - 1) / CH) > 0x7fffffffLL) return AUSSM_E_SHAPE;
  if (ck != AUSSM_TILE / 2 && (ck < AUSSM_TILE || ck % AUSSM_TILE != 0)) return AUSSM_E_CK;
  if (in_dtype != AUSSM_F32 && in_dtype != AUSSM_BF16) return AUSSM_E_DTYPE;
  return AUSSM_OK;
}

// Checkpoint interval of the recomputing backward kernels (complex, real)
constexpr int REC_CK = AUSSM_TILE / 2;

// A state handed out over the one handed in: such a call is not split along the sequence, since its first segments would still
// read what its last one writes (the adjoint of the state alike).
inline bool overlap(const float* p, const float* q, size_t n) { return p && q && p < q + n && q < p + n; }
inline bool misaligned(const void* p, size_t a) { return p && (reinterpret_cast<uintptr_t>(p) % a) != 0; }

// The matrix-core kernels cover the common unitary case (fp32 or bf16 inputs, 6 <= N <= 16, L a multiple of 4,
// 16-byte aligned tensors, checkpoint interval a multiple of 32); everything else takes the
// vector-ALU kernels.  aussm_set_option(AUSSM_OPT_UNITARY_FWD, m) selects the forward kernel for
// comparisons: 0 vector ALU, 2 / 3 bf16 matrix instructions on two- / three-piece operands built
// inside the scan kernel, 6 three-piece operands prepared by a pre-pass, two wavefronts per SIMD
// (the default when the call brings the workspace for them, i.e. an auxiliary buffer).
// AUSSM_OPT_UNITARY_BWD: 0 vector ALU, 2 two pieces everywhere, 3 three pieces along the sequence
// and two in the sums over the channel (dB, dC), 5 three pieces everywhere, 6 prepared operands.
//
// By time alone the matrix-core kernels would take every N: us, vector ALU / matrix cores, forward and backward pass and forward
// alone, 32 x 512 channels of 2048 steps: N = 2 591 / 526, 194 / 161; 4 595 / 535, 197 / 160; 6 603 / 546, 197 / 161; 8 603 / 553,
// 193 / 164; 8 x 256 of 1024: N = 4 97 / 90, 26.2 / 24.4; 8 96 / 93, 26.0 / 25.4.  But they take the channel sums behind dB and dC
// in two pieces, 4.6e-6 of their norm from a float64 scan where the vector ALU's are 1.1e-6 (2 x 64 x 4, 2048 steps; the other
// results agree to 20 %), so calls of fewer states, which the vector ALU has always served, stay there.  (The line is where the two
// took the same time when it was drawn.)
constexpr int MATRIX_MIN_STATE = 6;
constexpr int DEFAULT_FWD_MODE = 6, DEFAULT_BWD_MODE = 6;   // (6 falls back to 3 where the call brings no workspace)
inline int kernel_mode(int key, int dflt, int N) {
  const int e = opt(key);
  if (e >= 0) return e;                        // an explicit choice is honoured for every N <= 16
  return N >= MATRIX_MIN_STATE ? dflt : 0;
}
// Splitting the sequence (scan_seg_xdl.h): with few (batch, channel group) pairs the launch would
// leave most of the chip idle, so the sequence is cut into ns segments of whole checkpoint blocks
// until about one workgroup per compute unit exists: here in equal ones by halving, below in others (unitary_split), on the
// vector-ALU kernels by generic_split.  The segment states live behind the auxiliary buffer or in the call's workspace;
// aussm_unitary_fwd_static has room for equal segments only.
// aussm_set_option(AUSSM_OPT_SPLIT_CAP, c): 0 or 1 switches it off, more caps ns.
constexpr int SPLIT_MIN_WGS = 129;     // launches of at least this many workgroups are left alone
constexpr int SPLIT_TARGET_WGS = 256;
constexpr int SPLIT_MAX = 32;
constexpr int SPLIT_MIN_LEN = 128;
constexpr int GSPLIT_MAX = 64;         // segments of unequal runs of blocks, of the vector-ALU kernels' split
inline bool matrix_shape(int N, int L, int ck) { return N <= XN && L % 4 == 0 && ck >= XT && ck % XT == 0; }
inline int seg_capacity(int B, int D, int N, int L, int ck) {
  if (N < MATRIX_MIN_STATE || !matrix_shape(N, L, ck) || L % ck != 0) return 1;
  const long long wgs = (long long)B * ((D + CH - 1) / CH);
  if (wgs >= SPLIT_MIN_WGS) return 1;
  const int nblk = L / ck, target = (int)(SPLIT_TARGET_WGS / wgs);
  int ns = 1;
  while (ns * 2 <= target && ns * 2 <= SPLIT_MAX && nblk % (ns * 2) == 0 && L / (ns * 2) >= SPLIT_MIN_LEN) ns *= 2;
  return ns;
}
// The segment states are computed on finer segments than the scan proper uses (the kernel that
// forms them is light: several workgroups per compute unit hide its latencies); the scan takes
// every SPLIT_FINE-th of them.
inline int seg_fine(int L, int ns) {
  const int Ls = L / ns;
  for (int r = 4; r > 1; r /= 2)
    if (Ls % (r * XT) == 0 && Ls / r >= SPLIT_MIN_LEN) return r;
  return 1;
}
// Segments of a call on the matrix-core kernels: ns of ls steps (whole checkpoint blocks, the last one possibly shorter),
// each of r fine ones, nf fine ones per sequence.  Sequences that halve into equal segments do so (seg_capacity).  Others -
// a length that is no multiple of the checkpoint interval, a number of blocks that is no power of two - take as many equal
// runs of blocks as bring the launch near one workgroup per compute unit, where that makes at least twice as many segments;
// their fine segments are the segments, so that the states fit the area the vector-ALU kernels' split needs
// (generic_split: as many segments or more).  B6 D28 N16 L11312, bf16, training pass: 1918 us on 6 workgroups.
struct USplit { int ns, ls, r, nf; };
// room: floats there are for the states of unequal segments.
inline USplit unitary_split(int B, int D, int N, int L, int ck, bool use_cap, size_t room = ~(size_t)0) {
  const USplit whole{1, L, 1, 1};
  const int cap = use_cap ? opt(AUSSM_OPT_SPLIT_CAP) : -1;
  if (cap == 0 || cap == 1 || N < MATRIX_MIN_STATE || !matrix_shape(N, L, ck)) return whole;
  int ns = seg_capacity(B, D, N, L, ck);
  const int fine = ns * seg_fine(L, ns);
  if (cap > 1)
    while (ns > 1 && ns > cap) ns /= 2;
  const long long wgs = (long long)B * ((D + CH - 1) / CH);
  if (wgs < SPLIT_MIN_WGS && L >= 4 * SPLIT_MIN_LEN) {
    const int nblk = (L + ck - 1) / ck;
    int want = (int)(SPLIT_TARGET_WGS / wgs);
    if (want > GSPLIT_MAX) want = GSPLIT_MAX;
    if (cap > 1 && want > cap) want = cap;
    int bps = (nblk + want - 1) / want;
    if (bps * ck < SPLIT_MIN_LEN) bps = (SPLIT_MIN_LEN + ck - 1) / ck;
    const int nr = (nblk + bps - 1) / bps;
    if (nr >= 2 * ns && (size_t)B * nr * D * (2 * N + 2) <= room) return USplit{nr, bps * ck, 1, nr};
  }
  if (ns <= 1) return whole;
  int r = seg_fine(L, ns);
  // (no more fine ones than the area is sized for - fewer segments by option -, and few: a workgroup of the scan walks those
  // ahead of its segment.  B4 D256 N16 L16384 training pass with 64 / 32 / 16 of them 435 / 415 / 422 us, B8 L4096 with
  // 32 / 16 / 8 212 / 198 / 201, B2 L8192 with 64 / 32 136 / 124)
  while (r > 1 && (ns * r > fine || r > 2 || ns * r > 32)) r /= 2;
  return USplit{ns, L / ns, r, ns * r};
}
inline size_t round64(size_t n) { return (n + 63) & ~(size_t)63; }
inline size_t seg_floats(int B, int D, int N, int L, int ns) {
  return ns > 1 ? round64((size_t)B * ns * seg_fine(L, ns) * D * (2 * N + 2)) : 0;
}
// The complex and the real scan split the same way (scan_oct.h) when the call brings a workspace:
// ns segments of ls steps (whole tiles and checkpoint blocks), the last one possibly shorter.
// (segments of 64 steps, forward passes, us: S6 B1 D512 L300 28 -> 20 against 128, B2 D64 L256 27 -> 19; sequences of fewer than
// 256 steps stay whole: what is left to gain there is less than the launches of the first pass cost)
constexpr int GSPLIT_MIN_LEN = 64, GSPLIT_FROM = 256;
struct GSplit { int ns, ls; };
inline GSplit generic_split(int B, int D, int L, int ck, bool use_cap) {
  const long long wgs = (long long)B * ((D + CH - 1) / CH);
  const int cap = use_cap ? opt(AUSSM_OPT_SPLIT_CAP) : -1;
  if (wgs >= SPLIT_MIN_WGS || L < GSPLIT_FROM || cap == 0 || cap == 1) return GSplit{1, L};
  int want = (int)((SPLIT_TARGET_WGS + wgs - 1) / wgs);
  if (want > GSPLIT_MAX) want = GSPLIT_MAX;
  if (cap > 1 && want > cap) want = cap;
  const int unit = ck > XT ? ck : XT;
  int ls = ((L + want - 1) / want + unit - 1) / unit * unit;
  if (ls < GSPLIT_MIN_LEN) ls = (GSPLIT_MIN_LEN + unit - 1) / unit * unit;
  const int ns = (L + ls - 1) / ls;
  return ns > 1 ? GSplit{ns, ls} : GSplit{1, L};
}
inline size_t generic_split_floats(int variant, int B, int D, int N, int L, int ck) {
  const GSplit sp = generic_split(B, D, L, ck, false);
  const int C = variant == VAR_REAL ? 1 : 2;
  return sp.ns > 1 ? round64((size_t)B * sp.ns * D * (N * C + 2)) : 0;
}
// (bf16 inputs: the kernels read B_t / C_t as they are; the room for float copies of them stays part of the size that callers
// allocate by, and of what a call without a workspace is refused for)
inline size_t generic_bc_floats(int variant, int B, int N, int L, int in_dtype) {
  return in_dtype == AUSSM_BF16 ? round64((size_t)B * N * L * (variant == VAR_REAL ? 1 : 2)) : 0;
}

// Workspace of the prepared operands: per (batch element, chunk) one backward image and, behind
// all of those, one forward image.  The forward call of a training step writes both (one pre-pass);
// a backward call whose auxiliary buffer does not hold the images of its own tensors writes its own.
// The size does not depend on the option table: a buffer sized under one set of options fits every other.
inline size_t img_chunks(int B, int L) { return (size_t)B * ((L + XT - 1) / XT); }
inline size_t img_floats(int B, int N, int L, int ck) {
  if (!matrix_shape(N, L, ck)) return 0;
  return img_chunks(B, L) * (PXB_REC + PXF_REC) * 4;
}
// Layout of the auxiliary buffer: [B*D*L floats Im(P S)] [AUX_PAD] [segment states] [backward images] [forward images].
// A shape that only the vector-ALU kernels serve (more than 16 states, a length that is not a multiple of 4, ...)
// has no Im(P S) part and no images.  The segment area holds what either way of splitting a call along L
// needs (the matrix-core kernels' fine segments or the vector-ALU kernels' segments), so a call of a shape
// that could run on the matrix cores but does not (shared inputs, misaligned tensors, an option) can still split.
inline size_t aux_im_floats(int B, int D, int N, int L, int ck) { return matrix_shape(N, L, ck) ? (size_t)B * D * L : 0; }
inline size_t aux_seg_floats(int B, int D, int N, int L, int ck) {
  const size_t m = seg_floats(B, D, N, L, seg_capacity(B, D, N, L, ck)), g = generic_split_floats(VAR_COMPLEX, B, D, N, L, ck);
  return m > g ? m : g;
}
struct AuxLayout { float* seg; u4* img; u4* fimg; uint32_t* stamp; float* pad; float* gseg; size_t seg_room; };
inline AuxLayout aux_layout(float* aux, int B, int D, int N, int L, int ck) {
  if (!aux) return AuxLayout{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0};
  float* pad = aux + aux_im_floats(B, D, N, L, ck);
  float* seg = pad + AUX_PAD;
  u4* img = reinterpret_cast<u4*>(seg + aux_seg_floats(B, D, N, L, ck));
  if (!img_floats(B, N, L, ck)) return AuxLayout{seg, nullptr, nullptr, nullptr, pad, seg, aux_seg_floats(B, D, N, L, ck)};
  return AuxLayout{seg, img, img + img_chunks(B, L) * PXB_REC, reinterpret_cast<uint32_t*>(pad) + AUX_IMG_FP, pad, seg,
                   aux_seg_floats(B, D, N, L, ck)};
}

// Kernel family of a call whose tensors are 16-byte aligned: 0 vector ALU, 2 / 3 / 5 matrix-core kernels
// that prepare their operands themselves, 6 prepared-operand kernels.
inline int fwd_mode_for(int N, int L, int ck, int in_dtype, int urep, bool have_img) {
  int mode = kernel_mode(AUSSM_OPT_UNITARY_FWD, DEFAULT_FWD_MODE, N);
  if (mode <= 0 || urep != 1 || !matrix_shape(N, L, ck)) return 0;
  if (mode == 6 && !have_img) mode = 3;
  if (in_dtype != AUSSM_F32 && mode != 6) mode = 3;       // bf16 inputs: three-piece kernels only
  return mode;
}
inline int bwd_mode_for(int B, int D, int N, int L, int ck, int urep, bool have_img) {
  int mode = kernel_mode(AUSSM_OPT_UNITARY_BWD, DEFAULT_BWD_MODE, N);   // matrix-core kernels for the common case
  if (mode <= 0 || urep != 1 || !matrix_shape(N, L, ck)) return 0;
  // (the prepared-operand kernel addresses its tensors with 32-bit byte offsets)
  if (mode == 6 && (!have_img || (unsigned long long)B * D * L * 4 >= (1ull << 32) ||
                    (unsigned long long)B * N * L * 8 >= (1ull << 32)))
    mode = 3;
  return mode;
}
inline int mfma_fwd_mode(const FwdArgs& a, int in_dtype, bool have_img) {
  const int mode = fwd_mode_for(a.N, a.L, a.ck, in_dtype, a.urep, have_img);
  if (misaligned(a.u, 16) || misaligned(a.delta, 16) || misaligned(a.theta, 16) || misaligned(a.z, 16) ||
      misaligned(a.y, 16) || misaligned(a.Bm, 16) || misaligned(a.Cm, 16))
    return 0;
  return mode;
}

// ws: workspace of the call (segment states for a launch that is split along L, images of the
// prepared operands); either part may be null.
int launch_unitary_fwd(FwdArgs a, int in_dtype, hipStream_t s, AuxLayout ws) {
  const int mode = mfma_fwd_mode(a, in_dtype, ws.img != nullptr);
  // Im(P S) is only worth writing when a backward call can follow (it needs the checkpoints too);
  // a call that does not fill the buffer marks it as not filled, and a call that does not prepare
  // images clears the note about the ones behind the buffer
  const bool fill = a.aux && a.hck && mode >= 2;
  // (the prepared-operand kernel clears the fill tag itself, at its end: one launch less for a forward-only call)
  const bool clear_in_kernel = a.aux && !fill && mode == 6;
  // (the vector-ALU kernels do that too, at theirs)
  if (a.aux && mode)
    if (int e = run_aux_invalidate(ws.pad, !fill && !clear_in_kernel, mode != 6 && ws.stamp, s)) return e;
  const bool had_aux = a.aux != nullptr;
  if (!fill) a.aux = nullptr;
  const bool in_place = overlap(a.h0, a.hL, (size_t)a.B * a.D * a.N * 2);
  if (!mode) {
    // vector-ALU kernel; with a segment area and few (batch, channel group) pairs, split along the sequence
    const GSplit sp = ws.gseg && !in_place ? generic_split(a.B, a.D, a.L, a.ck, true) : GSplit{1, a.L};
    if (sp.ns > 1) {
      const int B = a.B;
      float* seg = ws.gseg;
      float* ptot = seg + (size_t)B * sp.ns * a.D * a.N * 2;
      // 1. end state of every segment from a zero state (no outputs) and the product of its a_l
      FwdArgs z = a;
      z.B = B * sp.ns; z.L = sp.ls; z.ns = sp.ns;
      z.y = nullptr; z.z = nullptr; z.Dskip = nullptr; z.h0 = nullptr; z.hL = seg; z.hck = nullptr; z.ptot = ptot;
      if (int e = run_oct_fwd(VAR_UNITARY, z, in_dtype, s)) return e;
      // 2. the scan proper over (batch, segment) pairs, each from what those before it make of the state
      a.B = B * sp.ns; a.L = sp.ls; a.ns = sp.ns; a.seg = seg; a.segq = ptot;
    }
    a.clear = had_aux ? ws.pad : nullptr;
    return run_oct_fwd(VAR_UNITARY, a, in_dtype, s);
  }
  const int B = a.B, L = a.L;
  SegArgs sa{};
  unsigned nseg = 0;                           // workgroups of the segment-state pass, run with the pre-pass (mode 6)
  if ((mode == 2 || mode == 3 || mode == 6) && ws.seg && !in_place) {
    const USplit sp = unitary_split(B, a.D, a.N, L, a.ck, true, ws.seg_room);
    if (sp.ns > 1) {
      // 1. end state of every segment from a zero start and its rotation; 2. the scan proper over (batch, segment) pairs,
      // each from what the segments before it make of the state
      float* seg = ws.seg;
      float* ptot = seg + (size_t)B * sp.nf * a.D * a.N * 2;
      sa = SegArgs{a.delta, a.u, a.theta, a.Bm, seg, ptot, a.D, a.N, sp.ls / sp.r, L, sp.nf, a.ncg};
      nseg = (unsigned)(B * sp.nf * a.ncg);
      if (mode != 6)
        if (int e = run_seg_state(false, sa, in_dtype, nseg, s)) return e;
      a.B = B * sp.ns; a.L = sp.ls; a.ns = sp.ns; a.seg = seg; a.segq = ptot; a.hs = sp.r; a.nf = sp.nf;
    }
  }
  if (mode == 6) {
    // one pre-pass for the step: the backward call that follows finds its images too (it needs the
    // checkpoints, so a call without them is not followed by one)
    const bool with_bwd = a.hck != nullptr;
    PrepArgs pa{a.Bm, a.Cm, ws.fimg, with_bwd ? ws.img : nullptr, a.N, L, (L + XT - 1) / XT, nullptr, ImgStamp{}};
    if (int e = nseg ? run_prep_seg(pa, B, sa, nseg, in_dtype, s) : run_px_prep(pa, B, in_dtype, s)) return e;
    const ImgNote note{ws.stamp, img_stamp(a.Bm, a.Cm, B, a.N, L, in_dtype, with_bwd), clear_in_kernel ? ws.pad : nullptr};
    return run_px_fwd(a, ws.fimg, note, in_dtype, s);
  }
  return run_xdl_fwd(mode, a, in_dtype, s);
}

// Complex and real scans: with a workspace and few (batch, channel group) pairs, split along the sequence.
int launch_generic_fwd(int variant, FwdArgs a, int in_dtype, float* ws, hipStream_t s) {
  if (in_dtype == AUSSM_BF16 && !ws) return AUSSM_E_NULL;
  if (misaligned(ws, 16)) return AUSSM_E_ALIGN;
  const bool in_place = overlap(a.h0, a.hL, (size_t)a.B * a.D * a.N * (variant == VAR_REAL ? 1 : 2));
  const GSplit sp = ws && !in_place ? generic_split(a.B, a.D, a.L, a.ck, true) : GSplit{1, a.L};
  if (sp.ns > 1) {
    const int B = a.B, C = variant == VAR_REAL ? 1 : 2;
    float* seg = ws;
    float* ptot = seg + (size_t)B * sp.ns * a.D * a.N * C;
    // 1. end state of every segment from a zero state (no outputs) and the product of its a_l
    FwdArgs z = a;
    z.B = B * sp.ns; z.L = sp.ls; z.ns = sp.ns;
    z.y = nullptr; z.z = nullptr; z.Dskip = nullptr; z.h0 = nullptr; z.hL = seg; z.hck = nullptr; z.ptot = ptot;
    if (int e = run_oct_fwd(variant, z, in_dtype, s)) return e;
    // 2. the scan proper over (batch, segment) pairs, each from what those before it make of the state
    a.B = B * sp.ns; a.L = sp.ls; a.ns = sp.ns; a.seg = seg; a.segq = ptot;
  }
  return run_oct_fwd(variant, a, in_dtype, s);
}

int launch_generic_bwd(int variant, RecBwdArgs a, int in_dtype, float* ws, hipStream_t s) {
  if (in_dtype == AUSSM_BF16 && !ws) return AUSSM_E_NULL;
  if (misaligned(ws, 16)) return AUSSM_E_ALIGN;
  const bool in_place = overlap(a.dhL, a.dh0, (size_t)a.B * a.D * a.N * (variant == VAR_REAL ? 1 : 2));
  const GSplit sp = ws && !in_place ? generic_split(a.B, a.D, a.L, REC_CK, true) : GSplit{1, a.L};
  if (sp.ns > 1) {
    const int B = a.B, C = variant == VAR_REAL ? 1 : 2;
    float* seg = ws;
    float* ptot = seg + (size_t)B * sp.ns * a.D * a.N * C;
    AdjSegArgs g{};
    g.dy = a.dy; g.z = a.z; g.delta = a.delta; g.theta = a.theta; g.rho = a.rho; g.A = a.A; g.Cm = a.Cm;
    g.delta_bias = a.delta_bias; g.out = seg; g.ptot = ptot;
    g.D = a.D; g.N = a.N; g.L = sp.ls; g.ld = a.L; g.ns = sp.ns; g.ncg = a.ncg; g.delta_softplus = a.delta_softplus;
    g.zrows = a.zrows; g.bcrows = a.bcrows;
    if (int e = run_oct_adj(variant, g, in_dtype, (unsigned)(B * sp.ns * a.ncg), s)) return e;
    a.B = B * sp.ns; a.L = sp.ls; a.ns = sp.ns; a.seg = seg; a.segq = ptot;
  }
  return run_oct_bwd(variant, a, in_dtype, s);
}

// ---- static workspace of aussm_unitary_fwd_static ---------------------------------------------
// A file-scope device array: every GPU the library runs on holds its own copy at its own address
// until the process ends.  In host code the array's NAME is only a handle for the runtime, not a
// device address: the address is looked up once per device (hipGetSymbolAddress) and that pointer
// is what the launches are given.
constexpr size_t STATIC_SCRATCH_FLOATS = AUSSM_STATIC_SCRATCH_BYTES / sizeof(float);
static __device__ __align__(256) float g_static_scratch[STATIC_SCRATCH_FLOATS];
constexpr int MAX_DEVICES = 64;
std::atomic<float*> g_static_scratch_ptr[MAX_DEVICES];

int static_scratch(float** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= MAX_DEVICES) return AUSSM_E_SHAPE;
  float* ptr = g_static_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!ptr) {
    e = hipGetSymbolAddress(reinterpret_cast<void**>(&ptr), HIP_SYMBOL(g_static_scratch));
    if (e != hipSuccess) return (int)e;
    if (!ptr) return AUSSM_E_NULL;
    g_static_scratch_ptr[dev].store(ptr, std::memory_order_release);
  }
  *out = ptr;
  return AUSSM_OK;
}

}  // namespace

extern "C" {

int aussm_version(void) { return 100; }

const char* aussm_error_string(int code) {
  switch (code) {
    case AUSSM_OK: return "ok";
    case AUSSM_E_NULL: return "a required pointer is NULL";
    case AUSSM_E_SHAPE: return "dimension out of the supported range (B,D,N,L >= 1, N <= 64)";
    case AUSSM_E_CK: return "checkpoint interval must be a multiple of 32 accepted by this function";
    case AUSSM_E_DTYPE: return "in_dtype must be AUSSM_F32 or AUSSM_BF16";
    case AUSSM_E_ALIGN: return "pointer not aligned to its element size";
    case AUSSM_E_SCRATCH: return "the call needs more workspace than the static scratch holds (use the _aux entry point)";
    default: return code > 0 ? hipGetErrorString((hipError_t)code) : "unknown aussm error";
  }
}

int aussm_set_option(int key, int value) {
  if (key < 0 || key >= AUSSM_OPT_COUNT) return AUSSM_E_SHAPE;
  g_opt[key].store(value < 0 ? -1 : value, std::memory_order_relaxed);
  return AUSSM_OK;
}

int aussm_get_option(int key) {
  if (key < 0 || key >= AUSSM_OPT_COUNT) return AUSSM_E_SHAPE;
  return opt(key);
}

int aussm_num_checkpoints(int L, int ck) { return (L < 1 || ck < 1) ? 0 : (L + ck - 1) / ck; }

int aussm_bwd_checkpoint_interval(int variant) { return variant == VAR_UNITARY ? 0 : REC_CK; }

int aussm_unitary_split_segments(int B, int D, int N, int L, int ck) {
  if (B < 1 || D < 1 || N < 1 || L < 1 || ck < 1) return 0;
  int ns = unitary_split(B, D, N, L, ck, false).ns;
  // shapes that the vector-ALU kernels serve by default split their way
  if (!(matrix_shape(N, L, ck) && N >= MATRIX_MIN_STATE)) {
    const int g = generic_split(B, D, L, ck, false).ns;
    if (g > ns) ns = g;
  }
  return ns;
}

size_t aussm_unitary_aux_floats(int B, int D, int N, int L, int ck) {
  if (B < 1 || D < 1 || N < 1 || L < 1) return 0;
  return aux_im_floats(B, D, N, L, ck) + AUX_PAD + aux_seg_floats(B, D, N, L, ck) + img_floats(B, N, L, ck);
}

size_t aussm_scan_workspace_floats(int variant, int B, int D, int N, int L, int ck, int in_dtype) {
  if (B < 1 || D < 1 || N < 1 || L < 1 || (variant != VAR_COMPLEX && variant != VAR_REAL)) return 0;
  if (ck != AUSSM_TILE / 2 && (ck < AUSSM_TILE || ck % AUSSM_TILE != 0)) return 0;
  return generic_split_floats(variant, B, D, N, L, ck) + 2 * generic_bc_floats(variant, B, N, L, in_dtype);
}

int aussm_unitary_kernel_mode(int backward, int B, int D, int N, int L, int ck, int in_dtype, int urep, int have_aux) {
  if (check_common(B, D, N, L, ck, in_dtype) != AUSSM_OK || urep < 1) return 0;
  const bool have_img = have_aux && img_floats(B, N, L, ck) > 0;
  return backward ? bwd_mode_for(B, D, N, L, ck, urep, have_img) : fwd_mode_for(N, L, ck, in_dtype, urep, have_img);
}

int aussm_hbm_probe(const float* a, const float* b, const float* c, float* o1, float* o2, int rows, int L,
                    int pattern, int write, void* stream) {
  if (rows < 64 || rows % 64 != 0 || L < 64 || L % 64 != 0 || (pattern != 0 && pattern != 1)) return AUSSM_E_SHAPE;
  if (!a || !b || !c || !o1 || (write && !o2)) return AUSSM_E_NULL;
  if (misaligned(a, 16) || misaligned(b, 16) || misaligned(c, 16) || misaligned(o1, 16) || misaligned(o2, 16))
    return AUSSM_E_ALIGN;
  return run_hbm_probe(a, b, c, o1, o2, rows, L, pattern, write, (hipStream_t)stream);
}

int aussm_unitary_fwd(const void* u, const void* delta, const float* theta, const void* Bc, const void* Cc,
                      const float* Dskip, const float* z, const float* h0, float* y, float* hL, float* hck,
                      int B, int D, int N, int L, int ck, int in_dtype, void* stream) {
  return aussm_unitary_fwd_aux(u, delta, theta, Bc, Cc, Dskip, z, h0, y, hL, hck, nullptr, B, D, N, L, ck, in_dtype,
                               1, stream);
}

int aussm_unitary_fwd_aux(const void* u, const void* delta, const float* theta, const void* Bc, const void* Cc,
                          const float* Dskip, const float* z, const float* h0, float* y, float* hL, float* hck,
                          float* aux, int B, int D, int N, int L, int ck, int in_dtype, int urep, void* stream) {
  if (int e = check_common(B, D, N, L, ck, in_dtype)) return e;
  if (urep < 1 || B % urep != 0) return AUSSM_E_SHAPE;
  if (misaligned(aux, 16)) return AUSSM_E_ALIGN;
  if (!u || !delta || !theta || !Bc || !Cc) return AUSSM_E_NULL;
  const size_t ca = in_dtype == AUSSM_BF16 ? 4 : 8;
  if (misaligned(Bc, ca) || misaligned(Cc, ca)) return AUSSM_E_ALIGN;
  FwdArgs a{};
  a.u = u; a.delta = delta; a.theta = theta; a.Bm = Bc; a.Cm = Cc; a.Dskip = Dskip; a.z = z;
  a.h0 = h0; a.y = y; a.hL = hL; a.hck = hck; a.aux = aux;
  a.B = B; a.D = D; a.N = N; a.L = L; a.ck = ck; a.nck = (L + ck - 1) / ck; a.ncg = (D + CH - 1) / CH;
  a.ld = L; a.ns = 1; a.urep = urep;
  a.auxtag = aux_tag(u, delta, theta, Bc, Cc, B, D, N, L, in_dtype);
  return launch_unitary_fwd(a, in_dtype, (hipStream_t)stream, aux_layout(aux, B, D, N, L, ck));
}

int aussm_static_init(void) {
  float* ptr = nullptr;
  return static_scratch(&ptr);
}

int aussm_unitary_fwd_static(const void* u, const void* delta, const float* theta, const void* Bc, const void* Cc,
                             const float* Dskip, const float* z, const float* h0, float* y, float* hL,
                             int B, int D, int N, int L, int ck, int in_dtype, void* stream) {
  if (int e = check_common(B, D, N, L, ck, in_dtype)) return e;
  if (!u || !delta || !theta || !Bc || !Cc) return AUSSM_E_NULL;
  const size_t ca = in_dtype == AUSSM_BF16 ? 4 : 8;
  if (misaligned(Bc, ca) || misaligned(Cc, ca)) return AUSSM_E_ALIGN;
  // the only workspace a forward call without checkpoints uses: the segment states of a launch
  // that is split along L
  const size_t need = seg_floats(B, D, N, L, seg_capacity(B, D, N, L, ck));
  if (need > STATIC_SCRATCH_FLOATS) return AUSSM_E_SCRATCH;
  float* scratch = nullptr;
  if (need > 0)
    if (int e = static_scratch(&scratch)) return e;
  FwdArgs a{};
  a.u = u; a.delta = delta; a.theta = theta; a.Bm = Bc; a.Cm = Cc; a.Dskip = Dskip; a.z = z;
  a.h0 = h0; a.y = y; a.hL = hL; a.hck = nullptr; a.aux = nullptr;
  a.B = B; a.D = D; a.N = N; a.L = L; a.ck = ck; a.nck = (L + ck - 1) / ck; a.ncg = (D + CH - 1) / CH;
  a.ld = L; a.ns = 1; a.urep = 1;
  // (every segment state the scan reads is written earlier in the same call: nothing in the
  // scratch has to start at zero)
  // (Neither the vector-ALU kernels, no gseg, nor sequences that do not halve into equal segments, no room, split here: all calls
  // on a GPU share one array, and those that need none of it may run on several streams at once.)
  return launch_unitary_fwd(a, in_dtype, (hipStream_t)stream, AuxLayout{scratch, nullptr, nullptr, nullptr, nullptr, nullptr, 0});
}

int aussm_complex_fwd(const void* u, const void* delta, const float* rho, const float* theta, const void* Bc,
                      const void* Cc, const float* Dskip, const float* z, const float* h0, float* y, float* hL,
                      float* hck, float* workspace, int B, int D, int N, int L, int ck, int in_dtype, void* stream) {
  if (int e = check_common(B, D, N, L, ck, in_dtype)) return e;
  if (!u || !delta || !rho || !theta || !Bc || !Cc) return AUSSM_E_NULL;
  const size_t ca = in_dtype == AUSSM_BF16 ? 4 : 8;
  if (misaligned(Bc, ca) || misaligned(Cc, ca)) return AUSSM_E_ALIGN;
  FwdArgs a{};
  a.u = u; a.delta = delta; a.rho = rho; a.theta = theta; a.Bm = Bc; a.Cm = Cc; a.Dskip = Dskip; a.z = z;
  a.h0 = h0; a.y = y; a.hL = hL; a.hck = hck;
  a.B = B; a.D = D; a.N = N; a.L = L; a.ck = ck; a.nck = (L + ck - 1) / ck; a.ncg = (D + CH - 1) / CH;
  a.ld = L; a.ns = 1; a.urep = 1;
  return launch_generic_fwd(VAR_COMPLEX, a, in_dtype, workspace, (hipStream_t)stream);
}

int aussm_real_fwd(const void* u, const void* delta, const float* A, const void* Bm, const void* Cm,
                   const float* Dskip, const float* z, const float* delta_bias, int delta_softplus,
                   const float* h0, float* y, float* hL, float* hck, float* workspace,
                   int B, int D, int N, int L, int ck, int in_dtype, void* stream) {
  return aussm_real_fwd_rows(u, delta, A, Bm, Cm, Dskip, z, delta_bias, delta_softplus, h0, y, hL, hck, workspace, nullptr, B, D, N, L, ck,
                             in_dtype, stream);
}

// (B_t / C_t as rows of wider tensors: float inputs only, as the Mamba block calls it; bf16 ones have never been taken)
static int real_rows_check(const aussm_real_rows* r, int D, int N, int in_dtype) {
  if (!r) return AUSSM_OK;
  if ((r->z_rows && r->z_rows < D) || (r->bc_rows && r->bc_rows < N)) return AUSSM_E_SHAPE;
  return r->bc_rows && in_dtype != AUSSM_F32 ? AUSSM_E_DTYPE : AUSSM_OK;
}

int aussm_real_fwd_rows(const void* u, const void* delta, const float* A, const void* Bm, const void* Cm,
                        const float* Dskip, const float* z, const float* delta_bias, int delta_softplus,
                        const float* h0, float* y, float* hL, float* hck, float* workspace, const aussm_real_rows* rows,
                        int B, int D, int N, int L, int ck, int in_dtype, void* stream) {
  if (int e = check_common(B, D, N, L, ck, in_dtype)) return e;
  if (!u || !delta || !A || !Bm || !Cm) return AUSSM_E_NULL;
  FwdArgs a{};
  a.u = u; a.delta = delta; a.A = A; a.Bm = Bm; a.Cm = Cm; a.Dskip = Dskip; a.z = z;
  a.delta_bias = delta_bias; a.delta_softplus = delta_softplus;
  a.h0 = h0; a.y = y; a.hL = hL; a.hck = hck;
  if (int e = real_rows_check(rows, D, N, in_dtype)) return e;
  if (rows) { a.zrows = rows->z_rows; a.bcrows = rows->bc_rows; a.u_act = rows->u_silu; }
  a.B = B; a.D = D; a.N = N; a.L = L; a.ck = ck; a.nck = (L + ck - 1) / ck; a.ncg = (D + CH - 1) / CH;
  a.ld = L; a.ns = 1; a.urep = 1;
  return launch_generic_fwd(VAR_REAL, a, in_dtype, workspace, (hipStream_t)stream);
}

int aussm_unitary_bwd(const float* dy, const float* dhL, const void* u, const void* delta, const float* theta,
                      const void* Bc, const void* Cc, const float* Dskip, const float* hck,
                      float* du, float* ddelta, float* dtheta, float* dB, float* dC, float* dD, float* dh0,
                      int B, int D, int N, int L, int ck, int in_dtype, void* stream) {
  return aussm_unitary_bwd_aux(dy, dhL, u, delta, theta, Bc, Cc, Dskip, hck, nullptr, du, ddelta, dtheta, dB, dC, dD,
                               dh0, B, D, N, L, ck, in_dtype, 1, stream);
}

int aussm_unitary_bwd_aux(const float* dy, const float* dhL, const void* u, const void* delta, const float* theta,
                          const void* Bc, const void* Cc, const float* Dskip, const float* hck, float* aux,
                          float* du, float* ddelta, float* dtheta, float* dB, float* dC, float* dD, float* dh0,
                          int B, int D, int N, int L, int ck, int in_dtype, int urep, void* stream) {
  const int g16 = take_flag(in_dtype, AUSSM_GRADS_IN_DTYPE), own_aux = take_flag(in_dtype, AUSSM_AUX_FILLED);
  if (int e = check_common(B, D, N, L, ck, in_dtype)) return e;
  if (urep < 1 || B % urep != 0) return AUSSM_E_SHAPE;
  if (misaligned(aux, 16)) return AUSSM_E_ALIGN;
  if (!dy || !u || !delta || !theta || !Bc || !Cc || !hck || !du || !ddelta || !dtheta || !dB || !dC)
    return AUSSM_E_NULL;
  const size_t ca = in_dtype == AUSSM_BF16 ? 4 : 8;
  if (misaligned(Bc, ca) || misaligned(Cc, ca)) return AUSSM_E_ALIGN;
  hipStream_t s = (hipStream_t)stream;
  UniBwdArgs a{};
  a.dy = dy; a.dhL = dhL; a.u = u; a.delta = delta; a.theta = theta; a.Bm = Bc; a.Cm = Cc; a.Dskip = Dskip;
  a.hck = hck; a.aux = aux; a.du = du; a.ddelta = ddelta; a.dtheta = dtheta; a.dB = dB; a.dC = dC; a.dD = dD; a.dh0 = dh0;
  a.B = B; a.D = D; a.N = N; a.L = L; a.ck = ck; a.nck = (L + ck - 1) / ck; a.ncg = (D + CH - 1) / CH;
  a.ld = L; a.ns = 1; a.urep = 1;
  a.urep = urep;
  a.g16 = g16 && in_dtype == AUSSM_BF16;
  a.auxtag = aux_tag(u, delta, theta, Bc, Cc, B, D, N, L, in_dtype);
  const AuxLayout ws = aux_layout(aux, B, D, N, L, ck);
  const int mode = bwd_mode_for(B, D, N, L, ck, urep, ws.img != nullptr);
  const bool in_place = overlap(dhL, dh0, (size_t)B * D * N * 2);
  if (mode > 0 &&
      !(misaligned(dy, 16) || misaligned(u, 16) || misaligned(delta, 16) || misaligned(theta, 16) ||
        misaligned(du, 16) || misaligned(ddelta, 16) || misaligned(dtheta, 16) || misaligned(Bc, 16) ||
        misaligned(Cc, 16))) {
    const USplit sp = aux && !in_place ? unitary_split(B, D, N, L, ck, true, ws.seg_room) : USplit{1, L, 1, 1};
    if (sp.ns > 1) {
      // adjoint at the start of every segment from a zero adjoint at its end
      float* seg = ws.seg;
      float* ptot = seg + (size_t)B * sp.nf * D * N * 2;
      SegArgs sa{dy, nullptr, theta, Cc, seg, ptot, D, N, sp.ls / sp.r, L, sp.nf, a.ncg};
      if (int e = run_seg_state(true, sa, in_dtype, (unsigned)(B * sp.nf * a.ncg), s)) return e;
      a.B = B * sp.ns; a.L = sp.ls; a.ns = sp.ns; a.seg = seg; a.segq = ptot; a.hs = sp.r; a.nf = sp.nf;
    }
    if (mode == 6) {
      // The prepared-operand kernel needs Im(P S) from the forward call in the auxiliary buffer; its
      // workgroups leave at once if the buffer's tag says it is not there, and the kernel that
      // recomputes it (launched behind, leaving at once in the opposite case) does the work.
      // A caller that made the forward call itself on these tensors and this buffer says so (AUSSM_AUX_FILLED), and
      // neither of the two launches that would find nothing to do takes place (5 us each).
      if (own_aux && aux) {
        a.tag_mode = 0;
        return run_px_bwd(a, ws.img, in_dtype, s);
      }
      // (the pre-pass leaves at once when the forward call of these tensors has left the images)
      PrepArgs pa{Bc, Cc, nullptr, ws.img, N, L, (L + XT - 1) / XT, ws.stamp, img_stamp(Bc, Cc, B, N, L, in_dtype, true)};
      if (int e = run_px_prep(pa, B, in_dtype, s)) return e;
      a.tag_mode = 1;
      if (int e = run_px_bwd(a, ws.img, in_dtype, s)) return e;
      a.tag_mode = 2;
      return run_xdl_bwd(3, a, in_dtype, s);
    }
    return run_xdl_bwd(mode, a, in_dtype, s);
  }
  // vector-ALU kernel; split along the sequence like the forward call
  const GSplit sp = ws.gseg && !in_place ? generic_split(B, D, L, ck, true) : GSplit{1, L};
  if (sp.ns > 1) {
    float* seg = ws.gseg;
    float* ptot = seg + (size_t)B * sp.ns * D * N * 2;
    AdjSegArgs g{};
    g.dy = dy; g.theta = theta; g.Cm = Cc; g.out = seg; g.ptot = ptot;
    g.D = D; g.N = N; g.L = sp.ls; g.ld = L; g.ns = sp.ns; g.ncg = a.ncg;
    if (int e = run_oct_adj(VAR_UNITARY, g, in_dtype, (unsigned)(B * sp.ns * a.ncg), s)) return e;
    a.B = B * sp.ns; a.L = sp.ls; a.ns = sp.ns; a.seg = seg; a.segq = ptot;
  }
  // (Blocks of 32 states add to what the first wrote, which bf16 would round.  8 x 72 x 37, 2957 steps: 237 us against 642.)
  if (N <= 32 || !a.g16) return run_oct_ubwd(a, in_dtype, s);
  return run_unitary_bwd_generic(a, pick_cfg(), s);
}

int aussm_complex_bwd(const float* dy, const float* dhL, const void* u, const void* delta, const float* rho,
                      const float* theta, const void* Bc, const void* Cc, const float* Dskip,
                      const float* h0, const float* hck,
                      float* du, float* ddelta, float* drho, float* dtheta, float* dB, float* dC,
                      float* dD, float* dh0, const float* z, float* dz, float* workspace,
                      int B, int D, int N, int L, int ck, int in_dtype, void* stream) {
  const int g16 = take_flag(in_dtype, AUSSM_GRADS_IN_DTYPE);
  if (int e = check_common(B, D, N, L, ck, in_dtype)) return e;
  if (ck != REC_CK) return AUSSM_E_CK;
  if (!dy || !u || !delta || !rho || !theta || !Bc || !Cc || !hck || !du || !ddelta || !drho || !dtheta ||
      !dB || !dC)
    return AUSSM_E_NULL;
  const size_t ca = in_dtype == AUSSM_BF16 ? 4 : 8;
  if (misaligned(Bc, ca) || misaligned(Cc, ca)) return AUSSM_E_ALIGN;
  RecBwdArgs a{};
  a.dy = dy; a.dhL = dhL; a.u = u; a.delta = delta; a.theta = theta; a.rho = rho; a.Bm = Bc; a.Cm = Cc;
  a.Dskip = Dskip; a.h0 = h0; a.hck = hck;
  a.du = du; a.ddelta = ddelta; a.dtheta = dtheta; a.drho = drho; a.dB = dB; a.dC = dC; a.dD = dD; a.dh0 = dh0;
  if ((z == nullptr) != (dz == nullptr)) return AUSSM_E_NULL;
  a.z = z; a.dz = dz;
  a.B = B; a.D = D; a.N = N; a.L = L; a.ck = ck; a.nck = (L + ck - 1) / ck; a.ncg = (D + CH - 1) / CH;
  // (several blocks of states add up in du and ddelta: those stay float)
  if (g16 && in_dtype == AUSSM_BF16 && N > 16) return AUSSM_E_DTYPE;
  a.g16 = g16 && in_dtype == AUSSM_BF16;
  a.ld = L; a.ns = 1;
  return launch_generic_bwd(VAR_COMPLEX, a, in_dtype, workspace, (hipStream_t)stream);
}

int aussm_real_bwd(const float* dy, const float* dhL, const void* u, const void* delta, const float* A,
                   const void* Bm, const void* Cm, const float* Dskip, const float* delta_bias,
                   int delta_softplus, const float* h0, const float* hck,
                   float* du, float* ddelta, float* dA, float* dB, float* dC, float* dD, float* dh0,
                   const float* z, float* dz, float* workspace,
                   int B, int D, int N, int L, int ck, int in_dtype, void* stream) {
  return aussm_real_bwd_rows(dy, dhL, u, delta, A, Bm, Cm, Dskip, delta_bias, delta_softplus, h0, hck, du, ddelta, dA, dB, dC, dD, dh0, z, dz,
                             workspace, nullptr, B, D, N, L, ck, in_dtype, stream);
}

int aussm_real_bwd_rows(const float* dy, const float* dhL, const void* u, const void* delta, const float* A,
                   const void* Bm, const void* Cm, const float* Dskip, const float* delta_bias,
                   int delta_softplus, const float* h0, const float* hck,
                   float* du, float* ddelta, float* dA, float* dB, float* dC, float* dD, float* dh0,
                   const float* z, float* dz, float* workspace, const aussm_real_rows* rows,
                   int B, int D, int N, int L, int ck, int in_dtype, void* stream) {
  const int g16 = take_flag(in_dtype, AUSSM_GRADS_IN_DTYPE);
  if (int e = check_common(B, D, N, L, ck, in_dtype)) return e;
  if (ck != REC_CK) return AUSSM_E_CK;
  if (!dy || !u || !delta || !A || !Bm || !Cm || !hck || !du || !ddelta || !dB || !dC) return AUSSM_E_NULL;
  RecBwdArgs a{};
  a.dy = dy; a.dhL = dhL; a.u = u; a.delta = delta; a.A = A; a.Bm = Bm; a.Cm = Cm; a.Dskip = Dskip;
  a.delta_bias = delta_bias; a.delta_softplus = delta_softplus; a.h0 = h0; a.hck = hck;
  a.du = du; a.ddelta = ddelta; a.dA = dA; a.dB = dB; a.dC = dC; a.dD = dD; a.dh0 = dh0;
  if ((z == nullptr) != (dz == nullptr)) return AUSSM_E_NULL;
  if (int e = real_rows_check(rows, D, N, in_dtype)) return e;
  if (rows) {
    a.zrows = rows->z_rows; a.bcrows = rows->bc_rows; a.u_act = rows->u_silu;
    a.dbias = rows->ddelta_bias; a.dbias_scale = rows->ddelta_bias_scale;
  }
  a.z = z; a.dz = dz;
  a.B = B; a.D = D; a.N = N; a.L = L; a.ck = ck; a.nck = (L + ck - 1) / ck; a.ncg = (D + CH - 1) / CH;
  // (several launches add up in du and ddelta: those stay float, 17 to 24 states, which one launch holds here, like more)
  if (g16 && in_dtype == AUSSM_BF16 && N > 16) return AUSSM_E_DTYPE;
  a.g16 = g16 && in_dtype == AUSSM_BF16;
  a.ld = L; a.ns = 1;
  return launch_generic_bwd(VAR_REAL, a, in_dtype, workspace, (hipStream_t)stream);
}

int aussm_causal_conv1d_fwd(const float* x, const float* w, const float* bias, float* y,
                            int B, int L, int D, int K, long long xs_b, long long xs_l, void* stream) {
  if (B < 1 || L < 1 || D < 1 || K < 1 || K > CONV_MAX_K || xs_l < D || xs_b < (long long)L * xs_l - (xs_l - D))
    return AUSSM_E_SHAPE;
  if (!x || !w || !y) return AUSSM_E_NULL;
  ConvArgs a{};
  a.x = x; a.w = w; a.bias = bias; a.y = y; a.xs_b = xs_b; a.xs_l = xs_l; a.B = B; a.L = L; a.D = D; a.K = K;
  const size_t rows = (size_t)B * L;
  if (rows > 0x7fffffffULL || (D + 255) / 256 > 65535) return AUSSM_E_SHAPE;
  return run_conv_fwd(a, (hipStream_t)stream);
}

int aussm_causal_conv1d_bwd(const float* dy, const float* x, const float* w, float* dx, float* dw, float* dbias,
                            int B, int L, int D, int K, long long xs_b, long long xs_l, void* stream) {
  if (B < 1 || L < 1 || D < 1 || K < 1 || K > CONV_MAX_K || xs_l < D || xs_b < (long long)L * xs_l - (xs_l - D))
    return AUSSM_E_SHAPE;
  if (!dy || !x || !w || !dx || !dw) return AUSSM_E_NULL;
  ConvArgs a{};
  a.x = x; a.w = w; a.dy = dy; a.dx = dx; a.dw = dw; a.dbias = dbias;
  a.xs_b = xs_b; a.xs_l = xs_l; a.B = B; a.L = L; a.D = D; a.K = K;
  const size_t rows = (size_t)B * L;
  if (rows > 0x7fffffffULL || (D + 255) / 256 > 65535 || (rows + CONV_ROWS - 1) / CONV_ROWS > 65535) return AUSSM_E_SHAPE;
  return run_conv_bwd(a, (hipStream_t)stream);
}

int aussm_swap_last2(const float* x, float* y, int B, int R, int C, long long xs_b, long long xs_r, void* stream) {
  if (B < 1 || R < 1 || C < 1 || B > 65535 || xs_r < C || xs_b < (long long)R * xs_r - (xs_r - C)) return AUSSM_E_SHAPE;
  if ((R + 31) / 32 > 65535) return AUSSM_E_SHAPE;
  if (!x || !y) return AUSSM_E_NULL;
  SwapArgs a{};
  a.x = x; a.y = y; a.xs_b = xs_b; a.xs_r = xs_r; a.R = R; a.C = C;
  return run_swap_last2(a, B, (hipStream_t)stream);
}

int aussm_swap_last2_act(const float* x, const float* bias, const float* pre, float* y, int B, int R, int C,
                         long long xs_b, long long xs_r, long long ps_b, long long ps_r, int act, int deriv,
                         void* stream) {
  if (B < 1 || R < 1 || C < 1 || B > 65535 || xs_r < C || xs_b < (long long)R * xs_r - (xs_r - C)) return AUSSM_E_SHAPE;
  if ((R + 31) / 32 > 65535 || act < 1 || act > 2) return AUSSM_E_SHAPE;
  if (!x || !y || (deriv && !pre)) return AUSSM_E_NULL;
  // pre has the output's shape (B, C, R): rows of R elements that do not overlap
  if (deriv && (ps_r < R || ps_b < (long long)C * ps_r - (ps_r - R))) return AUSSM_E_SHAPE;
  SwapArgs a{};
  a.x = x; a.y = y; a.xs_b = xs_b; a.xs_r = xs_r; a.R = R; a.C = C;
  a.bias = bias; a.pre = deriv ? pre : nullptr; a.ps_b = ps_b; a.ps_r = ps_r; a.act = act; a.deriv = deriv ? 1 : 0;
  return run_swap_last2(a, B, (hipStream_t)stream);
}

int aussm_gate_fwd(const float* y_pre, const float* z, float* y, size_t n, void* stream) {
  if (!y_pre || !z || !y) return AUSSM_E_NULL;
  if (n < 1) return AUSSM_E_SHAPE;
  if (misaligned(y_pre, 4) || misaligned(z, 4) || misaligned(y, 4)) return AUSSM_E_ALIGN;
  return run_gate(nullptr, y_pre, z, y, nullptr, n, (hipStream_t)stream);
}

int aussm_gate_bwd(const float* dy, const float* y_pre, const float* z, float* dy_pre, float* dz, size_t n, void* stream) {
  if (!dy || !y_pre || !z || !dy_pre || !dz) return AUSSM_E_NULL;
  if (n < 1) return AUSSM_E_SHAPE;
  if (misaligned(dy, 4) || misaligned(y_pre, 4) || misaligned(z, 4) || misaligned(dy_pre, 4) || misaligned(dz, 4))
    return AUSSM_E_ALIGN;
  return run_gate(dy, y_pre, z, dy_pre, dz, n, (hipStream_t)stream);
}

int aussm_gemm(const aussm_gemm_args* g, void* stream) {
  if (!g || !g->A || !g->B || !g->C) return AUSSM_E_NULL;
  if (g->M < 1 || g->N < 1 || g->K < 1 || g->Z < 1 || g->nper < 1) return AUSSM_E_SHAPE;
  if ((g->sam != 1 && g->sak != 1) || (g->sbk != 1 && g->sbn != 1) || (g->scm != 1 && g->scn != 1)) return AUSSM_E_SHAPE;
  if (g->act != 0 && g->act != 1) return AUSSM_E_SHAPE;
  if (g->reduce && (g->bias || g->add || g->act)) return AUSSM_E_SHAPE;
  XGemmArgs a{};
  a.A = g->A; a.B = g->B; a.C = g->C; a.bias = g->bias; a.add = g->add; a.alpha = g->alpha; a.bias_scale = g->bias_scale;
  a.act = g->act; a.sam = g->sam; a.sak = g->sak; a.saz = g->saz; a.sbk = g->sbk; a.sbn = g->sbn; a.sbb = g->sbb; a.sbz = g->sbz;
  a.scm = g->scm; a.scn = g->scn; a.scb = g->scb; a.M = g->M; a.N = g->N; a.K = g->K; a.Z = g->Z; a.nper = g->nper;
  a.reduce = g->reduce != 0;
  return run_xgemm(a, (hipStream_t)stream);
}

int aussm_conv_rows_fwd(const float* x, const float* w, const float* bias, float* y, int B, int D, int L, int K, long long xs_b, void* stream) {
  if (B < 1 || D < 1 || L < 1 || K < 1 || K > CONV_MAX_K || xs_b < (long long)D * L) return AUSSM_E_SHAPE;
  if (!x || !w || !y) return AUSSM_E_NULL;
  if (misaligned(y, 16)) return AUSSM_E_ALIGN;
  ConvRowsArgs a{};
  a.x = x; a.w = w; a.bias = bias; a.y = y; a.xs_b = (long)xs_b; a.B = B; a.D = D; a.L = L; a.K = K;
  return run_conv_rows_fwd(a, (hipStream_t)stream);
}
int aussm_conv_rows_bwd(const float* dy, const float* x, const float* w, float* dx, float* dw, float* dbias, int B, int D, int L, int K,
                        long long xs_b, long long dxs_b, void* stream) {
  if (B < 1 || D < 1 || L < 1 || K < 1 || K > CONV_MAX_K || xs_b < (long long)D * L || dxs_b < (long long)D * L) return AUSSM_E_SHAPE;
  if (!dy || !x || !w || !dx || !dw) return AUSSM_E_NULL;
  ConvRowsArgs a{};
  a.dy = dy; a.x = x; a.w = w; a.dx = dx; a.dw = dw; a.dbias = dbias; a.xs_b = (long)xs_b; a.dxs_b = (long)dxs_b;
  a.B = B; a.D = D; a.L = L; a.K = K;
  return run_conv_rows_bwd(a, (hipStream_t)stream);
}
int aussm_rms_norm_fwd(const float* x, const float* w, float* y, float* rstd, size_t rows, int d, float eps, void* stream) {
  if (rows < 1 || d < 1 || d > NORM_MAX_D) return AUSSM_E_SHAPE;
  if (!x || !w || !y) return AUSSM_E_NULL;
  NormArgs a{};
  a.x = x; a.w = w; a.y = y; a.rstd = rstd; a.rows = rows; a.d = d; a.eps = eps;
  return run_norm_fwd(a, (hipStream_t)stream);
}
int aussm_rms_norm_bwd(const float* dy, const float* x, const float* w, const float* rstd, const float* res, float* dx, float* dw,
                       size_t rows, int d, void* stream) {
  if (rows < 1 || d < 1 || d > NORM_MAX_D) return AUSSM_E_SHAPE;
  if (!dy || !x || !w || !rstd || !dx || !dw) return AUSSM_E_NULL;
  NormArgs a{};
  a.dy = dy; a.x = x; a.w = w; a.rstd = const_cast<float*>(rstd); a.res = res; a.dx = dx; a.dw = dw; a.rows = rows; a.d = d;
  return run_norm_bwd(a, (hipStream_t)stream);
}
int aussm_col_sum(const float* x, float* out, size_t rows, int d, float scale, void* stream) {
  if (rows < 1 || d < 1) return AUSSM_E_SHAPE;
  if (!x || !out) return AUSSM_E_NULL;
  return run_col_sum(x, out, rows, d, scale, (hipStream_t)stream);
}
int aussm_row_sum(const float* x, float* out, size_t rows, int d, int L, float scale, void* stream) {
  if (rows < 1 || d < 1 || L < 1) return AUSSM_E_SHAPE;
  if (!x || !out) return AUSSM_E_NULL;
  return run_row_sum(x, out, rows, d, L, scale, (hipStream_t)stream);
}
int aussm_neg_exp(const float* a_log, const float* dA, float* out, int n, void* stream) {
  if (n < 1) return AUSSM_E_SHAPE;
  if (!a_log || !out) return AUSSM_E_NULL;
  return run_neg_exp(a_log, dA, out, n, (hipStream_t)stream);
}
int aussm_zero_many(float* const* p, const size_t* n, int count, void* stream) {
  if (!p || !n) return AUSSM_E_NULL;
  if (count < 0 || count > FILL_MAX) return AUSSM_E_SHAPE;
  FillArgs f{};
  for (int i = 0; i < count; ++i) {
    if (!n[i]) continue;
    if (!p[i]) return AUSSM_E_NULL;
    if (misaligned(p[i], 4)) return AUSSM_E_ALIGN;
    f.dst[f.count] = p[i]; f.src[f.count] = nullptr; f.n[f.count] = n[i]; ++f.count;
  }
  return run_fill(f, (hipStream_t)stream);
}

int aussm_zero_f32(float* p, size_t n, void* stream) {
  if (!p) return AUSSM_E_NULL;
  if (misaligned(p, 4)) return AUSSM_E_ALIGN;
  return aussm_zero_many(&p, &n, 1, stream);
}

// ---- the reference's operator extension_cpp::ssm_adaptive_unitary as fused kernels (dropin.h)

// blocks of 16 states per channel, one per wavefront: 1, 2 or 4 (they have to divide the wavefronts of a workgroup)
static int dropin_state_blocks(int n) { const int k = (n + 15) / 16; return k == 3 ? 4 : k; }
static size_t dropin_xp_floats(int d, int n) { return (size_t)d * dropin_state_blocks(n) * dropin_records((d + 31) / 32, (d + 31) / 32) * 4; }
// The backward call works through the (batch, sequence) plane in blocks of bg batch elements x ct tiles
// of 16 timesteps: the workspace holds the phase adjoints of one block (about 100 MiB at most:
// at b = 32, d = 256, n = 16, L = 720 a block of 8 batch elements then spans the whole sequence, 1.39 ms per backward
// call against 1.64 ms with 50 MiB blocks).  bg is
// what fills the chip with one workgroup per compute unit (fewer would idle units, more would only
// shorten the blocks and repeat the per-launch set-up, the rows of x among it, more often).
// budget of a block (phase adjoints; prepared tiles of u), in floats
// (the option can only lower it: the workspace query sizes for the full budget, so a buffer obtained under
// one setting of the option holds what a call under any other setting uses)
constexpr int DROPIN_BLOCK_KFLOATS = 25600;
static size_t dropin_block_floats(bool largest) {
  const int o = opt(AUSSM_OPT_BLOCK_KFLOATS);
  return (size_t)(!largest && o > 0 && o < DROPIN_BLOCK_KFLOATS ? o : DROPIN_BLOCK_KFLOATS) << 10;
}
struct DropinBlocks { int bg, ct; };
static DropinBlocks dropin_blocks(int b, int d, int n, int L, bool largest = false) {
  const int nw = dropin_channels_per_workgroup((d + 31) / 32);
  const int wgs_per_b = (d * dropin_state_blocks(n) + nw - 1) / nw;
  int bg = (256 + wgs_per_b - 1) / wgs_per_b;
  if (bg > b) bg = b;
  const int ng = (b + bg - 1) / bg;
  bg = (b + ng - 1) / ng;
  const size_t per_tile = (size_t)bg * d * n * DT, cap = dropin_block_floats(largest);
  const int ntiles = (L + DT - 1) / DT;
  size_t tmax = cap / per_tile;
  if (tmax < 1) tmax = 1;
  const size_t nc = ((size_t)ntiles + tmax - 1) / tmax;
  return DropinBlocks{bg, (int)(((size_t)ntiles + nc - 1) / nc)};
}
static size_t round4(size_t v) { return (v + 3) & ~(size_t)3; }
static int dropin_check(int b, int d, int n, int L) {
  if (b < 1 || d < 1 || n < 1 || L < 1) return AUSSM_E_SHAPE;
  if (n > D_MAXN || d > 32 * D_MAXKS) return AUSSM_E_SHAPE;
  if ((long long)b * d > 0x7fffffffLL || (long long)d * n * L > 0x7fffffffLL) return AUSSM_E_SHAPE;
  return AUSSM_OK;
}

// floats of one prepared tile of u (all compiled steps of the contraction)
static size_t dropin_tile_floats(int d) { return dropin_records((d + 31) / 32, dropin_compiled_ks((d + 31) / 32)) * 4; }
// tiles per launch of the forward call: its prepared tiles of u (all batch elements) stay within the block budget
static int dropin_fwd_chunk_tiles(int b, int d, int L, bool largest = false) {
  const int ntiles = (L + DT - 1) / DT;
  size_t tmax = dropin_block_floats(largest) / ((size_t)b * dropin_tile_floats(d));
  if (tmax < 1) tmax = 1;
  const size_t nc = ((size_t)ntiles + tmax - 1) / tmax;
  return (int)(((size_t)ntiles + nc - 1) / nc);
}

// Tiles of a segment of a launch over nt tiles of `bg` batch elements (nt: one sweep).  As many segments as one workgroup per
// compute unit takes, two in the forward call up to d = 128, where registers leave room for them (16 x 64 pairs of 512 steps: 47 us
// in one sweep, 23 and 6 for the maps in four segments; 3 x 200: 30 in three segments, 39 in six), but at least two tiles each.
// The maps cost a third to a half of a sweep: two segments gain nothing (16 x 64 pairs, backward: 80 us, 60 and 22 in two), three
// do (3 x 200, 500 steps: 87, 46 and 25), and under 16 tiles their launch eats the rest (2 x 32 pairs, 7 tiles: 39 us both ways, 47
// in segments; 8 x 8, 16 tiles: 62, 49).  Those are kernels; whole passes, in one sweep / in segments, of 16 tiles: forward 8 x 16 22.6 /
// 15.1 us, 4 x 128 31.3 / 21.6, 16 x 64 28.0 / 25.7, but 3 x 200 41.0 / 42.0 (25 tiles of it: 55.5 / 52.5); with the gradients, where
// the host's launches set the time, 8 x 16 113-115 / 121, 2 x 32, 19 tiles 111-115 / 119-121, 31 tiles 117-122 / 119.
static int dropin_segment_tiles(int bg, int d, int n, int nt, bool backward) {
  const int nw = dropin_channels_per_workgroup((d + 31) / 32);
  const long wgs = (long)bg * ((d * dropin_state_blocks(n) + nw - 1) / nw);
  long most = (backward || d > 128 ? 256 : 512) / wgs;
  if (most > nt / 2) most = nt / 2;
  if (most < 3 || nt < 16) return nt;
  return (int)((nt + most - 1) / most);
}
// floats per state of a launch's maps, (E, F) each, backward also A, and the state and adjoint at the end
static size_t dropin_segment_floats(int bg, int d, int n, int nt, bool backward) {
  const int sl = dropin_segment_tiles(bg, d, n, nt, backward), nseg = (nt + sl - 1) / sl;
  return nseg < 2 ? 0 : (size_t)bg * d * n * (backward ? 6 * (size_t)nseg + 4 : 4 * (size_t)nseg);
}

size_t aussm_ssm_adaptive_unitary_workspace_floats(int b, int d, int n, int L, int backward) {
  if (dropin_check(b, d, n, L) != AUSSM_OK) return 0;
  size_t f = dropin_xp_floats(d, n);
  if (backward) {
    const DropinBlocks k = dropin_blocks(b, d, n, L, true);
    f += 2 * round4((size_t)b * d * n) + (size_t)k.bg * k.ct * DT * d * n + (size_t)k.bg * k.ct * dropin_tile_floats(d);
    f += dropin_segment_floats(k.bg, d, n, k.ct, true);
  } else {
    const int ct = dropin_fwd_chunk_tiles(b, d, L, true);
    f += (size_t)b * ct * dropin_tile_floats(d);
    if (ct == (L + DT - 1) / DT) f += dropin_segment_floats(b, d, n, ct, false);
  }
  return f;
}

// The call as the reference's operator gives it: polar parameters as they are, x and x_bias [d, n, ..], z a tensor of its own
static aussm_operator_args operator_args(const float* u, const float* dt, const float* x, const float* x_bias, const float* B_r,
                                         const float* B_theta, const float* C_r, const float* C_theta, const float* D, const float* z,
                                         const float* h_re, const float* h_im, int b, int d, int n, int L) {
  aussm_operator_args p{};
  p.u = u; p.dt = dt; p.x = x; p.x_bias = x_bias; p.B_r = B_r; p.B_theta = B_theta; p.C_r = C_r; p.C_theta = C_theta;
  p.D = D; p.z = z; p.h_re = h_re; p.h_im = h_im;
  p.b = b; p.d = d; p.n = n; p.L = L; p.polar_stride = 1; p.x_scale = 1.0f;
  return p;
}
static int operator_check(const aussm_operator_args* p) {
  if (!p) return AUSSM_E_NULL;
  if (int e = dropin_check(p->b, p->d, p->n, p->L)) return e;
  if (!p->u || !p->dt || !p->x || !p->x_bias || !p->B_r || !p->B_theta || !p->C_r || !p->C_theta || !p->D || !p->z) return AUSSM_E_NULL;
  if ((p->h_re == nullptr) != (p->h_im == nullptr)) return AUSSM_E_NULL;
  if (p->polar_stride < 1 || p->z_batch_stride < 0) return AUSSM_E_SHAPE;
  return AUSSM_OK;
}
static DropinArgs dropin_args(const aussm_operator_args& p) {
  DropinArgs a{};
  a.u = p.u; a.dt = p.dt; a.z = p.z; a.x_bias = p.x_bias; a.B_r = p.B_r; a.B_th = p.B_theta; a.C_r = p.C_r; a.C_th = p.C_theta;
  a.Dp = p.D; a.h_re = p.h_re; a.h_im = p.h_im; a.d = p.d; a.n = p.n; a.L = p.L; a.ks = (p.d + 31) / 32; a.nb = dropin_state_blocks(p.n);
  a.xsi = p.x_state_major ? 1 : p.n; a.xsj = p.x_state_major ? p.d : 1;
  a.bcs = p.polar_stride; a.raw = p.radius_raw; a.zs = p.z_batch_stride ? (long)p.z_batch_stride : (long)p.d * p.L;
  return a;
}

static DropinPrepArgs dropin_prep_args(const aussm_operator_args& p, const DropinArgs& f, u4* xp, u4* up) {
  DropinPrepArgs a{};
  a.x = p.x; a.x_bias = p.x_bias; a.u = p.u; a.xp = xp; a.up = up; a.d = p.d; a.n = p.n; a.L = p.L; a.ks = f.ks; a.nb = f.nb;
  a.xsi = f.xsi; a.xsj = f.xsj; a.scale = p.x_scale;
  return a;
}

int aussm_operator_fwd(const aussm_operator_args* op, float* y, float* nh_re, float* nh_im, float* workspace, void* stream) {
  return aussm_operator_fwd_keep(op, y, nh_re, nh_im, workspace, nullptr, nullptr, stream);
}
int aussm_operator_fwd_keep(const aussm_operator_args* op, float* y, float* nh_re, float* nh_im, float* workspace, float* x_out, float* x_bias_out,
                            void* stream) {
  if (int e = operator_check(op)) return e;
  if (!y || !nh_re || !nh_im || !workspace) return AUSSM_E_NULL;
  if (misaligned(workspace, 16)) return AUSSM_E_ALIGN;
  hipStream_t s = (hipStream_t)stream;
  const int b = op->b, d = op->d, n = op->n, L = op->L, ntiles = (L + DT - 1) / DT;
  const int ct = dropin_fwd_chunk_tiles(b, d, L);
  DropinArgs a = dropin_args(*op);
  u4* xp = (u4*)workspace;
  u4* up = (u4*)(workspace + dropin_xp_floats(d, n));
  DropinPrepArgs pa = dropin_prep_args(*op, a, xp, up);
  pa.x_out = x_out; pa.xb_out = x_bias_out;
  a.y = y; a.nh_re = nh_re; a.nh_im = nh_im; a.xp = xp; a.up = up; a.b = b;
  const size_t nstate = (size_t)b * d * n;
  auto apart = [nstate](const float* p, const float* q) { return !p || p + nstate <= q || q + nstate <= p; };
  if (ct == ntiles && apart(op->h_re, nh_re) && apart(op->h_re, nh_im) && apart(op->h_im, nh_re) && apart(op->h_im, nh_im)) {
    // (the first segment still reads the state when the last one writes)
    const int sl = dropin_segment_tiles(b, d, n, ntiles, false);
    if (sl < ntiles) {
      a.nseg = (ntiles + sl - 1) / sl; a.sl = sl;
      a.seg = (f4*)((float*)up + (size_t)b * ct * dropin_tile_floats(d));
    }
  }
  // the sequence in chunks of ct tiles (one chunk unless it is long): prepared tiles of u for the chunk, then the
  // scan over it, the state handed from chunk to chunk in the output buffers
  for (int t0 = 0; t0 < ntiles; t0 += ct) {
    const int t1 = t0 + ct < ntiles ? t0 + ct : ntiles;
    pa.t0 = t0; pa.nt = t1 - t0;
    if (int e = run_dropin_prep(pa, b, t0 == 0, FillArgs{}, s)) return e;
    if (t0) { a.h_re = nh_re; a.h_im = nh_im; }
    a.up_t0 = t0; a.up_nt = t1 - t0; a.t0 = t0; a.t1 = t1;
    if (a.nseg > 1) {
      DropinBwdArgs q{};
      q.f = a; q.bg = b; q.t0 = t0; q.t1 = t1;
      if (int e = run_dropin_seg(q, s)) return e;
    }
    if (int e = run_dropin_fwd(a, s)) return e;
  }
  return AUSSM_OK;
}

int aussm_ssm_adaptive_unitary_fwd(const float* u, const float* dt, const float* x, const float* x_bias,
                                   const float* B_r, const float* B_theta, const float* C_r, const float* C_theta,
                                   const float* D, const float* z, const float* h_re, const float* h_im,
                                   float* y, float* nh_re, float* nh_im, float* workspace,
                                   int b, int d, int n, int L, void* stream) {
  if (int e = dropin_check(b, d, n, L)) return e;
  if (!h_re || !h_im) return AUSSM_E_NULL;
  const aussm_operator_args p = operator_args(u, dt, x, x_bias, B_r, B_theta, C_r, C_theta, D, z, h_re, h_im, b, d, n, L);
  return aussm_operator_fwd(&p, y, nh_re, nh_im, workspace, stream);
}

int aussm_operator_bwd(const aussm_operator_args* op, const float* grad_y, const float* grad_nh_re, const float* grad_nh_im,
                       const float* nh_re, const float* nh_im, const aussm_operator_grads* g, float* workspace, void* stream) {
  if (int e = operator_check(op)) return e;
  if (!grad_y || !g || !g->u || !g->dt || !g->x || !g->x_bias || !g->B_r || !g->B_theta || !g->C_r || !g->C_theta || !g->D || !g->z ||
      !g->h_re || !g->h_im || !workspace)
    return AUSSM_E_NULL;
  if (misaligned(workspace, 16)) return AUSSM_E_ALIGN;
  hipStream_t s = (hipStream_t)stream;
  const int b = op->b, d = op->d, n = op->n, L = op->L;
  const DropinBlocks blk = dropin_blocks(b, d, n, L);
  const int ct = blk.ct, lc = ct * DT, ntiles = (L + DT - 1) / DT;
  const size_t nstate = (size_t)b * d * n;
  u4* xp = (u4*)workspace;
  float* hc_re = workspace + dropin_xp_floats(d, n);
  float* hc_im = hc_re + round4(nstate);
  float* dth = hc_im + round4(nstate);
  u4* up = (u4*)(dth + (size_t)blk.bg * ct * DT * d * n);
  f4* seg = (f4*)((float*)up + (size_t)blk.bg * ct * dropin_tile_floats(d));
  DropinArgs f = dropin_args(*op);
  f.xp = xp; f.up = up;
  DropinPrepArgs pa = dropin_prep_args(*op, f, xp, up);
  FillArgs fa{};
  auto fill = [&](float* dst, const float* src, size_t cnt) {
    fa.dst[fa.count] = dst; fa.src[fa.count] = src; fa.n[fa.count] = cnt; ++fa.count;
  };
  const bool have_end = nh_re && nh_im;
  if (have_end) {
    fill(hc_re, nh_re, nstate);
    fill(hc_im, nh_im, nstate);
  }
  fill(g->h_re, grad_nh_re, nstate);                  // the adjoint of the state travels in the output buffers
  fill(g->h_im, grad_nh_im, nstate);
  // the accumulated gradients start from zero; the polar ones are interleaved where their stride says so
  fill(g->x, nullptr, (size_t)d * n * d);
  fill(g->x_bias, nullptr, (size_t)d * n);
  if (op->polar_stride == 1) {
    fill(g->B_r, nullptr, n);
    fill(g->B_theta, nullptr, n);
    fill(g->C_r, nullptr, n);
    fill(g->C_theta, nullptr, n);
  } else {
    fill(g->B_r, nullptr, (size_t)(n - 1) * op->polar_stride + 2);
    fill(g->C_r, nullptr, (size_t)(n - 1) * op->polar_stride + 2);
  }
  fill(g->D, nullptr, d);
  if (g->dt_bias) fill(g->dt_bias, nullptr, d);
  bool first = true;                                  // the call's first preparation sets the buffers and lays out x, too
  auto prepare = [&](int b0, int bg, int t0, int nt) {
    pa.b0 = b0; pa.t0 = t0; pa.nt = nt;
    const int e = run_dropin_prep(pa, bg, first, first ? fa : FillArgs{}, s);
    first = false;
    return e;
  };
  const long dn = (long)d * n;
  const DropinBlocks blk_most = dropin_blocks(b, d, n, L, true);
  const size_t segf = dropin_segment_floats(blk_most.bg, d, n, blk_most.ct, true);      // what the workspace has for segments
  for (int b0 = 0; b0 < b; b0 += blk.bg) {
    const int bg = b - b0 < blk.bg ? b - b0 : blk.bg;
    f.b = bg; f.b0 = b0; f.up_b0 = b0;
    if (!have_end) {
      // the state at the end of the sequence: a forward sweep without outputs over this group's chunks
      for (int t0 = 0; t0 < ntiles; t0 += ct) {
        const int t1 = t0 + ct < ntiles ? t0 + ct : ntiles;
        if (int e = prepare(b0, bg, t0, t1 - t0)) return e;
        DropinArgs a = f;
        a.y = nullptr; a.nh_re = hc_re; a.nh_im = hc_im;
        if (t0) { a.h_re = hc_re; a.h_im = hc_im; }
        a.up_t0 = t0; a.up_nt = t1 - t0; a.t0 = t0; a.t1 = t1;
        if (int e = run_dropin_fwd(a, s)) return e;
      }
    }
    // the chunks in reverse: chunk c covers the tiles c ct .. (same cuts as the forward sweep above)
    for (int t0 = ((ntiles - 1) / ct) * ct; t0 >= 0; t0 -= ct) {
      const int t1 = t0 + ct < ntiles ? t0 + ct : ntiles;
      const int l0 = t0 * DT, len = (t1 * DT < L ? t1 * DT : L) - l0;
      if (int e = prepare(b0, bg, t0, t1 - t0)) return e;
      DropinBwdArgs q{};
      q.f = f;
      q.f.up_t0 = t0; q.f.up_nt = t1 - t0;
      q.gy = grad_y; q.hc_re = hc_re; q.hc_im = hc_im; q.dth = dth;
      q.du = g->u; q.ddt = g->dt; q.dz = g->z; q.dxb = g->x_bias;
      q.dB_r = g->B_r; q.dB_th = g->B_theta; q.dC_r = g->C_r; q.dC_th = g->C_theta; q.dD = g->D;
      q.dh_re = g->h_re; q.dh_im = g->h_im; q.b0 = b0; q.bg = bg; q.t0 = t0; q.t1 = t1; q.lc = lc;
      q.dt_act = op->dt_softplus; q.ddtb = g->dt_bias; q.ddtb_scale = op->dt_bias_scale;
      const int nt = t1 - t0, sl = dropin_segment_tiles(bg, d, n, nt, true), nseg = (nt + sl - 1) / sl;
      if (nseg > 1 && dropin_segment_floats(bg, d, n, nt, true) <= segf) {
        const size_t per = (size_t)bg * d * n;
        q.f.nseg = nseg; q.f.sl = sl; q.f.seg = seg;
        q.ent = seg + nseg * per; q.sega = (float2*)(q.ent + per);
        if (int e = run_dropin_seg(q, s)) return e;
      }
      if (int e = run_dropin_bwd(q, s)) return e;
      // grad_u[b, r, l0 + l] += scale sum_(i j) x[(i j), r] hat theta[b, (i j), l]   (rows (i j) in the order of x)
      XGemmArgs gu{};
      gu.A = op->x; gu.sam = 1; gu.sak = d;
      gu.B = dth; gu.sbk = lc; gu.sbn = 1; gu.sbb = dn * lc;
      gu.C = g->u + (size_t)b0 * d * L + l0; gu.scm = L; gu.scn = 1; gu.scb = (long)d * L;
      gu.M = d; gu.N = bg * len; gu.K = (int)dn; gu.Z = 1; gu.nper = len; gu.reduce = 1; gu.alpha = op->x_scale;
      if (int e = run_xgemm(gu, s)) return e;
      // grad_x[(i j), r] += scale sum_b sum_l hat theta[b, (i j), l] u[b, r, l0 + l]
      XGemmArgs gx{};
      gx.A = dth; gx.sam = lc; gx.sak = 1; gx.saz = dn * lc;
      gx.B = op->u + (size_t)b0 * d * L + l0; gx.sbk = 1; gx.sbn = L; gx.sbz = (long)d * L;
      gx.C = g->x; gx.scm = d; gx.scn = 1;
      gx.M = (int)dn; gx.N = d; gx.K = len; gx.Z = bg; gx.nper = d; gx.reduce = 1; gx.alpha = op->x_scale;
      if (int e = run_xgemm(gx, s)) return e;
    }
  }
  return AUSSM_OK;
}

int aussm_ssm_adaptive_unitary_bwd(const float* grad_y, const float* grad_nh_re, const float* grad_nh_im,
                                   const float* u, const float* dt, const float* x, const float* x_bias,
                                   const float* B_r, const float* B_theta, const float* C_r, const float* C_theta,
                                   const float* D, const float* z, const float* h_re, const float* h_im,
                                   const float* nh_re, const float* nh_im,
                                   float* du, float* ddt, float* dx, float* dx_bias, float* dB_r, float* dB_theta,
                                   float* dC_r, float* dC_theta, float* dD, float* dz, float* dh_re, float* dh_im,
                                   float* workspace, int b, int d, int n, int L, void* stream) {
  if (int e = dropin_check(b, d, n, L)) return e;
  if (!h_re || !h_im) return AUSSM_E_NULL;
  const aussm_operator_args p = operator_args(u, dt, x, x_bias, B_r, B_theta, C_r, C_theta, D, z, h_re, h_im, b, d, n, L);
  aussm_operator_grads g{};
  g.u = du; g.dt = ddt; g.x = dx; g.x_bias = dx_bias; g.B_r = dB_r; g.B_theta = dB_theta; g.C_r = dC_r; g.C_theta = dC_theta;
  g.D = dD; g.z = dz; g.h_re = dh_re; g.h_im = dh_im;
  return aussm_operator_bwd(&p, grad_y, grad_nh_re, grad_nh_im, nh_re, nh_im, &g, workspace, stream);
}

}  // extern "C"
