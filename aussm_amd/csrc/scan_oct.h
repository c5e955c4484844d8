// Vector-ALU scans, one wavefront per eight channels (all three variants, forward and reverse).
//
// Work split.  A workgroup of eight wavefronts owns (batch element or segment, 64 consecutive channels); wavefront w owns
// the eight channels d0 + 8 w .. + 7 with ALL their states.  Lane = 8 c + g is channel c of them and state group g, the
// states n = 8 s + g, s < S.  So
//   * the sums over the states (y, and in the reverse scan dw, ddelta / dtheta / drho) stay inside the wavefront: S of
//     them in registers, eight lanes by DPP (state_sums), with eight steps at a time so that every lane ends with one step;
//   * what a channel brings per step (u, delta, theta, rho, z, dy) is read, converted and stored by its own eight lanes, four
//     consecutive steps each (16-byte accesses, 128 bytes a row and tile of 32 steps), and passes through LDS that no other
//     wavefront touches: no barrier between staging, scan and output;
//   * B_t and C_t of a tile lie in LDS once per workgroup, a tile ahead, as rows [n][t] read 16 bytes at a time;
//   * in the reverse scan the sums over the channels behind dB_t, dC_t are taken over the wavefront's eight on the vector ALU
//     (channel_sums) and over the eight wavefronts through two alternating slabs in LDS; one barrier per 16 steps.
// In the split before this one (a wavefront = 64 channels x 2 states, B_t and C_t as scalar operands) every step's sums over
// the states went through LDS, two barriers per 16 steps held all wavefronts of the compute unit together, and up to 118
// scalar registers lived in vector lanes.  What bounds these kernels now is vector instructions: per state and step S6 7.5
// forward and 22 backward, complex 14 and 40, the vector ALU busy 68-82 % of the time.  Two wavefronts per SIMD hide an LDS
// read only if it is asked for a turn ahead of its use (forward kernel 213 -> 182 us, complex backward 967 -> 884).
// Forward and backward pass before and after, us, B32 D512 N16 L2048: S6 bf16 834 -> 630, complex 1493 -> 1040; S6 gated, softplus,
// L720 377 -> 290; unitary gated, B5 D200 N24 L1001 228 -> 126.
//
// Reference semantics: extension-cpp/extension_cpp/ops.py:215-223 (unitary loop), :270-291 (complex loop), :349-356 (real
// loop), the selective-scan call at ai-modules/wavesAI/model/aussm.py:791-802; gradient structure of
// extension-cpp/extension_cpp/csrc/cuda/ssm_adaptive_complex.cu:358-660 and ssm_adaptive_real.cu:267-488.
#pragma once
#include <type_traits>

#include "scan_common.h"

namespace aussm {

constexpr int OT = 32;           // steps per staged tile
constexpr int OG = 8;            // steps per group: sums are taken eight steps at a time
constexpr int OP = OT + 4;       // row stride of a wavefront's [channel][t] planes: eight rows of 16 bytes in distinct banks

// Workgroup barrier that publishes LDS contents only (__syncthreads() also waits for every load and store in flight).
__device__ __forceinline__ void oct_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// Orders LDS accesses of a wavefront for the compiler; the hardware executes them in order.
__device__ __forceinline__ void oct_wave_fence() { asm volatile("" ::: "memory"); }

// out[j]: a[j] + its partner's a[j] in the lanes of banks (four lanes) LOW, b[j] + its partner's b[j] in the others.  Two instructions
// that write their banks only, where selecting both summands takes two more at twice the price of an addition (a DPP addition
// and a select by a scalar mask take 5 cycles each); one wait for all sources.  S6, 32 x 512 x 16, 2048 steps: see below.
#define OCT_PAIR(CTRL_, LOW_, HIGH_, o_, a_, b_)                                                      \
  "v_add_f32_dpp " o_ ", " a_ ", " a_ " " CTRL_ " row_mask:0xf bank_mask:" LOW_ "\n\t"                  \
  "v_add_f32_dpp " o_ ", " b_ ", " b_ " " CTRL_ " row_mask:0xf bank_mask:" HIGH_ "\n\t"
__device__ __forceinline__ void bank_sums(const float (&v)[8], float (&q)[4]) {   // lane bit 2
#define P_(o_, a_, b_) OCT_PAIR("row_half_mirror", "0x5", "0xa", o_, a_, b_)
  asm("s_nop 1\n\t" P_("%0", "%4", "%8") P_("%1", "%5", "%9") P_("%2", "%6", "%10") P_("%3", "%7", "%11")
      : "=&v"(q[0]), "=&v"(q[1]), "=&v"(q[2]), "=&v"(q[3])
      : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]));
}
__device__ __forceinline__ void bank_sums(const float (&v)[4], float (&q)[2]) {
  asm("s_nop 1\n\t" P_("%0", "%2", "%4") P_("%1", "%3", "%5")
      : "=&v"(q[0]), "=&v"(q[1]) : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]));
#undef P_
}
__device__ __forceinline__ float bank_sum8(float a, float b) {                    // lane bit 3
  float o;
  asm("s_nop 1\n\t" OCT_PAIR("row_ror:8", "0x3", "0xc", "%0", "%1", "%2") : "=&v"(o) : "v"(a), "v"(b));
  return o;
}
#undef OCT_PAIR

// Sums over the eight channels of a wavefront (lane bits 3 .. 5) of eight values: lane 8 c + g returns the total of v[c]
// over the lanes 8 * + g.  14 instructions: two rounds of row swaps, one rotation by half a row.
__device__ __forceinline__ float channel_sums(const float (&v)[8]) {
  float q[4], r[2];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float a = v[j], b = v[j + 4];
    rows_swap32(a, b);
    q[j] = a + b;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    float a = q[j], b = q[j + 2];
    rows_swap16(a, b);
    r[j] = a + b;
  }
  return bank_sum8(r[0], r[1]);
}
// Sums over the eight state groups of a channel (lane bits 0 .. 2): lane 8 c + g returns the total of v[g] over the lanes
// 8 c + *.  The first step takes the mirrored lane of the half row, whose pairs the two steps inside the quads complete.
__device__ __forceinline__ float state_sums(const float (&v)[8], bool bit1, bool bit0) {
  float q[4], r[2];
  bank_sums(v, q);
#pragma unroll
  for (int j = 0; j < 2; ++j) r[j] = (bit1 ? q[j + 2] : q[j]) + dpp_perm<0x4E>(bit1 ? q[j] : q[j + 2]);    // quad_perm:[2,3,0,1]
  return (bit0 ? r[1] : r[0]) + dpp_perm<0xB1>(bit0 ? r[0] : r[1]);                                        // quad_perm:[1,0,3,2]
}
// The same sums of four values: lanes 8 c + g with bits 1 and 2 of c (of g) equal to j return the total of v[j] (7 and 8
// instructions; where registers for eight steps at a time are not there).
__device__ __forceinline__ float channel_sums(const float (&v)[4]) {
  float q[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    float a = v[j], b = v[j + 2];
    rows_swap32(a, b);
    q[j] = a + b;
  }
  rows_swap16(q[0], q[1]);
  const float r = q[0] + q[1];
  return r + dpp_perm<0x128>(r);
}
__device__ __forceinline__ float state_sums(const float (&v)[4], bool bit1, bool) {
  float q[2];
  bank_sums(v, q);
  const float r = (bit1 ? q[1] : q[0]) + dpp_perm<0x4E>(bit1 ? q[0] : q[1]);
  return r + dpp_perm<0xB1>(r);
}
// ... of one value (or the product of complex values), in every lane of the channel
__device__ __forceinline__ float group_sum(float v) {
  v += dpp_perm<0x141>(v);
  v += dpp_perm<0x4E>(v);
  return v + dpp_perm<0xB1>(v);
}
__device__ __forceinline__ void group_product(float& re, float& im) {
  auto step = [&](float pr, float pi) {
    const float x = fmaf(re, pr, -im * pi);
    im = fmaf(re, pi, im * pr);
    re = x;
  };
  step(dpp_perm<0x141>(re), dpp_perm<0x141>(im));
  step(dpp_perm<0x4E>(re), dpp_perm<0x4E>(im));
  step(dpp_perm<0xB1>(re), dpp_perm<0xB1>(im));
}

// An offset the compiler takes as new: the addresses of a tile's accesses are formed where they are used (one instruction
// each) instead of being kept, two registers a tensor, across the loop.
__device__ __forceinline__ size_t fresh(size_t o) {
  asm volatile("" : "+v"(o));
  return o;
}

// sin and cos of a lane's four steps: one check for the four
__device__ __forceinline__ void sincos4(const float (&x)[4], f4& sn, f4& cs) {
  float s_[4], c_[4];
  const float m = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
  if (__builtin_expect(__any(m > 1.0e4f), 0)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) fast_sincosf(x[i], &s_[i], &c_[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) sincos_1e4(x[i], &s_[i], &c_[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) { sn[i] = s_[i]; cs[i] = c_[i]; }
}

// The options of the S6 scan for a lane's four steps, behind one uniform branch each (the fence keeps the compiler from
// working them out for every call and selecting: a fifth of the forward kernel's instructions)
__device__ __forceinline__ void silu4(float (&v)[4]) {
  asm volatile("");
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = siluf_(v[i]);
}
__device__ __forceinline__ void softplus4(float (&v)[4]) {
  asm volatile("");
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = softplusf_(v[i]);
}

// One record of B_t / C_t as loaded: real or (re, im)
template <int C, typename T_> struct BcRec;
template <> struct BcRec<1, float> {
  float v;
  __device__ __forceinline__ void load(const float* p, size_t i) { v = p[i]; }
  __device__ __forceinline__ void put(float* o, bool ok) const { *o = ok ? v : 0.f; }
  __device__ __forceinline__ void touch() const { touch_vgpr(v); }
};
template <> struct BcRec<1, bf16_t> {
  bf16_t v;
  __device__ __forceinline__ void load(const bf16_t* p, size_t i) { v = p[i]; }
  __device__ __forceinline__ void put(float* o, bool ok) const { *o = ok ? to_f32(v) : 0.f; }
  __device__ __forceinline__ void touch() const { touch_vgpr(v); }
};
template <> struct BcRec<2, float> {
  float2 v;
  __device__ __forceinline__ void load(const float* p, size_t i) { v = *reinterpret_cast<const float2*>(p + 2 * i); }
  __device__ __forceinline__ void put(float* o, bool ok) const { *reinterpret_cast<float2*>(o) = ok ? v : make_float2(0.f, 0.f); }
  __device__ __forceinline__ void touch() const { touch_vgpr(v.x); touch_vgpr(v.y); }
};
template <> struct BcRec<2, bf16_t> {
  uint32_t v;
  __device__ __forceinline__ void load(const bf16_t* p, size_t i) { v = *reinterpret_cast<const uint32_t*>(p + 2 * i); }
  __device__ __forceinline__ void put(float* o, bool ok) const {
    *reinterpret_cast<float2*>(o) = ok ? make_float2(__uint_as_float(v << 16), __uint_as_float(v & 0xffff0000u)) : make_float2(0.f, 0.f);
  }
  __device__ __forceinline__ void touch() const { touch_vgpr(__uint_as_float(v)); }
};

// G consecutive steps of a row in LDS (16-byte reads)
template <int G>
__device__ __forceinline__ void ld_steps(float (&o)[G], const float* p) {
#pragma unroll
  for (int j = 0; j < G / 4; ++j) {
    const f4 a = *reinterpret_cast<const f4*>(p + 4 * j);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[4 * j + i] = a[i];
  }
}
template <int C, int G>
__device__ __forceinline__ void ld_rec(float (&re)[G], float (&im)[G], const float* p) {
  if constexpr (C == 1) {
    ld_steps(re, p);
  } else {
#pragma unroll
    for (int j = 0; j < G / 2; ++j) {
      const f4 a = *reinterpret_cast<const f4*>(p + 4 * j);
      re[2 * j] = a[0]; im[2 * j] = a[1]; re[2 * j + 1] = a[2]; im[2 * j + 1] = a[3];
    }
  }
}

// Rows of B_t and / or C_t: NK tensors x 8 S rows x RB steps, loaded and put into LDS by 512 threads.
template <int C, int S, int NK, int RB, typename Tbc>
struct OctRows {
  static constexpr int RS = RB * C + 4;                   // row stride in floats
  static constexpr int FLOATS = NK * 8 * S * RS;
  static constexpr int REC = NK * 8 * S * RB;
  static constexpr int PER = (REC + 511) / 512;
  BcRec<C, Tbc> v[PER];
  // row0: first record of row 0 at step 0 of the segment
  __device__ __forceinline__ void load(const Tbc* gB, const Tbc* gC, size_t row0, int ld, int l0, int L, int N, int tid) {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = tid + 512 * k, t = e % RB, r = e / RB;
      const int kind = NK == 2 ? (r >= 8 * S) : 0;
      int n = r - kind * 8 * S;
      n = n < N ? n : N - 1;
      const int l = l0 + t < L ? l0 + t : L - 1;
      v[k].load((NK == 1 || kind) ? gC : gB, row0 + (size_t)n * ld + l);
    }
  }
  __device__ __forceinline__ void touch() const {
#pragma unroll
    for (int k = 0; k < PER; ++k) v[k].touch();
  }
  // rows that do not exist and steps past the end are zero (never a clamped row's infinity)
  __device__ __forceinline__ void put(float* dst, int l0, int L, int N, int tid) const {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = tid + 512 * k, t = e % RB, r = e / RB;
      const int n = NK == 2 && r >= 8 * S ? r - 8 * S : r;
      if (REC % 512 == 0 || e < REC) v[k].put(dst + r * RS + t * C, n < N && l0 + t < L);
    }
  }
};

// The states are worked out here.  (Without the sums' stores nothing kept a pass without outputs from reading a whole tile's
// rows ahead: 220 spilled registers at 64 states.)
__device__ __forceinline__ void pin(float& a, float& b) { asm volatile("" : "+v"(a), "+v"(b) : : "memory"); }

// Inputs and results move four steps a lane at a time wherever a row starts; single elements are left to a last tile whose
// length is no multiple of four.  (With a second path for rows that do not start on 16 bytes: 8 x 256 x 16, 2957 steps, bf16,
// complex with the gate 395 us, now 342, S6 278 -> 246; and the longer code cost whole rows, too, 32 x 512 x 16, 2048 steps,
// complex 1133 -> 1046.)

// S: state groups of eight (8 S >= N).  FULLN: N = 8 S.  LEAN: no outputs but the end state and the product of the a_l (the
// first pass of a call that is split along the sequence).
template <int VAR, int S, bool FULLN, typename Tin, typename Tbc, bool LEAN>
__global__ __launch_bounds__(512) void oct_fwd_kernel(const FwdArgs p) {
  constexpr int C = VAR == VAR_REAL ? 1 : 2;
  constexpr int NK = LEAN ? 1 : 2;
  constexpr int NPL = VAR == VAR_REAL ? 2 : 3;             // planes: real (delta, w), else (Re a, Im a, w)
  constexpr int PW = NPL - 1;
  constexpr int G = C == 2 && S > 3 ? 4 : OG;              // steps at a time
  constexpr int RB = S <= 2 ? 2 * OT : OT;                 // steps of B_t, C_t in LDS at a time (twice): a barrier per RB steps
  using Rows = OctRows<C, S, NK, RB, Tbc>;
  __shared__ __align__(16) float s_bc[2][Rows::FLOATS];
  __shared__ __align__(16) float s_in[2][8][NPL][8 * OP];  // a tile being worked on, the next one being staged

  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
  const int c = lane >> 3, g = lane & 7;
  const bool bit1 = g & 2, bit0 = g & 1;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);
  const int vb = wg / p.ncg, d0 = (wg % p.ncg) * CH;
  const int b = vb / p.ns, sg = vb - b * p.ns;
  const int lbeg = sg * p.L, ld = p.ld;
  const int N = p.N, D = p.D;
  const int L = (ld - lbeg < p.L) ? ld - lbeg : p.L;       // steps of this segment
  const int d = d0 + 8 * wave + c;
  const bool dok = d < D, live = d0 + 8 * wave < D;        // live: wave-uniform
  const int dd = dok ? d : D - 1;

  const size_t uback = (size_t)(b - b / p.urep) * D * ld;  // (u, delta of [B / urep, D, L])
  const Tin* __restrict__ gu = static_cast<const Tin*>(p.u) - uback;
  const Tin* __restrict__ gdl = static_cast<const Tin*>(p.delta) - uback;
  const Tbc* __restrict__ gB = static_cast<const Tbc*>(p.Bm);
  const Tbc* __restrict__ gC = static_cast<const Tbc*>(LEAN ? p.Bm : p.Cm);
  const size_t goff = ((size_t)b * D + dd) * ld + lbeg;
  const size_t bc_row = (size_t)b * ((VAR == VAR_REAL && p.bcrows) ? p.bcrows : N) * ld + lbeg;
  const bool gated = !LEAN && p.z != nullptr;
  const float* __restrict__ gz = gated ? p.z + ((VAR == VAR_REAL && p.zrows) ? (size_t)b * (p.zrows - D) * ld : 0) : nullptr;

  float hr[S], hi[S], a2[S], mr[S], mi[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int n = 8 * s + g;
    hr[s] = 0.f; hi[s] = 0.f; a2[s] = 0.f; mr[s] = 0.f; mi[s] = 0.f;
    if (dok && n < N) {
      if (p.h0) {
        const size_t o = (((size_t)b * D + d) * N + n) * C;
        hr[s] = p.h0[o];
        if (C == 2) hi[s] = p.h0[o + C - 1];
      }
      if (VAR == VAR_REAL) a2[s] = p.A[(size_t)d * N + n] * LOG2E;
    }
  }
  if (!LEAN && p.seg && live) {
    int nn[S];
#pragma unroll
    for (int s = 0; s < S; ++s) nn[s] = 8 * s + g < N ? 8 * s + g : N - 1;
    const size_t e = (size_t)b * p.ns * D + dd;
    seg_chain<VAR, false, S>(p.seg + e * N * C, p.segq + e * 2, (ptrdiff_t)D * N * C, (ptrdiff_t)D * 2, sg, nn, a2, hr, hi);
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (8 * s + g >= N) { hr[s] = 0.f; hi[s] = 0.f; }
  }
  // Lanes without a state take no part in the sums over the states (their C is zero, but their state, from infinite inputs or
  // decays times zeros, may be a NaN).  They lie in the last group, with registers for 48 or 64 states in the last two.
  constexpr int WHOLE_S = FULLN ? S : S > 4 ? S - 2 : S - 1;   // groups whose lanes all have a state
  bool has[S - WHOLE_S > 0 ? S - WHOLE_S : 1];
#pragma unroll
  for (int s = WHOLE_S; s < S; ++s) has[s - WHOLE_S] = 8 * s + g < N;
  const float dsk = (!LEAN && p.Dskip && dok) ? p.Dskip[dd] : 0.f;
  const float dbias = (VAR == VAR_REAL && p.delta_bias && dok) ? p.delta_bias[dd] : 0.f;

  // two sets of loaded inputs: `rdy` has landed and is staged next, `fly` is a tile behind it
  struct Raw { Quad<Tin> u, dl; Quad<float> th, rho, z; } rdy, fly;
  fly.u.zero(); fly.dl.zero(); fly.th.zero(); fly.rho.zero(); fly.z.zero();
  auto load_tile = [&](Raw& raw, int l0) {
    const int ll = l0 + 4 * g;
    int idx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) idx[i] = ll + i < L ? ll + i : L - 1;
    const bool vec = l0 + OT <= L || L % 4 == 0;             // uniform: a lane's four steps exist or none
    const size_t o = fresh(goff + (vec ? min(ll, L - 4) : 0));
    raw.u.load(gu, o, vec, idx);
    raw.dl.load(gdl, o, vec, idx);
    if (VAR != VAR_REAL) raw.th.load(p.theta, o, vec, idx);
    if (VAR == VAR_COMPLEX) raw.rho.load(p.rho, o, vec, idx);
    if (gated) raw.z.load(gz, o, vec, idx);
  };
  Rows rows;
  auto land = [&]() {                                      // everything in flight has landed; fly becomes rdy
    fly.u.touch(); fly.dl.touch();
    if (VAR != VAR_REAL) fly.th.touch();
    if (VAR == VAR_COMPLEX) fly.rho.touch();
    if (gated) fly.z.touch();
    rows.touch();
    rdy = fly;
  };
  float pr = VAR == VAR_REAL ? 0.f : 1.f, pi = 0.f;        // LEAN: product of the lane's a_l / sum of its step sizes
  constexpr int PL = 8 * OP;
  float yin[4], gate[4], ynext[4], gnext[4];               // D u and z of the tile being worked on, of the one staged
  // the loaded inputs of the tile at l0 become what the scan reads
  // (whole: all of the tile's steps and of the wavefront's channels exist)
  auto stage_as = [&](int l0, int buf, auto whole) {
    constexpr bool WHOLE = decltype(whole)::value;
    f4 o0, o1, o2;
    float th[4];
    f4 sn, cs;
    bool ok[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ok[i] = WHOLE || (dok && l0 + 4 * g + i < L);
      th[i] = VAR != VAR_REAL && ok[i] ? rdy.th.get(i) : 0.f;
    }
    if constexpr (VAR != VAR_REAL) sincos4(th, sn, cs);
    float u4_[4], d4[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u4_[i] = ok[i] ? rdy.u.get(i) : 0.f;
      d4[i] = ok[i] ? rdy.dl.get(i) : 0.f;
      if (VAR == VAR_REAL) d4[i] += dbias;
    }
    if (VAR == VAR_REAL && p.u_act) silu4(u4_);              // uniform
    if (VAR == VAR_REAL && p.delta_softplus) softplus4(d4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float uu = u4_[i], dl = ok[i] ? d4[i] : 0.f;
      if (VAR == VAR_REAL) {
        o0[i] = dl; o1[i] = dl * uu;
        if (LEAN) pr += dl;
      } else {
        if (VAR == VAR_COMPLEX) { const float r = expf(ok[i] ? rdy.rho.get(i) : 0.f); cs[i] *= r; sn[i] *= r; }
        o0[i] = cs[i]; o1[i] = sn[i]; o2[i] = dl * uu;
        if (LEAN) { const float x = fmaf(pr, cs[i], -pi * sn[i]); pi = fmaf(pr, sn[i], pi * cs[i]); pr = x; }
      }
      ynext[i] = dsk * uu;
      gnext[i] = rdy.z.get(i);
    }
    float* q = &s_in[buf][wave][0][c * OP + 4 * g];
    *reinterpret_cast<f4*>(q) = o0;
    *reinterpret_cast<f4*>(q + PL) = o1;
    if constexpr (NPL == 3) *reinterpret_cast<f4*>(q + 2 * PL) = o2;
  };
  const bool all_ch = d0 + 8 * wave + 8 <= D;
  auto stage = [&](int l0, int buf) {
    if (all_ch && l0 + OT <= L) stage_as(l0, buf, std::true_type{});
    else stage_as(l0, buf, std::false_type{});
  };

  rows.load(gB, gC, bc_row, ld, 0, L, N, tid);
  if (live) load_tile(fly, 0);
  rows.put(s_bc[0], 0, L, N, tid);
  if (live) land();
  if (RB < L) rows.load(gB, gC, bc_row, ld, RB, L, N, tid);
  if (live) {
    if (OT < L) load_tile(fly, OT);
    stage(0, 0);
    land();
    if (2 * OT < L) load_tile(fly, 2 * OT);
  }
  oct_barrier();

  for (int l0 = 0, it = 0; l0 < L; l0 += OT, ++it) {
    if (!live) rows.touch();
    // ---- the next rows, whose loads are RB steps old, into the other buffer; request the ones after
    const int rb = l0 / RB, lr = (rb + 1) * RB;
    if (l0 % RB == 0 && lr < L) {
      rows.put(s_bc[(rb + 1) & 1], lr, L, N, tid);
      if (lr + RB < L) rows.load(gB, gC, bc_row, ld, lr + RB, L, N, tid);
    }
    if (live) {
#pragma unroll
      for (int i = 0; i < 4; ++i) { yin[i] = ynext[i]; gate[i] = gnext[i]; }
      float* __restrict__ in = &s_in[it & 1][wave][0][c * OP];
      const float* __restrict__ bc = s_bc[rb & 1] + g * Rows::RS + (l0 % RB) * C;
      oct_wave_fence();
      // what a turn - one state group, G steps - reads
      struct Steps { float x0[G], x1[G], w[G]; } sp[2];
      struct RowsAt { float br[G], bi[G], cr[G], ci[G]; } rw[2];
      auto ld_planes = [&](Steps& o, int q) {
        const float* x = in + q * G;
        ld_steps(o.x0, x);
        if constexpr (NPL == 3) ld_steps(o.x1, x + PL);
        ld_steps(o.w, x + PW * PL);
      };
      auto ld_rows = [&](RowsAt& o, int q, int s) {
        ld_rec<C>(o.br, o.bi, bc + s * 8 * Rows::RS + q * G * C);
        if constexpr (!LEAN) ld_rec<C>(o.cr, o.ci, bc + (S + s) * 8 * Rows::RS + q * G * C);
      };
      float ya[G];
      auto turn = [&](const Steps& x, const RowsAt& r, int s, int steps) {
#pragma unroll
        for (int t = 0; t < G; ++t) {
          if (t >= steps) break;                             // uniform
          float yt;
          if constexpr (VAR == VAR_REAL) {
            const float a = __builtin_amdgcn_exp2f(x.x0[t] * a2[s]);
            hr[s] = fmaf(a, hr[s], r.br[t] * x.w[t]);
            if constexpr (!LEAN) yt = fmaf(r.cr[t], hr[s], ya[t]);
          } else {
            const float nr = fmaf(x.x0[t], hr[s], fmaf(-x.x1[t], hi[s], r.br[t] * x.w[t]));
            const float ni = fmaf(x.x0[t], hi[s], fmaf(x.x1[t], hr[s], r.bi[t] * x.w[t]));
            hr[s] = nr; hi[s] = ni;
            if constexpr (!LEAN) yt = fmaf(-r.ci[t], ni, fmaf(r.cr[t], nr, ya[t]));
          }
          if constexpr (!LEAN) ya[t] = s < WHOLE_S || has[s < WHOLE_S ? 0 : s - WHOLE_S] ? yt : ya[t];
        }
      };
      auto clear = [&]() {
#pragma unroll
        for (int t = 0; t < G; ++t) ya[t] = 0.f;
      };
      auto sums = [&](int q) {                               // (over what the group has read)
        if constexpr (!LEAN) in[q * G + (G == 8 ? g : g >> 1)] = state_sums(ya, bit1, bit0);
        else {
#pragma unroll
          for (int s = 0; s < S; ++s) pin(hr[s], hi[s]);
        }
      };
      constexpr int NQ = OT / G;
      const bool next = l0 + OT < L;
      if (l0 + OT <= L) {
        // every turn's operands are read a turn ahead: with two wavefronts per SIMD the LDS latency of every turn would show
        ld_planes(sp[0], 0);
        ld_rows(rw[0], 0, 0);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          clear();
#pragma unroll
          for (int s = 0; s < S; ++s) {
            const int k = q * S + s;
            if (s == S - 1 && q + 1 < NQ) ld_planes(sp[(q + 1) & 1], q + 1);
            if (k + 1 < NQ * S) ld_rows(rw[(k + 1) & 1], (k + 1) / S, (k + 1) % S);
            sched_fence();
            turn(sp[q & 1], rw[k & 1], s, G);
            sched_fence();
          }
          sums(q);
          if (q == NQ / 2 - 1) {
#pragma unroll
            for (int s = 0; s < S; ++s) { mr[s] = hr[s]; mi[s] = hi[s]; }
            // (the other half of the tile between what the next one writes to LDS and its first reads there)
            if (next) stage(l0 + OT, (it + 1) & 1);
          }
        }
      } else {
        // the last tile of a segment: steps past the end leave the state alone
#pragma unroll 1
        for (int q = 0; q < NQ && l0 + q * G < L; ++q) {
          if (q <= NQ / 2) {
#pragma unroll
            for (int s = 0; s < S; ++s) { mr[s] = hr[s]; mi[s] = hi[s]; }      // (what the first half of the tile leaves)
          }
          clear();
          ld_planes(sp[0], q);
#pragma unroll
          for (int s = 0; s < S; ++s) {
            ld_rows(rw[0], q, s);
            turn(sp[0], rw[0], s, L - (l0 + q * G));
          }
          sums(q);
        }
      }
      oct_wave_fence();
      // Loads, stores and atomics share one in-order counter: the wait for the loads, a tile old, comes in front of this
      // tile's stores and the next loads behind them, so that no wait has a fresh store to retire.
      land();
      if constexpr (!LEAN) {
        if (p.y) {
          const f4 ys = *reinterpret_cast<const f4*>(in + 4 * g);
          float acc[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            acc[i] = yin[i] + ys[i];
            if (gated) acc[i] *= siluf_(gate[i]);
          }
          const int nvalid = L - (l0 + 4 * g);
          if (dok && nvalid > 0) store4(p.y, fresh(goff + l0 + 4 * g), acc, true, nvalid);
        }
        // checkpoint at the end of every ck-step block (and at the end of the sequence); ck: a multiple of the tile or half of it
        if (p.hck && dok) {
          auto put = [&](int kb, const float (&xr)[S], const float (&xi)[S]) {
            const size_t base = fresh((((size_t)b * p.nck + sg * (p.L / p.ck) + kb) * N + g) * C * D + d);
#pragma unroll
            for (int s = 0; s < S; ++s) {
              if (8 * s + g < N) {
                const size_t o = base + (size_t)(8 * s * C) * D;
                p.hck[o] = xr[s];
                if (C == 2) p.hck[o + D] = xi[s];
              }
            }
          };
          const int tmax = L - l0 < OT ? L - l0 : OT;
          if (p.ck == OT / 2) {
            if (tmax > OT / 2) put(l0 / (OT / 2), mr, mi);
            put((l0 + tmax - 1) / (OT / 2), hr, hi);
          } else if (((l0 + OT) % p.ck) == 0 || l0 + OT >= L) {
            put(l0 / p.ck, hr, hi);
          }
        }
      }
      if (l0 + 3 * OT < L) load_tile(fly, l0 + 3 * OT);
    }
    if (l0 % RB == RB - OT) oct_barrier();
  }

  if constexpr (LEAN) {
    if (live) {
      if constexpr (VAR == VAR_REAL) pr = group_sum(pr);
      else group_product(pr, pi);
      if (dok && g == 0) {
        p.ptot[((size_t)vb * D + d) * 2] = pr;
        p.ptot[((size_t)vb * D + d) * 2 + 1] = pi;
      }
    }
  }
  if (p.clear && blockIdx.x == 0 && (tid == 0 || (tid >= AUX_IMG_FP && tid < AUX_IMG_FP + 8))) p.clear[tid] = 0.f;
  if (p.hL && dok && (LEAN || sg == p.ns - 1)) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int n = 8 * s + g;
      if (n < N) {
        const size_t o = (((size_t)(LEAN ? vb : b) * D + d) * N + n) * C;
        p.hL[o] = hr[s];
        if (C == 2) p.hL[o + 1] = hi[s];
      }
    }
  }
}

// ---- Splitting along the sequence.  With few (batch, channel group) pairs a launch leaves most of the chip idle, so the sequence
// is cut into ns segments and the scan runs over (batch, segment) pairs:
//   forward   1. oct_fwd_kernel over the pairs from a zero state, outputs off (LEAN): end state Z_k of every segment and the
//                product q_k of its a_l (FwdArgs::ptot),
//             2. oct_fwd_kernel over the pairs, each from  h <- q_k h + Z_k  over the segments before it (seg_chain);
//   backward  1. oct_adj_kernel: adjoint Y_k of the state entering every segment from a zero adjoint at its end (the reverse
//                recurrence alone - no states are needed for it), and q_k,
//             2. oct_bwd_kernel over the pairs, each from  g <- conj(q_k) g + Y_k  over the segments behind it.
// The reference itself does not split.
//
// Adjoint of the state that enters a segment, from a zero adjoint at its end, and the product of its a_l: the reverse
// recurrence  g <- conj(a_l) (g + conj(C_l) dy_l silu(z_l))  alone.
template <int VAR, int S, bool FULLN, typename Tin, typename Tbc>
__global__ __launch_bounds__(512) void oct_adj_kernel(const AdjSegArgs p) {
  constexpr int C = VAR == VAR_REAL ? 1 : 2;
  constexpr int NPL = VAR == VAR_REAL ? 2 : 3;             // planes: real (delta, dy), else (Re a, Im a, dy)
  constexpr int PW = NPL - 1;
  using Rows = OctRows<C, S, 1, OT, Tbc>;
  __shared__ __align__(16) float s_bc[2][Rows::FLOATS];
  __shared__ __align__(16) float s_in[8][NPL][8 * OP];

  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
  const int c = lane >> 3, g = lane & 7;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);
  const int vb = wg / p.ncg, d0 = (wg % p.ncg) * CH;
  const int b = vb / p.ns, sg = vb - b * p.ns;
  const int lbeg = sg * p.L, ld = p.ld;
  const int N = p.N, D = p.D;
  const int L = (ld - lbeg < p.L) ? ld - lbeg : p.L;
  const int d = d0 + 8 * wave + c;
  const bool dok = d < D, live = d0 + 8 * wave < D;
  const int dd = dok ? d : D - 1;
  const Tin* __restrict__ gdl = static_cast<const Tin*>(p.delta);
  const Tbc* __restrict__ gC = static_cast<const Tbc*>(p.Cm);
  const size_t goff = ((size_t)b * D + dd) * ld + lbeg;
  const size_t zoff = (VAR == VAR_REAL && p.zrows) ? (size_t)b * (p.zrows - D) * ld : 0;
  const size_t bc_row = (size_t)b * ((VAR == VAR_REAL && p.bcrows) ? p.bcrows : N) * ld + lbeg;
  const bool gated = p.z != nullptr;

  float gr[S], gi[S], a2[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int n = 8 * s + g;
    gr[s] = 0.f; gi[s] = 0.f;
    a2[s] = (VAR == VAR_REAL && dok && n < N) ? p.A[(size_t)d * N + n] * LOG2E : 0.f;
  }
  const float dbias = (VAR == VAR_REAL && p.delta_bias && dok) ? p.delta_bias[dd] : 0.f;
  struct Raw { Quad<Tin> dl; Quad<float> dy, th, rho, z; } raw;
  raw.dl.zero(); raw.dy.zero(); raw.th.zero(); raw.rho.zero(); raw.z.zero();
  auto load_tile = [&](int l0) {
    const int ll = l0 + 4 * g;
    int idx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) idx[i] = ll + i < L ? ll + i : L - 1;
    const bool vec = l0 + OT <= L || L % 4 == 0;
    const size_t o = goff + (vec ? min(ll, L - 4) : 0);
    raw.dy.load(p.dy, o, vec, idx);
    if (VAR == VAR_REAL) raw.dl.load(gdl, o, vec, idx);
    else raw.th.load(p.theta, o, vec, idx);
    if (VAR == VAR_COMPLEX) raw.rho.load(p.rho, o, vec, idx);
    if (gated) raw.z.load(p.z + zoff, o, vec, idx);
  };
  Rows rows;
  float pr = VAR == VAR_REAL ? 0.f : 1.f, pi = 0.f;
  float* __restrict__ in = &s_in[wave][0][0];
  constexpr int PL = 8 * OP;

  const int ntiles = (L + OT - 1) / OT;
  rows.load(gC, gC, bc_row, ld, (ntiles - 1) * OT, L, N, tid);
  if (live) load_tile((ntiles - 1) * OT);
  rows.put(s_bc[(ntiles - 1) & 1], (ntiles - 1) * OT, L, N, tid);
  if (ntiles > 1) rows.load(gC, gC, bc_row, ld, (ntiles - 2) * OT, L, N, tid);
  oct_barrier();
  for (int it = ntiles - 1; it >= 0; --it) {
    const int l0 = it * OT;
    if (live) {
      f4 o0, o1, o2;
      float d4[4];
      if constexpr (VAR == VAR_REAL) {
#pragma unroll
        for (int i = 0; i < 4; ++i) d4[i] = (l0 + 4 * g + i < L ? raw.dl.get(i) : 0.f) + dbias;
        if (p.delta_softplus) softplus4(d4);                 // uniform
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool ok = dok && l0 + 4 * g + i < L;
        float gy = ok ? raw.dy.get(i) : 0.f;
        if (gated) gy = ok ? gy * siluf_(raw.z.get(i)) : 0.f;
        if (VAR == VAR_REAL) {
          const float dl = ok ? d4[i] : 0.f;
          o0[i] = dl; o1[i] = gy;
          pr += dl;
        } else {
          float sn, cs;
          fast_sincosf(ok ? raw.th.get(i) : 0.f, &sn, &cs);
          if (VAR == VAR_COMPLEX) { const float r = expf(ok ? raw.rho.get(i) : 0.f); cs *= r; sn *= r; }
          o0[i] = cs; o1[i] = sn; o2[i] = gy;
          const float x = fmaf(pr, cs, -pi * sn);
          pi = fmaf(pr, sn, pi * cs);
          pr = x;
        }
      }
      float* q = in + c * OP + 4 * g;
      *reinterpret_cast<f4*>(q) = o0;
      *reinterpret_cast<f4*>(q + PL) = o1;
      if constexpr (NPL == 3) *reinterpret_cast<f4*>(q + 2 * PL) = o2;
      if (it > 0) load_tile(l0 - OT);
    }
    if (it > 0) {
      rows.put(s_bc[(it - 1) & 1], l0 - OT, L, N, tid);
      if (it > 1) rows.load(gC, gC, bc_row, ld, l0 - 2 * OT, L, N, tid);
    }
    if (live) {
      oct_wave_fence();
      const float* __restrict__ bc = s_bc[it & 1] + g * Rows::RS;
      auto group = [&](int q, auto tail_tag) {
        constexpr bool TAIL = decltype(tail_tag)::value;
        float x0[8], x1[8], w[8];
        const float* x = in + c * OP + q * OG;
        ld_steps(x0, x);
        if constexpr (NPL == 3) ld_steps(x1, x + PL);
        ld_steps(w, x + PW * PL);
#pragma unroll
        for (int s = 0; s < S; ++s) {
          float cr[8], ci[8];
          ld_rec<C>(cr, ci, bc + s * 8 * Rows::RS + q * OG * C);
#pragma unroll
          for (int t = 7; t >= 0; --t) {
            if (TAIL && l0 + q * OG + t >= L) continue;                    // uniform
            const float yr = fmaf(cr[t], w[t], gr[s]);       // (lanes without a state: whatever it is, nobody reads it)
            if constexpr (VAR == VAR_REAL) {
              gr[s] = yr * __builtin_amdgcn_exp2f(x0[t] * a2[s]);
            } else {
              const float yi = fmaf(-ci[t], w[t], gi[s]);
              gr[s] = fmaf(x0[t], yr, x1[t] * yi);
              gi[s] = fmaf(x0[t], yi, -x1[t] * yr);
            }
          }
        }
      };
#pragma unroll
      for (int q = OT / OG - 1; q >= 0; --q) {
        const int lq = l0 + q * OG;
        if (lq + OG <= L) group(q, std::false_type{});
        else if (lq < L) group(q, std::true_type{});
      }
      oct_wave_fence();
    }
    oct_barrier();
  }
  if (live) {
    if constexpr (VAR == VAR_REAL) pr = group_sum(pr);
    else group_product(pr, pi);
    if (dok) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int n = 8 * s + g;
        if (n < N) {
          const size_t o = (((size_t)vb * D + d) * N + n) * C;
          p.out[o] = gr[s];
          if (C == 2) p.out[o + 1] = gi[s];
        }
      }
      if (g == 0) {
        p.ptot[((size_t)vb * D + d) * 2] = pr;
        p.ptot[((size_t)vb * D + d) * 2 + 1] = pi;
      }
    }
  }
}

// Reverse scan.  Complex and real (S6) variant: with |a_l| < 1 the recurrence cannot be run backwards (dividing by
// a_l amplifies rounding errors without bound): the states of HT steps are recomputed from the checkpoint before them and
// kept in registers, then the steps are walked backwards with the adjoint state g_l = dLoss/dh_l
//     g_l = conj(C_l) dy_l + conj(a_{l+1}) g_{l+1},
//     dC_l[n] = sum_d dy_l conj(h_l)        dB_l[n] = sum_d w_l g_l        (w = delta u)
//     dw_l    = sum_n Re(conj(B_l) g_l)
//     complex: drho_l + i dtheta_l = sum_n conj(conj(a_l) g_l) h_{l-1} by parts, a_l taken out of the sum:
//              s_l = sum_n conj(g_l) h_{l-1};  drho_l = Re(a_l s_l),  dtheta_l = -Im(a_l s_l)
//     real:    x = g_l a_l h_{l-1};  dA[d,n] += x delta_l;  ddelta_l = sum_n x A[d,n] + dw_l u_l.
// Gate: with z given the forward output was y = y_pre silu(z); dy is scaled by silu(z) on the way in, y_pre = sum_n Re(C h) +
// D u is recomputed with the states, and dz = dy y_pre silu'(z) leaves with the other gradients (GATED).
// Checkpoints every 16 steps.
// Unitary variant: |a_l| = 1, the recurrence runs backwards from the checkpoint at the end, h_{l-1} = conj(a_l) (h_l - B_l w_l),
// and takes every checkpoint it passes (ck a multiple of 32) instead of what it has come to;
//     dtheta_l = -sum_n Im(conj(g_l) p_l),  p_l = h_l - B_l w_l.
// 30 vector instructions per state and step, no states kept; B5 D200 N24 L1001 85 -> 68 us.
// States nbase .. nbase + 8 S - 1 (RecBwdArgs).
// RAGGED: the sequence may end inside an interval, whose steps past the end the walk then leaves out.  Real and unitary, that walk is
// a second copy of the code with 5 to 20 registers more, so lengths that are a multiple of 16 have an instance without it: in one
// instance for all, S6 gated, 32 x 512 x 16, 720 steps 290.5 -> 292.7 us; apart 290.5, and 8 x 256 x 16, 1001 steps (unitary) 96.7 -> 98.3,
// 32 x 512 x 24, 721 steps (S6 gated, where it costs two spilled registers) 389.8 -> 400.1.
//
// Time is cut into intervals of OH steps (16, or 8 where the slabs of the unitary scan's 24 and 32 states need the room) with one barrier each; 32 steps are staged at a time, at the end of every other
// interval.  (Tiles 16 steps apart in the two wavefronts of a SIMD, so that one computes while the other stages: no faster, and
// a third more HBM reads where a tile no longer starts on a 128-byte line.)
template <int VAR, int S, bool FULLN, bool RAGGED, typename Tin, typename Tbc, bool GATED>
__global__ __launch_bounds__(512) void oct_bwd_kernel(const RecBwdArgs p) {
  constexpr int C = VAR == VAR_REAL ? 1 : 2;
  constexpr bool UNI = VAR == VAR_UNITARY;
  constexpr bool WALK_TAIL = RAGGED && VAR != VAR_COMPLEX;   // (complex: what passes by stays in its step)
  constexpr int OH = UNI && S > 2 ? 8 : 16;
  static_assert(!(UNI && GATED), "the unitary scan's gate has kernels of its own");
  // planes [channel][step] of a wavefront: what the steps read - real (delta, w, dy), complex (Re a, Im a, w, dy) -, the
  // sums over the states (the first in the place of w), and what the end of the tile wants back and registers have no room for
  constexpr int PX = 0, PW = C, PG = C + 1, PKA = PW, PXA = C + 2;
  constexpr int PZA = PXA + 1;                              // complex: sum behind drho, dtheta (imaginary part)
  constexpr int PU = PXA + 1, PRAW = PXA + 2, PACT = PXA + 3;   // real: u, delta before the softplus, silu'(u)
  constexpr int PYA = VAR == VAR_REAL ? PACT + 1 : PZA + 1, PGZ = PYA + 1;
  constexpr int NPL = VAR == VAR_REAL ? (GATED ? PGZ + 1 : PACT + 1) : UNI ? PXA + 1 : (GATED ? PYA + 1 : PZA + 1);
  constexpr int PL = 8 * OP;
  using Rows = OctRows<C, S, 2, OT, Tbc>;
  // a wavefront's sums over its channels of 16 steps: [dB, dC][state row][step], rows 4 floats apart from a power of two
  constexpr int G = (VAR == VAR_COMPLEX ? S > 1 : S > 2) ? 4 : OG;   // steps at a time on the way back
  constexpr int SR = OH * C + 4, SLAB = 2 * 8 * S * SR;
  __shared__ __align__(16) float s_bc[2][Rows::FLOATS];
  __shared__ __align__(16) float s_in[8][NPL][PL];
  __shared__ __align__(16) float s_slab[2][8][SLAB];

  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
  const int c = lane >> 3, g = lane & 7;
  const bool bit1 = g & 2, bit0 = g & 1;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);
  const int vb = wg / p.ncg, d0 = (wg % p.ncg) * CH;
  const int b = vb / p.ns, sg = vb - b * p.ns;
  const int lbeg = sg * p.L, ld = p.ld;
  const int D = p.D, NT_ = p.N;                             // NT_: states of the call
  const int N = NT_ - p.nbase < 8 * S ? NT_ - p.nbase : 8 * S;
  const int L = (ld - lbeg < p.L) ? ld - lbeg : p.L;
  const int d = d0 + 8 * wave + c;
  const bool dok = d < D, live = d0 + 8 * wave < D;
  const int dd = dok ? d : D - 1;

  const size_t uback = UNI ? (size_t)(b - b / p.urep) * D * ld : 0;   // (u, delta of [B / urep, D, L])
  const Tin* __restrict__ gu = static_cast<const Tin*>(p.u) - uback;
  const Tin* __restrict__ gdl = static_cast<const Tin*>(p.delta) - uback;
  const size_t goff = ((size_t)b * D + dd) * ld + lbeg;
  const size_t zoff = (VAR == VAR_REAL && p.zrows) ? (size_t)b * (p.zrows - D) * ld : 0;   // (z, dz: rows of a wider tensor)
  const size_t bc_row = ((size_t)b * ((VAR == VAR_REAL && p.bcrows) ? p.bcrows : NT_) + p.nbase) * ld + lbeg;
  const Tbc* __restrict__ gB = static_cast<const Tbc*>(p.Bm);
  const Tbc* __restrict__ gC = static_cast<const Tbc*>(p.Cm);

  float a2[S], an[S], dAacc[S], gr[S], gi[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int n = p.nbase + 8 * s + g;
    a2[s] = 0.f; an[s] = 0.f; dAacc[s] = 0.f; gr[s] = 0.f; gi[s] = 0.f;
    if (dok && n < NT_) {
      if (VAR == VAR_REAL) { an[s] = p.A[(size_t)d * NT_ + n]; a2[s] = an[s] * LOG2E; }
      if (p.dhL) {
        const size_t o = (((size_t)b * D + d) * NT_ + n) * C;
        gr[s] = p.dhL[o];
        if (C == 2) gi[s] = p.dhL[o + 1];
      }
    }
  }
  if (p.seg && live) {
    int nn[S];
#pragma unroll
    for (int s = 0; s < S; ++s) nn[s] = p.nbase + (8 * s + g < N ? 8 * s + g : N - 1);
    const size_t e = ((size_t)b * p.ns + p.ns - 1) * D + dd;
    seg_chain<VAR, true, S>(p.seg + e * NT_ * C, p.segq + e * 2, -(ptrdiff_t)D * NT_ * C, -(ptrdiff_t)D * 2, p.ns - 1 - sg, nn, a2, gr, gi);
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (!dok || 8 * s + g >= N) { gr[s] = 0.f; gi[s] = 0.f; }   // (lanes behind the last channel read that one's)
  }
  // Lanes of the last group without a state.  Complex and unitary: nothing comes in there (w and dy count as zero), so state and
  // adjoint stay zero wherever the other lanes' are not NaN.  Real: an infinite step makes a NaN of zero state and zero decay rate
  // where the other lanes have a zero or an infinity, so what they add to the sums over the states is dropped (`mine`).
  const bool has_last = FULLN || 8 * (S - 1) + g < N;
  auto seen = [&](float v, int s) { return C == 1 || s < S - 1 || has_last ? v : 0.f; };

  // ---- state before step l of the segment (a multiple of 16; unitary: of ck, or its end): the checkpoint there, or the initial
  // state
  struct Start { float r[S], i[S]; };
  auto load_start = [&](Start& st, int l) {
    const int lg = lbeg + l;
    const size_t base = fresh((((size_t)b * p.nck + (lg > 0 ? (lg - 1) / p.ck : 0)) * NT_ + p.nbase + g) * C * D + d);
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int n = p.nbase + 8 * s + g;
      st.r[s] = 0.f; st.i[s] = 0.f;
      if (dok && n < NT_) {
        if (lg > 0) {
          const size_t o = base + (size_t)(8 * s * C) * D;
          st.r[s] = p.hck[o];
          if (C == 2) st.i[s] = p.hck[o + D];
        } else if (p.h0) {
          const size_t o = (((size_t)b * D + d) * NT_ + n) * C;
          st.r[s] = p.h0[o];
          if (C == 2) st.i[s] = p.h0[o + 1];
        }
      }
    }
  };

  struct Raw { Quad<Tin> u, dl; Quad<float> dy, th, rho, z; } raw;
  raw.u.zero(); raw.dl.zero(); raw.dy.zero(); raw.th.zero(); raw.rho.zero(); raw.z.zero();
  auto load_tile = [&](int l0) {
    const int ll = l0 + 4 * g;
    int idx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) idx[i] = ll + i < L ? ll + i : L - 1;
    const bool vec = l0 + OT <= L || L % 4 == 0;             // uniform: a lane's four steps exist or none
    const size_t o = fresh(goff + (vec ? min(ll, L - 4) : 0));
    raw.u.load(gu, o, vec, idx);
    raw.dl.load(gdl, o, vec, idx);
    raw.dy.load(p.dy, o, vec, idx);
    if (GATED) raw.z.load(p.z + zoff, o, vec, idx);
    if (C == 2) raw.th.load(p.theta, o, vec, idx);
    if (VAR == VAR_COMPLEX) raw.rho.load(p.rho, o, vec, idx);
  };
  Rows rows;
  Start st, st_next;                                        // of this interval, of the next (its loads in flight)
  auto land = [&]() {
    raw.u.touch(); raw.dl.touch(); raw.dy.touch();
    if (GATED) raw.z.touch();
    if (C == 2) raw.th.touch();
    if (VAR == VAR_COMPLEX) raw.rho.touch();
  };
  auto land_start = [&]() {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      touch_vgpr(st_next.r[s]);
      if (C == 2) touch_vgpr(st_next.i[s]);
    }
    st = st_next;
  };
  const float dsk = (p.Dskip && dok) ? p.Dskip[dd] : 0.f;
  const float dbias = (VAR == VAR_REAL && p.delta_bias && dok) ? p.delta_bias[dd] : 0.f;
  float accD = 0.f, accB = 0.f;
  float* __restrict__ in = &s_in[wave][0][0];

  // what the eight wavefronts left of the OH steps from lh on: added up, one atomic per element
  auto flush = [&](int buf, int lh) {
    constexpr int TOT = 2 * 8 * S * OH * C;
#pragma unroll
    for (int k = 0; k < (TOT + 511) / 512; ++k) {
      const int e = tid + 512 * k;
      if (TOT % 512 != 0 && e >= TOT) continue;
      const int x = e % (OH * C), r = e / (OH * C);          // r: [dB, dC][state row]
      const int kind = r >= 8 * S, n = r - kind * 8 * S;
      const float* q = &s_slab[buf][0][r * SR + x];
      float v[8];
#pragma unroll
      for (int w = 0; w < 8; ++w) v[w] = q[w * SLAB];
      const float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
      if (n < N && lh + x / C < L) atomicAdd((kind ? p.dC : p.dB) + (bc_row + (size_t)n * ld + lh) * C + x, sum);
    }
  };

  const int last = (L - 1) / OH;                             // index of the last interval
  const int lastb = (L - 1) / OT;                            // ... of the block of rows it lies in
  int tile0 = lastb * OT;                                    // first step of the staged tile
  float eu[4], edl[4], egz[4];                               // of the staged tile (complex: kept in registers; egz: dy silu'(z))
  // (whole: all of the tile's steps and of the wavefront's channels exist)
  auto stage_as = [&](int l0, auto whole) {
    constexpr bool WHOLE = decltype(whole)::value;
    f4 o0, o1, ow, og, ou, oraw, oact, oz;
    bool ok[4];
    float th[4];
    f4 sn, cs;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ok[i] = WHOLE || (dok && l0 + 4 * g + i < L);
      th[i] = C == 2 && ok[i] ? raw.th.get(i) : 0.f;
    }
    if constexpr (C == 2) sincos4(th, sn, cs);
    float u4_[4], d4[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u4_[i] = ok[i] ? raw.u.get(i) : 0.f;
      d4[i] = ok[i] ? raw.dl.get(i) : 0.f;
      if (VAR == VAR_REAL) {
        d4[i] += dbias;
        oraw[i] = d4[i];
      }
    }
    if (VAR == VAR_REAL && p.u_act) {                        // uniform
#pragma unroll
      for (int i = 0; i < 4; ++i) oact[i] = dsiluf_(u4_[i]);
      silu4(u4_);
    }
    if (VAR == VAR_REAL && p.delta_softplus) softplus4(d4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float uu = u4_[i], dl = ok[i] ? d4[i] : 0.f;
      float gy = ok[i] ? raw.dy.get(i) : 0.f;
      egz[i] = 0.f;
      if (GATED) {
        const float zz = ok[i] ? raw.z.get(i) : 0.f;
        egz[i] = gy * dsiluf_(zz);
        gy *= siluf_(zz);
      }
      oz[i] = egz[i];
      if (VAR == VAR_REAL) {
        o0[i] = dl;
      } else {
        const float r = VAR == VAR_COMPLEX ? expf(ok[i] ? raw.rho.get(i) : 0.f) : 1.f;
        o0[i] = cs[i] * r; o1[i] = sn[i] * r;
      }
      ow[i] = dl * uu; og[i] = gy; ou[i] = uu;
      eu[i] = uu; edl[i] = dl;
    }
    float* q = in + c * OP + 4 * g;
    *reinterpret_cast<f4*>(q) = o0;
    if constexpr (C == 2) *reinterpret_cast<f4*>(q + PL) = o1;
    *reinterpret_cast<f4*>(q + PW * PL) = ow;
    *reinterpret_cast<f4*>(q + PG * PL) = og;
    if constexpr (VAR == VAR_REAL) {
      *reinterpret_cast<f4*>(q + PU * PL) = ou;
      if (p.delta_softplus) *reinterpret_cast<f4*>(q + PRAW * PL) = oraw;
      if (p.u_act) *reinterpret_cast<f4*>(q + PACT * PL) = oact;
      if (GATED) *reinterpret_cast<f4*>(q + PGZ * PL) = oz;
    }
  };
  const bool all_ch = d0 + 8 * wave + 8 <= D;
  auto stage = [&](int l0) {
    if (all_ch && l0 + OT <= L) stage_as(l0, std::true_type{});
    else stage_as(l0, std::false_type{});
  };

  // What the walk back reads of a group of steps (planes) and of a state group's rows there, a turn ahead of their use: with
  // two wavefronts per SIMD the LDS latency of every group would show.
  struct Steps { float x0[G], x1[G], w[G], gy[G]; };
  struct RowsAt { float br[G], bi[G], cr[G], ci[G]; };
  auto ld_planes = [&](Steps& o, int t, bool with_gy) {
    const float* x = in + c * OP + t;
    ld_steps(o.x0, x);
    if constexpr (C == 2) ld_steps(o.x1, x + PL);
    ld_steps(o.w, x + PW * PL);
    if (with_gy) ld_steps(o.gy, x + PG * PL);
  };
  auto ld_rows = [&](RowsAt& o, const float* __restrict__ bc, int q, int s, bool with_c) {
    ld_rec<C>(o.br, o.bi, bc + s * 8 * Rows::RS + q * G * C);
    if (with_c) ld_rec<C>(o.cr, o.ci, bc + (S + s) * 8 * Rows::RS + q * G * C);
  };
  constexpr int NQ = OH / G;                                 // groups of an interval
  Steps sp[2];
  RowsAt rw[2];

  // Steps lh .. lh + OH - 1 from the start state st; t0: their place in the staged tile, bc: in the rows.  TAIL: some of them lie
  // past the end; state and adjoint pass through those unchanged.
  // states; real: hsi holds the decay factors of the steps; unitary: the state behind the step being worked on
  float hsr[UNI ? 1 : OH][S], hsi[UNI ? 1 : OH][S];
  auto recompute = [&](int lh, int t0, const float* __restrict__ bc, auto tail_tag) {
    constexpr bool TAIL = decltype(tail_tag)::value;
    float xr[S], xi[S];
#pragma unroll
    for (int s = 0; s < S; ++s) { xr[s] = st.r[s]; xi[s] = st.i[s]; }
    ld_planes(sp[0], t0, false);
    ld_rows(rw[0], bc, 0, 0, false);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int turn = q * S + s;
        // the next turn's; behind the last one what the walk starts with
        if (s == S - 1 && q + 1 < NQ) ld_planes(sp[(q + 1) & 1], t0 + (q + 1) * G, false);
        if (turn + 1 < NQ * S) ld_rows(rw[(turn + 1) & 1], bc, (turn + 1) / S, (turn + 1) % S, false);
        sched_fence();
        const Steps& x = sp[q & 1];
        const RowsAt& r = rw[turn & 1];
#pragma unroll
        for (int t = 0; t < G; ++t) {
          const int tt = q * G + t;
          const bool skip = TAIL && lh + tt >= L;            // uniform
          const float wt = seen(x.w[t], s);
          if constexpr (VAR == VAR_REAL) {
            const float a = skip ? 1.f : __builtin_amdgcn_exp2f(x.x0[t] * a2[s]);
            xr[s] = fmaf(a, xr[s], r.br[t] * wt);
            hsr[tt][s] = xr[s];
            hsi[tt][s] = a;
          } else {
            const float nr = fmaf(x.x0[t], xr[s], fmaf(-x.x1[t], xi[s], r.br[t] * wt));
            const float ni = fmaf(x.x0[t], xi[s], fmaf(x.x1[t], xr[s], r.bi[t] * wt));
            xr[s] = nr; xi[s] = ni;
            hsr[tt][s] = nr; hsi[tt][s] = ni;
          }
        }
        sched_fence();
      }
    }
  };
  // walk back over those steps; the sums over the channels go to slab `buf`.  TAIL: steps past the end are left out (their
  // zeros times an infinite last state would be NaN)
  auto walk = [&](int lh, int t0, const float* __restrict__ bc, int buf, auto tail_tag) {
    constexpr bool TAIL = decltype(tail_tag)::value;
    float* __restrict__ slab = &s_slab[buf][wave][0];
    // the step of a group whose sums the lane holds (four at a time: two lanes hold, and write, the same)
    const int cs_ = G == 8 ? c : c >> 1, gs_ = G == 8 ? g : g >> 1;
    ld_planes(sp[(NQ - 1) & 1], t0 + (NQ - 1) * G, true);
    ld_rows(rw[0], bc, NQ - 1, 0, true);
#pragma unroll
    for (int qq = NQ - 1; qq >= 0; --qq) {
      float ka[G], xa[G], za[G], ya[G];
#pragma unroll
      for (int t = 0; t < G; ++t) { ka[t] = 0.f; xa[t] = 0.f; za[t] = 0.f; ya[t] = 0.f; }
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int turn = (NQ - 1 - qq) * S + s;
        if (s == 0 && qq > 0) ld_planes(sp[(qq - 1) & 1], t0 + (qq - 1) * G, true);
        if (turn + 1 < NQ * S) ld_rows(rw[(turn + 1) & 1], bc, NQ - 1 - (turn + 1) / S, (turn + 1) % S, true);
        sched_fence();
        const Steps& x = sp[qq & 1];
        const RowsAt& r = rw[turn & 1];
        float vb_r[G], vb_i[G], vc_r[G], vc_i[G];
#pragma unroll
        for (int t = G - 1; t >= 0; --t) {
          const int tt = qq * G + t;
          if (TAIL && lh + tt >= L) {                        // uniform
            vb_r[t] = vb_i[t] = vc_r[t] = vc_i[t] = 0.f;
            continue;
          }
          const float wt = seen(x.w[t], s), gy = seen(x.gy[t], s);
          const bool mine = s < S - 1 || has_last;
          const float hpr = !UNI && tt > 0 ? hsr[!UNI && tt > 0 ? tt - 1 : 0][s] : st.r[s];
          if constexpr (UNI) {
            float& hr = hsr[0][s];
            float& hi = hsi[0][s];
            gr[s] = fmaf(r.cr[t], gy, gr[s]);
            gi[s] = fmaf(-r.ci[t], gy, gi[s]);
            vb_r[t] = wt * gr[s];
            vb_i[t] = wt * gi[s];
            vc_r[t] = gy * hr;
            vc_i[t] = -gy * hi;
            ka[t] = fmaf(r.br[t], gr[s], ka[t]);
            ka[t] = fmaf(r.bi[t], gi[s], ka[t]);
            const float pr = fmaf(-r.br[t], wt, hr), pi = fmaf(-r.bi[t], wt, hi);
            xa[t] = fmaf(gr[s], pi, xa[t]);                  // Im(conj(g) p)
            xa[t] = fmaf(-gi[s], pr, xa[t]);
            const float tg = fmaf(x.x0[t], gr[s], x.x1[t] * gi[s]);
            gi[s] = fmaf(x.x0[t], gi[s], -x.x1[t] * gr[s]);
            gr[s] = tg;
            hr = fmaf(x.x0[t], pr, x.x1[t] * pi);
            hi = fmaf(x.x0[t], pi, -x.x1[t] * pr);
          } else if constexpr (VAR == VAR_REAL) {
            gr[s] = fmaf(r.cr[t], gy, gr[s]);
            vb_r[t] = wt * gr[s];
            if (GATED) ya[t] = mine ? fmaf(r.cr[t], hsr[tt][s], ya[t]) : ya[t];
            ka[t] = mine ? fmaf(r.br[t], gr[s], ka[t]) : ka[t];
            gr[s] *= hsi[tt][s];
            const float xx = gr[s] * hpr;
            dAacc[s] = fmaf(xx, x.x0[t], dAacc[s]);
            xa[t] = mine ? fmaf(xx, an[s], xa[t]) : xa[t];
          } else {
            const float hpi = tt > 0 ? hsi[tt > 0 ? tt - 1 : 0][s] : st.i[s];
            gr[s] = fmaf(r.cr[t], gy, gr[s]);
            gi[s] = fmaf(-r.ci[t], gy, gi[s]);
            vb_r[t] = wt * gr[s];
            vb_i[t] = wt * gi[s];
            if (GATED) ya[t] = fmaf(r.cr[t], hsr[tt][s], fmaf(-r.ci[t], hsi[tt][s], ya[t]));
            ka[t] = fmaf(r.br[t], gr[s], ka[t]);
            ka[t] = fmaf(r.bi[t], gi[s], ka[t]);
            xa[t] = fmaf(gr[s], hpr, xa[t]);               // conj(g) h_{l-1}
            xa[t] = fmaf(gi[s], hpi, xa[t]);
            za[t] = fmaf(gr[s], hpi, za[t]);
            za[t] = fmaf(-gi[s], hpr, za[t]);
            const float tg = fmaf(x.x0[t], gr[s], x.x1[t] * gi[s]);
            gi[s] = fmaf(x.x0[t], gi[s], -x.x1[t] * gr[s]);
            gr[s] = tg;
          }
        }
        float* o = slab + (8 * s + g) * SR + (qq * G + cs_) * C;
        auto put = [&](float* o_) {
          if constexpr (C == 1) {
            o_[0] = channel_sums(vb_r);
          } else {
            const float re = channel_sums(vb_r), im = channel_sums(vb_i);
            *reinterpret_cast<float2*>(o_) = make_float2(re, im);
          }
        };
        put(o);
        sched_fence();
#pragma unroll
        for (int t = 0; t < G; ++t) {
          const float gy = seen(x.gy[t], s);
          vb_r[t] = UNI ? vc_r[t] : gy * hsr[UNI ? 0 : qq * G + t][s];
          if (C == 2) vb_i[t] = UNI ? vc_i[t] : -gy * hsi[UNI ? 0 : qq * G + t][s];
        }
        put(o + 8 * S * SR);
        sched_fence();
      }
      // sums over the states, over what the group has read
      float* o = in + c * OP + t0 + qq * G + gs_;
      o[PKA * PL] = state_sums(ka, bit1, bit0);
      o[PXA * PL] = state_sums(xa, bit1, bit0);
      if constexpr (VAR == VAR_COMPLEX) o[PZA * PL] = state_sums(za, bit1, bit0);
      if constexpr (GATED) o[PYA * PL] = state_sums(ya, bit1, bit0);
    }
  };

  // gradients of the tile's steps; then the next tile is staged
  auto finish = [&](bool more) {
    const int l0 = tile0;
    oct_wave_fence();
    // (loads, stores and atomics share one in-order counter: the wait for the loads, two intervals old, comes in front of
    // the stores, the next loads behind them)
    land();
    const float* q = in + c * OP + 4 * g;
    auto plane = [&](int k) { return *reinterpret_cast<const f4*>(q + k * PL); };
    const f4 ka = plane(PKA), xa = plane(PXA), gy = plane(PG);
    f4 x1 = {0, 0, 0, 0}, za = x1, ya = x1, uu = {eu[0], eu[1], eu[2], eu[3]}, dl = {edl[0], edl[1], edl[2], edl[3]};
    f4 act = {1, 1, 1, 1}, pre = x1, gz = {egz[0], egz[1], egz[2], egz[3]};
    const f4 x0 = plane(0);
    if constexpr (VAR == VAR_COMPLEX) { x1 = plane(1); za = plane(PZA); }
    if constexpr (VAR == VAR_REAL) {
      dl = x0; uu = plane(PU);
      if (p.u_act) act = plane(PACT);
      if (p.delta_softplus) pre = plane(PRAW);
      if (GATED) gz = plane(PGZ);
    }
    if constexpr (GATED) ya = plane(PYA);
    f4 dsp = {1, 1, 1, 1};                                   // softplus'
    if (VAR == VAR_REAL && p.delta_softplus) {               // uniform
      asm volatile("");
#pragma unroll
      for (int i = 0; i < 4; ++i) dsp[i] = pre[i] > 20.0f ? 1.0f : sigmoidf_(pre[i]);
    }
    const bool acc = p.accum != 0;                         // uniform
    float duv[4], dd_[4], dth[4], drh[4], dzv[4];
    const int nvalid = dok ? L - (l0 + 4 * g) : 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      duv[i] = acc ? ka[i] * dl[i] : fmaf(ka[i], dl[i], dsk * gy[i]);
      if (VAR == VAR_REAL && p.u_act) duv[i] *= act[i];
      dd_[i] = ka[i] * uu[i];
      dth[i] = drh[i] = 0.f;
      if (VAR == VAR_REAL) {
        dd_[i] += xa[i];
        dd_[i] *= dsp[i];
        if (i < nvalid) accB += dd_[i];
      } else if (UNI) {
        dth[i] = -xa[i];
      } else {
        drh[i] = fmaf(x0[i], xa[i], -x1[i] * za[i]);       // Re(a s)
        dth[i] = -fmaf(x0[i], za[i], x1[i] * xa[i]);       // -Im(a s)
      }
      dzv[i] = GATED ? gz[i] * (acc ? ya[i] : fmaf(dsk, uu[i], ya[i])) : 0.f;
      if (i < nvalid) accD = fmaf(gy[i], uu[i], accD);
    }
    if (nvalid > 0) {
      const size_t o = fresh(goff + l0 + 4 * g);
      auto put = [&](float* dst, const float (&v)[4]) {
        if (acc) {
          float w[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) w[i] = i < nvalid ? dst[i] + v[i] : 0.f;
          store4(dst, 0, w, true, nvalid);
        } else {
          store4(dst, 0, v, true, nvalid);
        }
      };
      if (sizeof(Tin) == 2 && p.g16) {                     // uniform
        auto put16 = [&](float* base, const float (&v)[4]) {
          bf16_t* dst = reinterpret_cast<bf16_t*>(base) + o;
          if (nvalid >= 4) {
            *reinterpret_cast<u2h*>(dst) = u2h{(uint32_t)to_bf16(v[0]) | ((uint32_t)to_bf16(v[1]) << 16),
                                               (uint32_t)to_bf16(v[2]) | ((uint32_t)to_bf16(v[3]) << 16)};
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (i < nvalid) dst[i] = to_bf16(v[i]);
          }
        };
        put16(p.du, duv);
        put16(p.ddelta, dd_);
      } else {
        put(p.du + o, duv);
        put(p.ddelta + o, dd_);
      }
      if (C == 2) put(p.dtheta + o, dth);
      if (VAR == VAR_COMPLEX) put(p.drho + o, drh);
      if (GATED) put(p.dz + o + zoff, dzv);
    }
    if (more) {
      oct_wave_fence();
      tile0 -= OT;
      stage(tile0);
      if (tile0 > 0) load_tile(tile0 - OT);
    }
  };

  // ---- prologue: the rows of the last 32-step block, the wavefront's last tile, the last interval's start state
  rows.load(gB, gC, bc_row, ld, lastb * OT, L, N, tid);
  if (live) {
    load_tile(tile0);
    load_start(st_next, UNI ? L : last * OH);
  } else {
    for (int i = lane; i < SLAB; i += 64) { s_slab[0][wave][i] = 0.f; s_slab[1][wave][i] = 0.f; }
  }
  rows.put(s_bc[lastb & 1], lastb * OT, L, N, tid);
  if (lastb > 0) rows.load(gB, gC, bc_row, ld, (lastb - 1) * OT, L, N, tid);
  if (live) {
    stage(tile0);
    land_start();
    if constexpr (UNI) {
#pragma unroll
      for (int s = 0; s < S; ++s) { hsr[0][s] = st.r[s]; hsi[0][s] = st.i[s]; }
    }
    if (tile0 > 0) load_tile(tile0 - OT);
  }
  oct_barrier();

  for (int j = last; j >= 0; --j) {
    const int lh = j * OH;
    // ---- the rows of the next block, whose loads are two intervals old, into the other buffer; request the ones after
    const int rb = lh / OT;
    if ((lh % OT == OT - OH || j == last) && rb > 0) {
      rows.put(s_bc[(rb - 1) & 1], (rb - 1) * OT, L, N, tid);
      if (rb > 1) rows.load(gB, gC, bc_row, ld, (rb - 2) * OT, L, N, tid);
    }
    if (live) {
      if (!UNI && j > 0) load_start(st_next, lh - OH);
      const int t0 = lh - tile0;
      const float* __restrict__ bc = s_bc[rb & 1] + g * Rows::RS + (lh & (OT - 1)) * C;
      oct_wave_fence();
      if constexpr (!UNI) {
        if (lh + OH <= L) recompute(lh, t0, bc, std::false_type{});
        else recompute(lh, t0, bc, std::true_type{});
      }
      if (j < last) flush((j + 1) & 1, lh + OH);
      if (!WALK_TAIL || lh + OH <= L) walk(lh, t0, bc, j & 1, std::false_type{});
      else walk(lh, t0, bc, j & 1, std::integral_constant<bool, WALK_TAIL>{});
      if constexpr (UNI) {
        // a checkpoint: its state instead of the one run back to (plain loads, once per block)
        if (lh > 0 && lh % p.ck == 0) {
          load_start(st, lh);
#pragma unroll
          for (int s = 0; s < S; ++s) { hsr[0][s] = st.r[s]; hsi[0][s] = st.i[s]; }
        }
      } else {
        land_start();
      }
      rows.touch();
      if (t0 == 0) finish(j > 0);
    } else if (j < last) {
      flush((j + 1) & 1, lh + OH);
    }
    oct_barrier();
  }
  flush(0, 0);

  // ---- per-channel results
  if (live) {
    if (dok) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int n = p.nbase + 8 * s + g;
        if (n < NT_) {
          if (p.dh0 && sg == 0) {
            const size_t o = (((size_t)b * D + d) * NT_ + n) * C;
            p.dh0[o] = gr[s];
            if (C == 2) p.dh0[o + 1] = gi[s];
          }
          if (VAR == VAR_REAL && p.dA) atomicAdd(p.dA + (size_t)d * NT_ + n, dAacc[s]);
        }
      }
    }
    if (p.dD && !p.accum) {
      const float v = group_sum(accD);
      if (dok && g == 0) atomicAdd(p.dD + d, v);
    }
    if (VAR == VAR_REAL && p.dbias) {
      const float v = group_sum(accB);
      if (dok && g == 0) atomicAdd(p.dbias + d, p.dbias_scale * v);
    }
  }
}

}  // namespace aussm
