// Shared device helpers for the gfx950 selective-scan kernels.
//
// Two splits of the work: scan_oct.h and scan_bwd_unitary.h (vector ALU) give a workgroup CH = 64 channels of one batch element
// - a wavefront eight of them with all their states, or a lane a channel and a wavefront a few states -, the matrix-core
// kernels (scan_fwd_xdl.h, scan_bwd_xdl.h, scan_px.h) a wavefront 16 channels and chunks of 32 steps.  In all of them the
// inputs [B, D, L], L fastest, are read along L and turned in LDS, and B_t, C_t, shared by the channels, once a workgroup.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "scan_args.h"

namespace aussm {

constexpr int T = 32;         // timesteps per staged tile (AUSSM_TILE)
constexpr int TS = CH + 1;    // padded row stride of [t][channel] LDS tiles (bank-conflict free)
constexpr int NXCD = 8;       // accelerator complex dies, each with a private L2

constexpr float LOG2E = 1.4426950408889634f;

typedef uint16_t bf16_t;

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16_t v) { return __uint_as_float(((uint32_t)v) << 16); }

// round to nearest even (finite values; a NaN keeps its sign and stays one)
__device__ __forceinline__ bf16_t to_bf16(float v) {
  typedef __bf16 b1;
  return __builtin_bit_cast(bf16_t, (b1)v);
}

__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// Workgroups are dealt round-robin to the XCDs (workgroup i runs on XCD i % 8).  Remap so that
// logically consecutive workgroups, which share the B_t/C_t rows of one batch element and
// accumulate into the same dB/dC rows, land on the same XCD and hit in its L2.
__device__ __forceinline__ int xcd_remap(int i, int G) {
  const int q = G / NXCD, r = G % NXCD;
  const int x = i % NXCD, k = i / NXCD;
  return x * q + (x < r ? x : r) + k;
}

// (reciprocal: the hardware's and one Newton step, 4 instructions where an IEEE division takes 11 and the same error; the
// maximum takes the step away, 0 * inf, where 1 + e^-v is infinite)
__device__ __forceinline__ float sigmoidf_(float v) {
  const float x = 1.0f + __expf(-v), r = __builtin_amdgcn_rcpf(x);
  return fmaf(r, fmaxf(fmaf(-x, r, 1.0f), -1.0f), r);
}
__device__ __forceinline__ float siluf_(float v) { return v * sigmoidf_(v); }
// d/dv silu(v) = s + v s (1 - s)
__device__ __forceinline__ float dsiluf_(float v) { float s = sigmoidf_(v); return s * (1.0f + v * (1.0f - s)); }
// softplus with torch's threshold of 20 (F.softplus default), 33 vector instructions; log1pf(__expf(v)) takes 118, which was
// a fifth of the gated S6 forward kernel.  Root mean square of the relative error for N(0, 1) 3.6e-8 against 4.3e-8, for
// -20 .. 20 3.5e-8 against 2.3e-7.
//   t = e^v, with the rounding of v log2(e) made up for (the maximum: v = -inf);  w = fl(1 + t) = 2^k m, m in
//   [1 / sqrt 2, sqrt 2);  f = m - 1 plus what 1 + t was rounded by;  log(1 + f) = f - s (f - R), s = f / (2 + f),
//   R = s^2 (2/3 + 2/5 s^2 + ..): the series of 2 artanh(s) (Abramowitz and Stegun, 4.1.27; the reduction to one octave
//   around 1 is that of Cody and Waite, Software Manual for the Elementary Functions, chapter 5)
__device__ __forceinline__ float softplusf_(float v) {
  const float h = v * 1.44269504088896341f;
  const float lo = fmaxf(fmaf(v, 1.92596299112661746887e-8f, fmaf(v, 1.44269504088896341f, -h)), -1.0f);
  const float e = __builtin_amdgcn_exp2f(h);
  const float t = fmaf(e, lo * 0.693147180559945309f, e), w = 1.0f + t;
  const int u = __float_as_int(w) - 0x3f3504f3, k = u >> 23;
  const float f = __builtin_amdgcn_ldexpf(t - (w - 1.0f), -k) + (__int_as_float((u & 0x7fffff) + 0x3f3504f3) - 1.0f);
  const float s = f * __builtin_amdgcn_rcpf(2.0f + f), z = s * s;
  const float R = z * fmaf(fmaf(fmaf(0.22222222f, z, 0.28571429f), z, 0.4f), z, 0.66666667f);
  const float r = fmaf((float)k, 0.693147180559945309f, fmaf(-s, f - R, f));
  return v > 20.0f ? v : r;
}

// sin and cos of one argument, about 25 VALU instructions and no branch on the common path.
// Cody-Waite reduction by pi/2 in three fused steps, then the minimax polynomials on [-pi/4, pi/4] of sinf and cosf in
// S. L. Moshier's Cephes library (max error ~1 ulp of 1.0 for |x| < 1e4, which covers accumulated phases of practical length).
// Larger arguments take the library routine (fast_sincosf; sincos_1e4 leaves the check to its caller).
__device__ __forceinline__ void sincos_1e4(float x, float* sn, float* cs) {
  const float kf = rintf(x * 0.636619772367581343f);
  float r = fmaf(-kf, 1.57079637050628662109375f, x);
  r = fmaf(-kf, -4.37113900018624283e-8f, r);
  r = fmaf(-kf, -1.71512449782676e-15f, r);
  const float r2 = r * r;
  float ps = fmaf(-1.9515295891e-4f, r2, 8.3321608736e-3f);
  ps = fmaf(ps, r2, -1.6666654611e-1f);
  const float s = fmaf(r * r2, ps, r);
  float pc = fmaf(2.443315711809948e-5f, r2, -1.388731625493765e-3f);
  pc = fmaf(pc, r2, 4.166664568298827e-2f);
  const float c = fmaf(r2 * r2, pc, fmaf(-0.5f, r2, 1.0f));
  const int q = (int)kf;
  const float s1 = (q & 1) ? c : s;
  const float c1 = (q & 1) ? s : c;
  *sn = (q & 2) ? -s1 : s1;
  *cs = ((q + 1) & 2) ? -c1 : c1;
}
__device__ __forceinline__ void fast_sincosf(float x, float* sn, float* cs) {
  if (__builtin_expect(fabsf(x) > 1.0e4f, 0)) sincosf(x, sn, cs);
  else sincos_1e4(x, sn, cs);
}

// wave-uniform loads of B_t / C_t.  idx is uniform across the wavefront.  The tensors are inputs
// that no kernel of this library writes, so they are read through the constant address space:
// that lets the compiler select scalar (SMEM) loads whose results sit in SGPRs and feed the FMAs
// directly.  Complex records are (re, im) pairs.
#define AUSSM_CONST_AS __attribute__((address_space(4)))
template <typename V>
__device__ __forceinline__ const AUSSM_CONST_AS V* const_as(const void* p) {
  return reinterpret_cast<const AUSSM_CONST_AS V*>(reinterpret_cast<uintptr_t>(p));
}
__device__ __forceinline__ float2 ld_c(const float* __restrict__ p, size_t idx) {
  const AUSSM_CONST_AS float* q = const_as<float>(p) + 2 * idx;
  return make_float2(q[0], q[1]);
}
__device__ __forceinline__ float2 ld_c(const bf16_t* __restrict__ p, size_t idx) {
  const uint32_t raw = const_as<uint32_t>(p)[idx];
  return make_float2(__uint_as_float(raw << 16), __uint_as_float(raw & 0xffff0000u));
}
// ---- eight consecutive timesteps of one state row in one scalar load (one 64-byte line for
// complex fp32).  TG is the number of timesteps the scan consumes per row "turn".
constexpr int TG = 8;
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
struct __attribute__((aligned(8))) f32x16_a8 { f32x16 v; };
struct __attribute__((aligned(4))) u32x8_a4 { u32x8 v; };

// complex rows: idx counts (re, im) records; result = re0, im0, re1, im1, ...
__device__ __forceinline__ f32x16 ld_c8(const float* __restrict__ p, size_t idx) {
  return const_as<f32x16_a8>(p + 2 * idx)->v;
}
__device__ __forceinline__ f32x16 ld_c8(const bf16_t* __restrict__ p, size_t idx) {
  const u32x8 raw = const_as<u32x8_a4>(p + 2 * idx)->v;
  f32x16 r;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    r[2 * i] = __uint_as_float(raw[i] << 16);
    r[2 * i + 1] = __uint_as_float(raw[i] & 0xffff0000u);
  }
  return r;
}
// Orders the instruction stream at this point: nothing is scheduled across it.
__device__ __forceinline__ void sched_fence() { __builtin_amdgcn_sched_barrier(0); }
// A use of a wave-uniform value that emits no instruction: makes the compiler place its
// "scalar loads have landed" wait here rather than at the first arithmetic use.
__device__ __forceinline__ void touch_uniform(float v) { asm volatile("" ::"s"(v)); }
__device__ __forceinline__ void touch_uniform(uint32_t v) { asm volatile("" ::"s"(v)); }
// The same for a per-lane value.  Vector loads, stores and atomics share ONE in-order counter on
// this architecture, and the compiler waits for "everything" whenever control flow hides how many
// younger stores follow a load.  Touching prefetched values at a point where the count is known
// (or where nothing younger is in flight) keeps that wait from also draining recent stores.
__device__ __forceinline__ void touch_vgpr(float v) { asm volatile("" ::"v"(v)); }
__device__ __forceinline__ void touch_vgpr(bf16_t v) { asm volatile("" ::"v"((uint32_t)v)); }

// ---- sums and moves across the four 16-lane rows of a wavefront (lane = 16 g + c) on the vector ALU.  gfx950 swaps
// rows between two registers in one instruction (v_permlane16_swap: rows 1 and 3 of the first with rows 0 and 2 of
// the second; v_permlane32_swap: the upper half of the first with the lower half of the second), so none of these
// takes the LDS round trip of a lane shuffle (ds_bpermute), and the scans take two dependent steps instead of three.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void rows_swap16(float& a, float& b) {
  const u32x2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]); b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void rows_swap32(float& a, float& b) {
  const u32x2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]); b = __uint_as_float(r[1]);
}
// x = [x0 x1 x2 x3] by rows.  incl: row g gets x0 + .. + xg; tot: every row gets x0 + x1 + x2 + x3.
__device__ __forceinline__ void rows_prefix(float x, int g, float* incl, float* tot) {
  float a = x, b = x;
  rows_swap16(a, b);                              // a = [x0 x0 x2 x2], b = [x1 x1 x3 x3]
  const float pair = a + b;                       // [x0+x1, x0+x1, x2+x3, x2+x3]
  float c = pair, d = pair;
  rows_swap32(c, d);                              // c = x0+x1 in every row, d = x2+x3
  float y = (g & 1) ? pair : x;
  if (g >= 2) y += c;
  *incl = y; *tot = c + d;
}
// incl: row g gets xg + .. + x3
__device__ __forceinline__ void rows_suffix(float x, int g, float* incl, float* tot) {
  float a = x, b = x;
  rows_swap16(a, b);
  const float pair = a + b;
  float c = pair, d = pair;
  rows_swap32(c, d);
  float y = (g & 1) ? x : pair;
  if (g < 2) y += d;
  *incl = y; *tot = c + d;
}
__device__ __forceinline__ float rows_max(float x) {
  float a = x, b = x;
  rows_swap16(a, b);
  float c = fmaxf(a, b), d = c;
  rows_swap32(c, d);
  return fmaxf(c, d);
}
__device__ __forceinline__ float rows_sum(float x) {
  float a = x, b = x;
  rows_swap16(a, b);
  float c = a + b, d = c;
  rows_swap32(c, d);
  return c + d;
}
// the value of row 3 of the same column, in every row
__device__ __forceinline__ float rows_last(float x) {
  float c = x, d = x;
  rows_swap32(c, d);                              // d = [x2 x3 x2 x3]
  float a = d, b = d;
  rows_swap16(a, b);                              // b = [x3 x3 x3 x3]
  return b;
}
// DPP moves inside a row of 16 lanes (every lane has a source for the patterns used here)
template <int CTRL>
__device__ __forceinline__ float dpp_perm(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// Sums over the 64 lanes of 16 values per lane on the vector ALU alone (35 instructions, no LDS): lane (g, c) returns
// the total of value 4 (c % 4) + g.  Two rounds of row swaps fold the four rows - 16 values, 8, 4: row g of q[j]
// holds value 4 j + g summed over the rows -; two transposing steps inside the quads leave q[lane % 4]'s quad sums,
// and two rotations by 4 and 8 lanes add the four quads of the row.
__device__ __forceinline__ float lanes_sum16(const float (&v)[16], int lane) {
  float q[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float a0 = v[4 * j], b0 = v[4 * j + 1], a1 = v[4 * j + 2], b1 = v[4 * j + 3];
    rows_swap16(a0, b0);
    rows_swap16(a1, b1);
    float c = a0 + b0, d = a1 + b1;
    rows_swap32(c, d);
    q[j] = c + d;
  }
  const bool b0 = lane & 1, b1 = lane & 2;
  const float r01 = (b0 ? q[1] : q[0]) + dpp_perm<0xB1>(b0 ? q[0] : q[1]);   // quad_perm:[1,0,3,2]
  const float r23 = (b0 ? q[3] : q[2]) + dpp_perm<0xB1>(b0 ? q[2] : q[3]);
  float r = (b1 ? r23 : r01) + dpp_perm<0x4E>(b1 ? r01 : r23);               // quad_perm:[2,3,0,1]
  r += dpp_perm<0x124>(r);                                                    // row_ror:4
  r += dpp_perm<0x128>(r);                                                    // row_ror:8
  return r;
}

// 16-byte loads and stores that are only known to be 4-byte aligned, and 8-byte ones of four bf16 (rows start anywhere when the
// row length is not a multiple of four): the memory pipeline takes them, the type tells the compiler so
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t u2h __attribute__((ext_vector_type(2), aligned(2)));

// Four consecutive raw input elements, kept exactly as loaded (no arithmetic may touch a loaded
// register before the tile is collected, or the wait for the load moves up to the load).
template <typename Tin> struct Quad;
template <> struct Quad<float> {
  float4 v;
  __device__ __forceinline__ float get(int i) const { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }
  __device__ __forceinline__ void touch() const { touch_vgpr(v.x); touch_vgpr(v.y); touch_vgpr(v.z); touch_vgpr(v.w); }
  __device__ __forceinline__ void zero() { v = make_float4(0.f, 0.f, 0.f, 0.f); }
  // vec: one load of all four at element offset o (the caller guarantees the range; no alignment beyond the element's);
  // otherwise four element loads at o + idx[i].
  __device__ __forceinline__ void load(const float* __restrict__ p, size_t o, bool vec, const int (&idx)[4]) {
    if (vec) { const f4u r = *reinterpret_cast<const f4u*>(p + o); v = make_float4(r[0], r[1], r[2], r[3]); }
    else v = make_float4(p[o + idx[0]], p[o + idx[1]], p[o + idx[2]], p[o + idx[3]]);
  }
};
template <> struct Quad<bf16_t> {
  uint2 v;
  __device__ __forceinline__ float get(int i) const {
    const uint32_t w = (i < 2) ? v.x : v.y;
    return __uint_as_float((i & 1) ? (w & 0xffff0000u) : (w << 16));
  }
  __device__ __forceinline__ void touch() const { touch_vgpr(__uint_as_float(v.x)); touch_vgpr(__uint_as_float(v.y)); }
  __device__ __forceinline__ void zero() { v = make_uint2(0u, 0u); }
  __device__ __forceinline__ void load(const bf16_t* __restrict__ p, size_t o, bool vec, const int (&idx)[4]) {
    if (vec) { const u2h r = *reinterpret_cast<const u2h*>(p + o); v = make_uint2(r[0], r[1]); }
    else v = make_uint2((uint32_t)p[o + idx[0]] | ((uint32_t)p[o + idx[1]] << 16),
                        (uint32_t)p[o + idx[2]] | ((uint32_t)p[o + idx[3]] << 16));
  }
};

// Four consecutive float32 outputs at element offset o: one 16-byte store (on any element) when `vec`, else
// element stores for the timesteps < nvalid.
__device__ __forceinline__ void store4(float* __restrict__ p, size_t o, const float (&x)[4], bool vec, int nvalid) {
  if (vec && nvalid >= 4) {
    *reinterpret_cast<f4u*>(p + o) = f4u{x[0], x[1], x[2], x[3]};
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < nvalid) p[o + i] = x[i];
  }
}

// four consecutive results at byte offset ob (of a float tensor): float, or bf16 at half the offset (g16, uniform)
template <typename Tin>
__device__ __forceinline__ void store_grad4(float* p, size_t ob, const f4& v, int g16) {
  if (sizeof(Tin) == 2 && g16) {
    uint2 w;
    w.x = (uint32_t)to_bf16(v[0]) | ((uint32_t)to_bf16(v[1]) << 16);
    w.y = (uint32_t)to_bf16(v[2]) | ((uint32_t)to_bf16(v[3]) << 16);
    *reinterpret_cast<uint2*>(reinterpret_cast<char*>(p) + ob / 2) = w;
  } else {
    *reinterpret_cast<f4*>(reinterpret_cast<char*>(p) + ob) = v;
  }
}

// A call that is split along the sequence: what enters a segment, from what the segments before it (ADJ: behind it) make of a
// zero state.  Each of them acts on the state as h -> q h + Z with Z [entry][D][N][C] and q from [entry][D][2] (complex: the
// product of the a_l; real: the sum of the step sizes, q = exp(A sum)); the adjoint takes conj(q).  Every workgroup walks the
// entries ahead of its segment itself, K states per lane, four entries in flight: a chain kernel between the two passes took
// 5 - 9 us and a launch gap (B16 D128 N16 L1024 unitary forward: chain 6.5, scan 16.4 -> 17.4 us without).  z, q: first entry, at the lane's channel; zs, qs: floats from one entry to the next walked;
// n: the lane's states (valid indices); a2: real, A log2(e).
template <int VAR, bool ADJ, int K>
__device__ __forceinline__ void seg_chain(const float* __restrict__ z, const float* __restrict__ q, ptrdiff_t zs, ptrdiff_t qs, int cnt,
                                          const int (&n)[K], const float (&a2)[K], float (&hr)[K], float (&hi)[K]) {
  constexpr int U = 4;
#pragma unroll 1
  for (int j = 0; j < cnt; j += U) {
    float zr[U][K], zi[U][K], qr[U], qi[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const ptrdiff_t e = j + i < cnt ? j + i : cnt - 1;
      const f2u qq = *reinterpret_cast<const f2u*>(q + e * qs);      // (real: behind an odd number of floats, maybe)
      qr[i] = qq[0]; qi[i] = qq[1];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        if (VAR == VAR_REAL) {
          zr[i][k] = z[e * zs + n[k]]; zi[i][k] = 0.f;
        } else {
          const float2 v = *reinterpret_cast<const float2*>(z + e * zs + 2 * n[k]);
          zr[i][k] = v.x; zi[i][k] = v.y;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      if (j + i < cnt) {                                     // uniform
#pragma unroll
        for (int k = 0; k < K; ++k) {
          if (VAR == VAR_REAL) {
            hr[k] = fmaf(__builtin_amdgcn_exp2f(qr[i] * a2[k]), hr[k], zr[i][k]);
          } else {
            const float x = qr[i], y = ADJ ? -qi[i] : qi[i];
            const float nr = fmaf(x, hr[k], fmaf(-y, hi[k], zr[i][k]));
            hi[k] = fmaf(x, hi[k], fmaf(y, hr[k], zi[i][k]));
            hr[k] = nr;
          }
        }
      }
    }
  }
}

// sin and cos without the large-argument branch: the caller keeps |x| below ~150.
__device__ __forceinline__ void sincos_small(float x, float* sn, float* cs) {
  const float kf = rintf(x * 0.636619772367581343f);
  float r = fmaf(-kf, 1.57079637050628662109375f, x);
  r = fmaf(-kf, -4.37113900018624283e-8f, r);
  const float r2 = r * r;
  float ps = fmaf(-1.9515295891e-4f, r2, 8.3321608736e-3f);
  ps = fmaf(ps, r2, -1.6666654611e-1f);
  const float s = fmaf(r * r2, ps, r);
  float pc = fmaf(2.443315711809948e-5f, r2, -1.388731625493765e-3f);
  pc = fmaf(pc, r2, 4.166664568298827e-2f);
  const float c = fmaf(r2 * r2, pc, fmaf(-0.5f, r2, 1.0f));
  const int q = (int)kf;
  const float s1 = (q & 1) ? c : s;
  const float c1 = (q & 1) ? s : c;
  *sn = (q & 2) ? -s1 : s1;
  *cs = ((q + 1) & 2) ? -c1 : c1;
}

// The same through the hardware's sine and cosine (arguments in revolutions): the argument is first reduced
// to a remainder of at most half a turn in two steps, as above, so what the units see is accurate to a rounding.
__device__ __forceinline__ void sincos_small_hw(float x, float* sn, float* cs) {
  const float kf = rintf(x * 0.159154943091895336f);
  float r = fmaf(-kf, 6.283185482025146484375f, x);
  r = fmaf(-kf, -1.74845560007449e-7f, r);
  const float t = r * 0.159154943091895336f;
  *sn = __builtin_amdgcn_sinf(t);
  *cs = __builtin_amdgcn_cosf(t);
}

__device__ __forceinline__ void touch4(const f4& v) { touch_vgpr(v[0]); touch_vgpr(v[1]); touch_vgpr(v[2]); touch_vgpr(v[3]); }

// ---- global memory -> LDS without passing through registers: a wavefront moves 64 records (1 KiB)
// per instruction, lane i's record to lds + i.  The data is in LDS once the wavefront's vector-memory
// counter says so (px_loads_done / px_wait) and a barrier has published it.  The instruction is
// written out: left to the compiler, every later LDS read of the wavefront waits for ALL of its
// outstanding loads of this kind, which would serialise the prefetch.
__device__ __forceinline__ void px_load_block(const u4* __restrict__ src, u4* lds, int lane) {
  const uint32_t dst = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds);
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src + lane), "s"(dst) : "memory");
}
__device__ __forceinline__ void px_loads_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

}  // namespace aussm
