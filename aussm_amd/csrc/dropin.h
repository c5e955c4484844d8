// The reference's operator, extension_cpp::ssm_adaptive_unitary, as fused kernels.
//
// Semantics (extension-cpp/extension_cpp/csrc/cuda/ssm_adaptive_unitary_forward.cu:83-181), per batch
// b, channel i, state j, with ut = silu(u), Bt_j = B_r[j] e^{i B_theta[j]}, Ct_j likewise:
//     theta_l[b,i,j] = sum_r x[i,j,r] u_l[b,r] + x_bias[i,j]
//     h_l[b,i,j]     = exp(i theta_l) h_{l-1}[b,i,j] + Bt_j dt_l[b,i] ut_l[b,i]
//     y_l[b,i]       = silu(z_l[b,i]) ( sum_j Re(Ct_j h_l[b,i,j]) + D_i ut_l[b,i] )
//
// The phase tensor theta[b,i,j,l] (n times the size of every other tensor) never exists in memory.
// A wavefront owns one (batch, channel) pair - with more than 16 states per channel, one block of 16
// states of it - and walks the sequence in tiles of 16 timesteps:
//   * the tile's RUNNING phases G = prefix(theta), a (16 states) x (16 timesteps) block, are one small matrix
//     product x[i] (16 x d) . U (d x 16) on the 16-bit matrix cores with both operands split, fp32-accurate
//     (Phase below), where U is the tile of u[b] prefix-summed along
//     the tile (sum_{l' <= l} x.u_{l'} = x.U_l), plus (l + 1) x_bias.  The wavefront keeps its rows of x in
//     registers for the whole launch; the tiles of U, which all wavefronts of a batch element share, are
//     prepared once per call by a pre-pass (dropin_prep_kernel) and copied into LDS once per workgroup;
//   * the product lands with the timestep along the lanes of a 16-lane row (lane = (timestep l,
//     state group g), states 4 g .. 4 g + 3 in registers), so the rest of the recurrence is prefix sums
//     along the row (DPP row shifts, no LDS): E = e^{iG}, p = conj(E) Bt w, R = h_in + prefix(p), h = E R.
//     This is the cumulative-sum form the reference itself uses (:122-162), tile by tile, with the state h
//     handed from tile to tile - so G restarts at every tile and stays small;
//   * one sincos per (state, timestep), the sum over the states inside the wavefront, the gates
//     and the skip fused into the store.
#pragma once
#include "dropin_args.h"
#include "scan_fwd_xdl.h"
#include "split_half.h"

namespace aussm {

// How the operands of the phase product are split, by the steps of 32 that the contraction takes.  Up to two (d <= 64) three bf16
// pieces and six partial products (scan_fwd_xdl.h); from three on two f16 pieces and three partial products (split_half.h), the
// rows of x and the columns of U scaled by powers of two of their own: half the matrix instructions, which no vector instruction
// of the other wavefronts hides.  Two accumulators, the pieces' product and the mixed ones: 2^11 apart, and two chains of matrix
// instructions instead of one.  Relative error of sums of N(0, 1) products against 64 bits, six bf16 / three f16 products: 32 terms
// 3.8e-8 / 9.1e-8, 64 9.3e-8 / 9.8e-8, 128 1.53e-7 / 1.11e-7, 256 2.3e-7 / 1.3e-7, 512 3.4e-7 / 1.7e-7 - hence where the line lies.
// Records: [step][piece][64 lanes], behind them (f16) the exponent of each of the 16 rows or columns.
template <int KS>
struct Phase {
  static constexpr bool HALF = KS >= PHASE_HALF_KS;
  static constexpr int NP = HALF ? 2 : 3, REC = KS * NP * 64, TILE = REC + (HALF ? 4 : 0);   // 16-byte records of a tile of U
  f4 hi = {0, 0, 0, 0}, lo = {0, 0, 0, 0};
  __device__ __forceinline__ void step(const u4 (&x)[NP], const u4* __restrict__ s, int lane) {
    u4 v[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) v[q] = s[q * 64 + lane];
    if constexpr (HALF) {
      hi = xdl_half(x[0], v[0], hi);
      lo = xdl_half(x[1], v[0], lo);
      lo = xdl_half(x[0], v[1], lo);
    } else {
      hi = xmm<3>(x, v, hi);
    }
  }
  // exponents e of the row and of the column together
  __device__ __forceinline__ float value(int a, int e) const {
    return HALF ? __builtin_amdgcn_ldexpf(fmaf(lo[a], HALF_LO_INV, hi[a]), e) : hi[a];
  }
};
// the exponents of the columns of tile t
template <int KS>
__device__ __forceinline__ const int* phase_columns(const u4* __restrict__ upb, int t) {
  return reinterpret_cast<const int*>(upb + (size_t)t * Phase<KS>::TILE + Phase<KS>::REC);
}
// the rows of x of (channel, state block) vc, ks steps of them, into registers; what stands behind them
template <int KS>
__device__ __forceinline__ const int* phase_rows(const u4* __restrict__ xp, int ks, int vc, int lane, u4 (&xa)[KS][Phase<KS>::NP]) {
  constexpr int NP = Phase<KS>::NP;
  const u4* const r = xp + (size_t)vc * (ks * NP * 64 + (Phase<KS>::HALF ? 4 : 0));
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int q = 0; q < NP; ++q) xa[k][q] = k < ks ? r[(k * NP + q) * 64 + lane] : u4{0, 0, 0, 0};
  return reinterpret_cast<const int*>(r + ks * NP * 64);
}

// sin and cos of any argument, in revolutions for the hardware's units: the turns drop out in the first fused step, the second one adds
// what the constant 1 / 2 pi leaves (the result is as exact as the fp32 argument itself).  A branch here would cut the four state
// groups of a lane into separate blocks that the scheduler cannot interleave.  (x and x_bias in revolutions from the start would save
// two more instructions of four, but their rounding is the same at every step and adds up: y off by 1.2e-5 where it is 4.9e-6, 1 x 32 x
// 64, 2048 steps of u in {0, 1}.)
__device__ __forceinline__ void sincos_any(float x, float* sn, float* cs) {
  constexpr float C = 0.15915493667125702f, C_REST = 6.4206383e-9f;
  float t = fmaf(x, C, -rintf(x * C));
  t = fmaf(x, C_REST, t);
  *sn = __builtin_amdgcn_sinf(t);
  *cs = __builtin_amdgcn_cosf(t);
}

// silu and its derivative with the hardware reciprocal (1 ulp) instead of an IEEE division (ten instructions)
__device__ __forceinline__ float sigm_fast(float v) { return __builtin_amdgcn_rcpf(1.0f + __expf(-v)); }
__device__ __forceinline__ float silu_fast(float v) { return v * sigm_fast(v); }
__device__ __forceinline__ float dsilu_fast(float v) { const float sg = sigm_fast(v); return sg * (1.0f + v * (1.0f - sg)); }

// polar parameters of the operator: radius (softplus of it when given raw) and phase of state j
__device__ __forceinline__ float op_radius(const DropinArgs& p, const float* r, int j) {
  const float v = r[(size_t)j * p.bcs];
  return p.raw ? softplusf_(v) : v;
}
__device__ __forceinline__ float op_phase(const DropinArgs& p, const float* th, int j) { return th[(size_t)j * p.bcs]; }
// The polar parameters of every state, 0 past n.  For the maps of the segments (Re Bt, Im Bt, Re Ct, Im Ct).  With TURNED, for the sweeps,
// (B_r, 0, Re Ct', Im Ct') and the units (e^{i B_theta}, e^{i (B_theta + C_theta)}): a sweep works on states (and adjoints) turned by
// e^{-i B_theta}, whose inputs are real, with Ct' = Ct e^{i B_theta} - three operations of six for p, one of two for hat w, three of
// four for hat G (8 x 256 x 16, 720 steps: reverse sweep 131 -> 126 us, an instruction less per sine in it).
// Made by the first 128 threads of a workgroup, one polar number each: a sine with its branches in every lane for its own four states,
// at either end of a kernel, was half of the kernels' code and 3 to 4 us of every launch, mostly fetching it (5 x 48 pairs, 64 steps: 10.9 -> 9.0 us
// forward, 21.5 -> 15.8 backward).
template <bool TURNED>
__device__ __forceinline__ void polar_params(const DropinArgs& p, f4* s_par, f4* s_unit, int tid) {
  if (tid >= 2 * D_MAXN) return;
  const int j = tid >> 1, c = tid & 1, jc = j < p.n ? j : 0;      // (neighbouring lanes: Bt, Ct of a state)
  float sn, cs;
  fast_sincosf(op_phase(p, c ? p.C_th : p.B_th, jc), &sn, &cs);
  const float r = j < p.n ? op_radius(p, c ? p.C_r : p.B_r, jc) : 0.0f;
  if (TURNED) {
    const float bc = __shfl_xor(cs, 1), bs = __shfl_xor(sn, 1);
    const float2 unit = c ? make_float2(cs * bc - sn * bs, sn * bc + cs * bs) : make_float2(cs, sn);
    reinterpret_cast<float2*>(s_par)[2 * j + c] = c ? make_float2(r * unit.x, r * unit.y) : make_float2(r, 0.0f);
    reinterpret_cast<float2*>(s_unit)[2 * j + c] = unit;
  } else {
    reinterpret_cast<float2*>(s_par)[2 * j + c] = make_float2(r * cs, r * sn);
  }
}
// A state or an adjoint into a sweep's frame and out of it
__device__ __forceinline__ void turn_in(const f4& unit, float& re, float& im) {
  const float r = re * unit[0] + im * unit[1];
  im = im * unit[0] - re * unit[1];
  re = r;
}
__device__ __forceinline__ float2 turn_out(const f4& unit, float re, float im) {
  return make_float2(re * unit[0] - im * unit[1], re * unit[1] + im * unit[0]);
}
// Derivative of the softplus behind dt, from dt itself: 1 - e^-dt, below 1 by its Taylor series (the next term is below
// 2^-28 of the value).  Measured through the gradient of dt's argument, the rounding of the product included: root mean
// square of the relative error 4.0e-8 below 0.3, 4.5e-8 up to 1, 3.7e-8 from there on.  (The difference alone cancels:
// 2.7e-7 for dt between 0.05 and 0.1.)
__device__ __forceinline__ float dsoftplus_of(float dt) {
  float p = 2.5052108e-8f;                             // 1 / 11!
  p = fmaf(-dt, p, 2.7557319e-7f);
  p = fmaf(-dt, p, 2.7557319e-6f);
  p = fmaf(-dt, p, 2.4801587e-5f);
  p = fmaf(-dt, p, 1.9841270e-4f);
  p = fmaf(-dt, p, 1.3888889e-3f);
  p = fmaf(-dt, p, 8.3333333e-3f);
  p = fmaf(-dt, p, 4.1666667e-2f);
  p = fmaf(-dt, p, 1.6666667e-1f);
  p = fmaf(-dt, p, 0.5f);
  p = fmaf(-dt, p, 1.0f);
  return dt < 1.0f ? dt * p : 1.0f - __expf(-dt);
}

// ---- prefix / suffix sums along a row of 16 lanes
template <int CTRL>
__device__ __forceinline__ float dpp_mov0(float v) {   // lanes that have no source read 0
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float row_prefix(float v) {   // inclusive, towards higher lanes
  v += dpp_mov0<0x111>(v);    // row_shr:1
  v += dpp_mov0<0x112>(v);
  v += dpp_mov0<0x114>(v);
  v += dpp_mov0<0x118>(v);
  return v;
}
__device__ __forceinline__ float row_suffix(float v) {   // inclusive, towards lower lanes
  v += dpp_mov0<0x101>(v);    // row_shl:1
  v += dpp_mov0<0x102>(v);
  v += dpp_mov0<0x104>(v);
  v += dpp_mov0<0x108>(v);
  return v;
}
// Prefix sums of the first UP of N values and suffix sums of the others, a step of all before the next one of any: left to the compiler
// they came one after the other, with two idle cycles and a full latency between two steps of one sum.  (The values are kept apart
// from the sums they enter: a product fused into its first step takes three instructions instead of two.  Matrix instructions, LDS reads
// and scalar work may cross the fences.)
template <int UP, int N>
__device__ __forceinline__ void rows_side_by_side(float (&v)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) asm("" : "+v"(v[k]));
#define ROWS_STEP(C_)                                                                        \
  _Pragma("unroll") for (int k = 0; k < N; ++k) v[k] += k < UP ? dpp_mov0<0x110 + C_>(v[k]) : dpp_mov0<0x100 + C_>(v[k]); \
  __builtin_amdgcn_sched_barrier(0x10C);
  ROWS_STEP(1) ROWS_STEP(2) ROWS_STEP(4) ROWS_STEP(8)      // row_shr, row_shl
#undef ROWS_STEP
}
// value of the row's last / first lane in every lane of the row (DPP row broadcast: one vector instruction, where a
// lane shuffle is an LDS round trip on the chain that hands the state from tile to tile)
__device__ __forceinline__ float row_last(float v, int) { return dpp_perm<0x15F>(v); }    // row_newbcast:15
__device__ __forceinline__ float row_first(float v, int) { return dpp_perm<0x150>(v); }   // row_newbcast:0


// Operand records of 16 rows (or columns) of ks steps of 32, by a workgroup of 256 threads: load(k, lane, v) reads what the eight values of
// lane (row = lane % 16, g = lane / 16) of step k, terms 32 k + 8 g .. + 7, are made of, form(k, lane, v) makes them.  A row is scaled by one
// power of two, found from its largest value first: a thread keeps its records of up to 512 terms between the two passes, and requests
// them all before it works on the first - a launch lasts little longer than its loads (360 tiles of d = 256
// 10.2 -> 5.4 us, 687 workgroups for d = 180 8.5 -> 5.8).
template <typename Load, typename Form>
__device__ __forceinline__ void phase_records(Load&& load, Form&& form, int ks, bool half, u4* __restrict__ dst) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (!half) {
    const SplitK sk = make_splitk();
    for (int k = wave; k < ks; k += 4) {
      float v[8];
      load(k, lane, v);
      form(k, lane, v);
      u4 pc[3];
      split8<3>(sk, v, pc);
#pragma unroll
      for (int q = 0; q < 3; ++q) dst[(k * 3 + q) * 64 + lane] = pc[q];
    }
    return;
  }
  __shared__ float s_most[4][16];
  constexpr int R = D_MAXKS / 4;
  float v[R][8], most = 0.0f;
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (wave + 4 * r < ks) load(wave + 4 * r, lane, v[r]);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (wave + 4 * r >= ks) break;
    form(wave + 4 * r, lane, v[r]);
#pragma unroll
    for (int q = 0; q < 8; ++q) most = fmaxf(most, fabsf(v[r][q]));
  }
  most = rows_max(most);
  if (lane < 16) s_most[wave][lane] = most;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 4; ++w) most = fmaxf(most, s_most[w][lane & 15]);
  const int e = half_exponent(most);
  if (threadIdx.x < 16) reinterpret_cast<int*>(dst + ks * 2 * 64)[threadIdx.x] = -e;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int k = wave + 4 * r;
    if (k >= ks) break;
    u4 pc[2];
    split8_half<true>(v[r], exp2_of(e), pc);
    dst[(k * 2) * 64 + lane] = pc[0];
    dst[(k * 2 + 1) * 64 + lane] = pc[1];
  }
}

// x (rows of d: (channel i, state j) at row i xsi + j xsj), times scale -> operand records of (channel, state block) v = i nb + sb: row j - 16 sb.
// x_out [d, n, d], xb_out [d, n] (or null): scale x and x_bias in the operator's own order, for a caller that keeps them.
__device__ __forceinline__ void xprep_block(const DropinPrepArgs& a, unsigned vc) {
  const int d = a.d, n = a.n, nb = a.nb, xsi = a.xsi, xsj = a.xsj;
  const float scale = a.scale;
  const float* __restrict__ x = a.x;
  float* __restrict__ x_out = a.x_out;
  const int i = vc / nb, jb = 16 * (vc % nb);
  auto load = [&](int k, int lane, float (&v)[8]) {
    const int j = jb + (lane & 15), r0 = 32 * k + 8 * (lane >> 4);
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = x[((size_t)i * xsi + (size_t)min(j, n - 1) * xsj) * d + min(r0 + q, d - 1)];   // (no branch)
  };
  auto form = [&](int k, int lane, float (&v)[8]) {
    const int j = jb + (lane & 15), r0 = 32 * k + 8 * (lane >> 4);
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = (j < n && r0 + q < d) ? v[q] * scale : 0.0f;
    if (x_out && j < n) {
      float* const o = x_out + ((size_t)i * n + j) * d + r0;
      if (r0 + 8 <= d) {
        *reinterpret_cast<f4u*>(o) = f4u{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<f4u*>(o + 4) = f4u{v[4], v[5], v[6], v[7]};
      } else {
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (r0 + q < d) o[q] = v[q];
      }
    }
    if (a.xb_out && j < n && r0 == 0) a.xb_out[(size_t)i * n + j] = a.x_bias[(size_t)i * xsi + (size_t)j * xsj];
  };
  const bool half = a.KS >= PHASE_HALF_KS;
  phase_records(load, form, a.ks, half, a.xp + (size_t)vc * (a.ks * (half ? 2 : 3) * 64 + (half ? 4 : 0)));
}

// Tiles of u as the second operand of the phase product, one workgroup per (batch element, tile): column l holds U[r][l],
// U[r][l] = sum_{l' <= l} u[b, r, l0 + l'] - the prefix sum along the tile - so that
// the matrix product hands the scan kernels the running phase G = prefix(theta) directly
// (sum_{l' <= l} sum_r x[i,j,r] u[r,l'] = sum_r x[i,j,r] U[r,l]); timesteps past L count as zero.  All KS steps the
// kernels are compiled for are written, the ones past ceil(d / 32) as zeros.
__device__ __forceinline__ void uprep_block(const DropinPrepArgs& a, unsigned block) {
  const int d = a.d, L = a.L, t = a.t0 + block % a.nt;
  const float* __restrict__ ub = a.u + (size_t)(a.b0 + block / a.nt) * d * L;
  auto load = [&](int k, int lane, float (&v)[8]) {
    const int l = t * DT + (lane & 15), r0 = 32 * k + 8 * (lane >> 4);
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = ub[(size_t)min(r0 + q, d - 1) * L + min(l, L - 1)];
  };
  auto form = [&](int k, int lane, float (&v)[8]) {
    const int l = t * DT + (lane & 15), r0 = 32 * k + 8 * (lane >> 4);
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = r0 + q < d && l < L ? v[q] : 0.0f;
    rows_side_by_side<8>(v);
  };
  const bool half = a.KS >= PHASE_HALF_KS;
  phase_records(load, form, a.KS, half, a.up + (size_t)block * (a.KS * (half ? 2 : 3) * 64 + (half ? 4 : 0)));
}

// A tile's records, global memory -> registers -> LDS, in two steps so that the loads of the next tile fly
// while the current one is computed.
template <int NT, int NREC, int REC>
__device__ __forceinline__ void tile_load(const u4* __restrict__ src, u4 (&v)[NREC], int tid) {
#pragma unroll
  for (int e = 0; e < NREC; ++e) {
    const int rec = tid + e * NT;
    if (rec < REC) v[e] = src[rec];
  }
}
template <int NT, int NREC, int REC>
__device__ __forceinline__ void tile_store(const u4 (&v)[NREC], u4* __restrict__ dst, int tid) {
#pragma unroll
  for (int e = 0; e < NREC; ++e) {
    const int rec = tid + e * NT;
    if (rec < REC) dst[rec] = v[e];
  }
}

// ---- the sequence in segments
//
// A call of few (batch, channel) pairs leaves most of the chip idle while each pair walks its sequence alone (64 pairs of 2048
// steps: 163 us forward, 262 backward, on 8 compute units).  Its tiles are cut into nseg segments of sl, walked side by side.
// What a segment makes of the state that enters it is linear, h -> E h + F: dropin_seg_kernel finds E and F first, for the
// backward sweep also what it adds to the adjoint, and every wavefront of the scan composes the segments before (behind) its own.

// The states (and with ADJ their adjoints) of a lane's four rows after `cnt` segments, whose maps are `step` apart from `mp` (`ma`)
// + off[a] on in the order of the walk.  Lane l of a row takes map l, four shifts compose the row's sixteen in order into its
// last lane.  All lanes of a row return the same.
template <bool ADJ>
__device__ __forceinline__ void seg_enter_row(const f4* __restrict__ mp, const float2* __restrict__ ma, const int (&off)[4], ptrdiff_t step, int cnt,
                                              int l_, float (&hr)[4], float (&hi)[4], float* ar, float* ai) {
  for (int k0 = 0; k0 < cnt; k0 += 16) {
    const int k = k0 + l_;
    f4 m[4];
    float2 c[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      m[a] = k < cnt ? mp[k * step + off[a]] : f4{1, 0, 0, 0};
      c[a] = ADJ && k < cnt ? ma[k * step + off[a]] : make_float2(0.0f, 0.0f);
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      float Er = m[a][0], Ei = m[a][1], Fr = m[a][2], Fi = m[a][3], Ar = c[a].x, Ai = c[a].y;
      auto fold = [&](float er, float ei, float fr, float fi, float cr, float ci) {   // the earlier map comes first
        Fr += Er * fr - Ei * fi;
        Fi += Er * fi + Ei * fr;
        if (ADJ) {
          Ar += Er * cr - Ei * ci;
          Ai += Er * ci + Ei * cr;
        }
        const float t = Er * er - Ei * ei;
        Ei = Er * ei + Ei * er;
        Er = t;
      };
#define SEG_FOLD(C_) fold(dpp_mov0<C_>(Er), dpp_mov0<C_>(Ei), dpp_mov0<C_>(Fr), dpp_mov0<C_>(Fi), ADJ ? dpp_mov0<C_>(Ar) : 0.0f, ADJ ? dpp_mov0<C_>(Ai) : 0.0f)
      SEG_FOLD(0x111); SEG_FOLD(0x112); SEG_FOLD(0x114); SEG_FOLD(0x118);   // row_shr:1, 2, 4, 8: the last lane's sources are all in its row
#undef SEG_FOLD
      Er = row_last(Er, 0); Ei = row_last(Ei, 0);
      const float h = Er * hr[a] - Ei * hi[a] + row_last(Fr, 0);
      hi[a] = Er * hi[a] + Ei * hr[a] + row_last(Fi, 0);
      hr[a] = h;
      if (ADJ) {
        const float t = Er * ar[a] - Ei * ai[a] + row_last(Ar, 0);
        ai[a] = Er * ai[a] + Ei * ar[a] + row_last(Ai, 0);
        ar[a] = t;
      }
    }
  }
}

// The maps of the segments: all but the last one's for the forward kernel, all but the first one's for the backward one
// (blockIdx.x = segment, batch element, channel group).  With Q_l the rotation from the segment's start to step l - tile by
// tile, from the phases that the scans form, in their order -, S = sum w conj(Q) and T = sum a conj(Q):
//     E = Q_end,  F = E Bt S;        towards the front M = conj(E),  N = -Bt S,  A = conj(Ct) T.
// The sums stay with their lanes until the end, so a tile costs its phases, one sincos and eight operations a (state, step):
// of 256 pairs and 512 steps 7 us in segments of two tiles (forward) and 9 of four (backward), before scans of 9.7 and 28 us.
template <int KS, int NW, bool BWD>
__global__ __launch_bounds__(NW * 64) void dropin_seg_kernel(const DropinBwdArgs q) {
  typedef Phase<KS> P;
  __shared__ u4 s_u[2][P::REC];
  __shared__ f4 s_par[D_MAXN];
  const DropinArgs& p = q.f;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
  const int nb = p.nb, ncg = (p.d * nb + NW - 1) / NW;
  const int sq = blockIdx.x / (q.bg * ncg), cell = blockIdx.x - sq * q.bg * ncg, sg = sq + (BWD ? 1 : 0);
  const int zb = cell / ncg, b = q.b0 + zb, v = (cell % ncg) * NW + wave;
  const int i = v / nb, sb = v % nb, j0 = 16 * sb;
  const bool iok = i < p.d;
  const int ic = iok ? i : p.d - 1, vc = ic * nb + sb;
  const int l_ = lane & 15, g = lane >> 4;
  const int d = p.d, n = p.n, L = p.L;
  const size_t row = ((size_t)b * d + ic) * L, zrow = (size_t)b * p.zs + (size_t)ic * L;
  const u4* __restrict__ upb = p.up + ((size_t)(b - p.up_b0) * p.up_nt - p.up_t0) * P::TILE;   // + tile * TILE
  const int tb = q.t0 + sg * p.sl, te = min(tb + p.sl, q.t1);

  u4 xa[KS][P::NP];
  const int* const xe = phase_rows<KS>(p.xp, p.ks, vc, lane, xa);
  float xb[4], Qr[4], Qi[4], Sr[4], Si[4], Tr[4], Ti[4];
  int ex[4];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int j = j0 + 4 * g + a;
    xb[a] = j < n ? p.x_bias[(size_t)ic * p.xsi + (size_t)j * p.xsj] : 0.0f;
    ex[a] = P::HALF ? xe[4 * g + a] : 0;
    Qr[a] = 1.0f;
    Qi[a] = Sr[a] = Si[a] = Tr[a] = Ti[a] = 0.0f;
  }
  constexpr int NT = NW * 64, NREC = (P::REC + NT - 1) / NT;
  u4 sv[NREC];
  tile_load<NT, NREC, P::REC>(upb + (size_t)tb * P::TILE, sv, tid);
  tile_store<NT, NREC, P::REC>(sv, s_u[tb & 1], tid);
  polar_params<false>(p, s_par, nullptr, tid);
  __syncthreads();
  float un = 0.0f, dtn = 0.0f, zn = 0.0f, gyn = 0.0f;
  int en = 0;                                          // exponent of the tile's column
  auto inputs = [&](int l) {                           // a tile ahead; steps past the end count as zero
    if (P::HALF) en = phase_columns<KS>(upb, l / DT)[l_];
    const bool ok = l < L;
    un = ok ? p.u[row + l] : 0.0f;
    dtn = ok ? p.dt[row + l] : 0.0f;
    if (BWD) {
      zn = ok ? p.z[zrow + l] : 0.0f;
      gyn = ok ? q.gy[row + l] : 0.0f;
    }
  };
  inputs(tb * DT + l_);
  for (int t = tb; t < te; ++t) {
    const int l0 = t * DT;
    const float w = dtn * silu_fast(un), av = BWD ? gyn * silu_fast(zn) : 0.0f;
    const int eu = en;
    if (t + 1 < te) {
      inputs(l0 + DT + l_);
      tile_load<NT, NREC, P::REC>(upb + (size_t)(t + 1) * P::TILE, sv, tid);
    }
    P th;
    const u4* su = s_u[t & 1];
#pragma unroll
    for (int k = 0; k < KS; ++k) th.step(xa[k], su + k * P::NP * 64, lane);
    const float cnt = (float)(min(l_ + 1, L - l0));
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      float sn, cs;
      sincos_any(fmaf(xb[a], cnt, th.value(a, ex[a] + eu)), &sn, &cs);
      const float qr = Qr[a] * cs - Qi[a] * sn, qi = Qr[a] * sn + Qi[a] * cs;
      Sr[a] += w * qr;
      Si[a] -= w * qi;
      if (BWD) {
        Tr[a] += av * qr;
        Ti[a] -= av * qi;
      }
      Qr[a] = row_last(qr, lane);
      Qi[a] = row_last(qi, lane);
    }
    if (t + 1 < te) tile_store<NT, NREC, P::REC>(sv, s_u[(t + 1) & 1], tid);
    __syncthreads();
  }
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int j = j0 + 4 * g + a;
    const float sr = row_last(row_prefix(Sr[a]), lane), si = row_last(row_prefix(Si[a]), lane);
    float tr = 0.0f, ti = 0.0f;
    if (BWD) {
      tr = row_last(row_prefix(Tr[a]), lane);
      ti = row_last(row_prefix(Ti[a]), lane);
    }
    if (iok && l_ == 0 && j < n) {
      const size_t at = ((size_t)zb * d + i) * n + j, to = (size_t)sg * q.bg * d * n + at;
      const f4 par = s_par[j];
      const float Nr = par[0] * sr - par[1] * si, Ni = par[0] * si + par[1] * sr;    // Bt S
      if (BWD) {
        p.seg[to] = f4{Qr[a], -Qi[a], -Nr, -Ni};
        q.sega[to] = make_float2(par[2] * tr + par[3] * ti, par[2] * ti - par[3] * tr);
        if (sg == 1) {
          const size_t sidx = ((size_t)b * d + i) * n + j;
          q.ent[at] = f4{q.hc_re[sidx], q.hc_im[sidx], q.dh_re[sidx], q.dh_im[sidx]};
        }
      } else {
        p.seg[to] = f4{Qr[a], Qi[a], Qr[a] * Nr - Qi[a] * Ni, Qr[a] * Ni + Qi[a] * Nr};
      }
    }
  }
}

// Workgroup = (batch b, NW consecutive (channel, state block) pairs), one pair per wavefront; the nb
// wavefronts of a channel are neighbours (nb divides NW) and add their shares of y through LDS.
// KS: 32-wide steps of the contraction over r (d <= 32 KS).
// The kernel waits more than it works, so it takes the registers of four workgroups of four wavefronts to a compute unit at 128 < d:
// the tiles of U go straight to LDS (there and up to d = 128, in workgroups of eight), and at d > 192 the polar parameters are read
// from LDS where they are used.  Whole call of 32 x 256 x 16, 720 steps: 339 us with three bf16 pieces and three workgroups, then
// 234 (249 with three workgroups, 307 in workgroups of eight); 32 x 180 198 -> 167, 32 x 128 107 -> 99.
// One wavefront on a SIMD (d > 256) or two of wide x gain nothing from it: 8 x 300, 400 steps 109 -> 113, 8 x 250, 720 86 -> 90.
template <int KS, int NW>
__global__ __launch_bounds__(NW * 64, NW == 4 && KS <= 8 ? 4 : 1) void dropin_fwd_kernel(const DropinArgs p) {
  typedef Phase<KS> P;
  __shared__ u4 s_u[2][P::REC];
  __shared__ f4 s_par[D_MAXN], s_unit[D_MAXN];
  __shared__ float s_y[2][NW][DT];                     // shares of y of the tile, by tile parity (nb > 1)
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
  const int nb = p.nb, ncg = (p.d * nb + NW - 1) / NW;
  const int sg = blockIdx.x / (p.b * ncg), cell = blockIdx.x - sg * p.b * ncg;
  const int b = p.b0 + cell / ncg, v = (cell % ncg) * NW + wave;
  const int i = v / nb, sb = v % nb, j0 = 16 * sb;
  const bool iok = i < p.d;
  const int ic = iok ? i : p.d - 1, vc = ic * nb + sb;
  const int l_ = lane & 15, g = lane >> 4;
  const int d = p.d, n = p.n, L = p.L;
  const size_t row = ((size_t)b * d + ic) * L, zrow = (size_t)b * p.zs + (size_t)ic * L;
  const u4* __restrict__ upb = p.up + ((size_t)(b - p.up_b0) * p.up_nt - p.up_t0) * P::TILE;   // + tile * TILE
  const int tb = p.nseg > 1 ? p.t0 + sg * p.sl : p.t0, ntiles = p.nseg > 1 ? min(tb + p.sl, p.t1) : p.t1;

  // this wavefront's rows of x, split, for the whole launch
  u4 xa[KS][P::NP];
  const int* const xe = phase_rows<KS>(p.xp, p.ks, vc, lane, xa);
  // per state j = j0 + 4 g + a: bias and exponent of the phase (PAR_LDS: in LDS), carried state
  constexpr bool PAR_LDS = NW == 4 && KS == 8;
  __shared__ float2 s_row[PAR_LDS ? NW : 1][16];
  float2 xrow[4];
  float hr[4], hi[4];
  int at[4];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int j = j0 + 4 * g + a;
    const bool ok = j < n;
    const int jc = ok ? j : 0;
    const size_t cell_ = ((size_t)(b - p.b0) * d + ic) * n + jc;
    xrow[a] = make_float2(ok ? p.x_bias[(size_t)ic * p.xsi + (size_t)jc * p.xsj] : 0.0f, __int_as_float(P::HALF ? xe[4 * g + a] : 0));
    if (PAR_LDS && l_ == 0) s_row[wave][4 * g + a] = xrow[a];
    hr[a] = ok && p.h_re ? p.h_re[(size_t)p.b0 * d * n + cell_] : 0.0f;
    hi[a] = ok && p.h_im ? p.h_im[(size_t)p.b0 * d * n + cell_] : 0.0f;
    at[a] = (int)cell_;                                // (of use with segments, where there are few)
  }
  if (sg > 0) {                                        // through the segments in front
    seg_enter_row<false>(p.seg, nullptr, at, (ptrdiff_t)p.b * d * n, sg, l_, hr, hi, nullptr, nullptr);
#pragma unroll
    for (int a = 0; a < 4; ++a)
      if (j0 + 4 * g + a >= n) hr[a] = hi[a] = 0.0f;
  }
  const float Di = p.Dp[ic];

  constexpr bool DIRECT = KS <= 4 || (KS <= 8 && NW == 4);
  constexpr int NT = NW * 64, NREC = DIRECT ? 1 : (P::REC + NT - 1) / NT;
  u4 sv[NREC];
  auto fetch = [&](int t) {                            // a tile's records towards s_u[t & 1], directly 1 KiB at a time
    const u4* __restrict__ src = upb + (size_t)t * P::TILE;
    if constexpr (DIRECT) {
      for (int c = wave; c < KS * P::NP; c += NW) px_load_block(src + c * 64, s_u[t & 1] + c * 64, lane);
    } else {
      tile_load<NT, NREC, P::REC>(src, sv, tid);
    }
  };
  auto landed = [&](int t) {
    if constexpr (DIRECT) px_loads_done();
    else tile_store<NT, NREC, P::REC>(sv, s_u[t & 1], tid);
  };
  fetch(tb);
  polar_params<true>(p, s_par, s_unit, tid);
  landed(tb);
  __syncthreads();
  f4 par[4];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    if constexpr (!PAR_LDS) par[a] = s_par[j0 + 4 * g + a];
    turn_in(s_unit[j0 + 4 * g + a], hr[a], hi[a]);
  }
  // the wavefront's own inputs, requested one tile ahead
  const int lf = tb * DT + l_;
  float un = lf < L ? p.u[row + lf] : 0.0f, dtn = lf < L ? p.dt[row + lf] : 0.0f, zn = lf < L ? p.z[zrow + lf] : 0.0f;
  int en = P::HALF ? phase_columns<KS>(upb, tb)[l_] : 0;   // exponent of the tile's column
  for (int t = tb; t < ntiles; ++t) {
    const int l0 = t * DT, l = l0 + l_;
    const bool lok = l < L;
    const float uv = un, dtv = dtn, zv = zn;
    const int eu = en;
    {
      const bool nok = l + DT < L;
      un = nok ? p.u[row + l + DT] : 0.0f;
      dtn = nok ? p.dt[row + l + DT] : 0.0f;
      zn = nok ? p.z[zrow + l + DT] : 0.0f;
    }
    if (t + 1 < ntiles) {
      if (P::HALF) en = phase_columns<KS>(upb, t + 1)[l_];
      fetch(t + 1);
    }
    // ---- running phases of the tile, less the bias: lane (column l, rows j = 4 g + a)
    P th;
    const u4* su = s_u[t & 1];
#pragma unroll
    for (int k = 0; k < KS; ++k) th.step(xa[k], su + k * P::NP * 64, lane);
    const float ut = silu_fast(uv), w = dtv * ut;
    const float cnt = (float)(min(l_ + 1, L - l0));      // timesteps of the tile up to this one that exist
    float ysum = 0.0f;
    // GS states side by side (rows_side_by_side; all four would spill registers where the parameters stay in LDS).  32 x 256 x 16, 720
    // steps, in workgroups of four 243 -> 237 us; 8 x 180, 700 steps 70 -> 57
    constexpr int GS = PAR_LDS ? 2 : 4;
#pragma unroll
    for (int a0 = 0; a0 < 4; a0 += GS) {
      float sn[GS], cs[GS], pq[2 * GS];
      f4 pa[GS];
#pragma unroll
      for (int k = 0; k < GS; ++k) {
        const int a = a0 + k;
        const float2 xr = PAR_LDS ? s_row[wave][4 * g + a] : xrow[a];
        pa[k] = PAR_LDS ? s_par[j0 + 4 * g + a] : par[a];
        sincos_any(fmaf(xr.x, cnt, th.value(a, __float_as_int(xr.y) + eu)), &sn[k], &cs[k]);
        // p = conj(E) B_r w = pr - i qi
        const float rw = pa[k][0] * w;
        pq[2 * k] = cs[k] * rw;
        pq[2 * k + 1] = sn[k] * rw;
      }
      rows_side_by_side<2 * GS>(pq);
#pragma unroll
      for (int k = 0; k < GS; ++k) {
        const int a = a0 + k;
        const float Rr = hr[a] + pq[2 * k], Ri = hi[a] - pq[2 * k + 1];
        // h = E R
        const float her = cs[k] * Rr - sn[k] * Ri, hei = cs[k] * Ri + sn[k] * Rr;
        ysum = fmaf(pa[k][2], her, fmaf(-pa[k][3], hei, ysum));
        hr[a] = row_last(her, lane);
        hi[a] = row_last(hei, lane);
      }
      if (PAR_LDS) __builtin_amdgcn_sched_barrier(0);
    }
    ysum = rows_sum(ysum);
    if (t + 1 < ntiles) landed(t + 1);                 // (in front of this tile's store, which the counter would wait for, too)
    if (nb == 1) {
      if (p.y && iok && lok && g == 0) p.y[row + l] = silu_fast(zv) * (ysum + Di * ut);
    } else if (g == 0) {
      s_y[t & 1][wave][l_] = ysum;
    }
    __syncthreads();
    if (nb > 1 && sb == 0 && g == 0 && p.y && iok && lok) {      // the channel's first wavefront adds the shares up
      float tot = ysum;
      for (int k = 1; k < nb; ++k) tot += s_y[t & 1][wave + k][l_];
      p.y[row + l] = silu_fast(zv) * (tot + Di * ut);
    }
  }
  if (p.nh_re && iok && l_ == 0 && ntiles == p.t1) {
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int j = j0 + 4 * g + a;
      if (j < n) {
        const float2 h = turn_out(s_unit[j], hr[a], hi[a]);
        p.nh_re[((size_t)b * d + i) * n + j] = h.x;
        p.nh_im[((size_t)b * d + i) * n + j] = h.y;
      }
    }
  }
}

// ---- backward ---------------------------------------------------------------------------------
//
// Reverse sweep of the same tiles (the reference's ssm_adaptive_unitary_backward.cu:90-330 computes the
// same gradients from the same twelve inputs).  With hats for adjoints (hat h = dL/dRe h + i dL/dIm h),
// a_l = grad_y_l silu(z_l), and inside a tile G, E, p, R, h as in the forward kernel:
//     hat R_l = conj(E_l) a_l conj(Ct)                      (+ conj(E_last) hat h_out at the tile's last step)
//     hat p_s = sum_{l >= s} hat R_l,      hat h_in = hat p_first
//     hat w_s = Re(E_s conj(Bt) hat p_s)   summed over the states
//     hat G_l = -Im(conj(a_l conj(Ct)) h_l) + Im(conj(hat p_l) p_l)   (- Im(conj(hat h_out) h_last) at the last step)
//     hat theta_s = sum_{l >= s} hat G_l                    (suffix sum inside the tile only: the state handed
//                                                            to the next tile carries the rotation)
//     hat Bt += E_s w_s hat p_s,   hat Ct += a_l conj(h_l),   hat D += a_l ut_l
// The state at the end of each tile is recovered backwards (the recurrence is unitary, so this is
// stable): R_last = conj(E_last) h_out, h_in = R_last - sum p.  h at the end of the sequence comes from
// one forward sweep without outputs.
//
// hat theta is what the two products with x and u need:
//     grad_x[i,j,r] = sum_{b,l} hat theta[b,i,j,l] u[b,r,l],   grad_u[b,r,l] += sum_{i,j} x[i,j,r] hat theta[b,i,j,l].
// The second one sums over every channel of a batch element, so hat theta has to leave the wavefront
// that made it: it goes to a workspace that holds it for a CHUNK of the sequence only (tens of MB,
// cache resident), and the matrix-core GEMM (gemm.h) consumes it before the next chunk overwrites it.
// A launch therefore covers the tiles t0 .. t1 - 1 of every (batch, channel) pair; the state and its
// adjoint pass from launch to launch through two small buffers.

__device__ __forceinline__ float row_sum(float v) {     // total of the row in its first lane (others: partial)
  return row_suffix(v);
}

// The share of a tile's phase product that goes with state group a of 4: its steps k = a KS / 4 .. (KS < 4: all with a = 0).
// The sums run in the order of the forward kernel: the states are recovered from its end state with these phases, and
// phases that differ in their last bit would add up from tile to tile (gradients off by 1e-5 where the order differed).
template <int KS>
__device__ __forceinline__ void phase_part(int a, const u4 (&xa)[KS][Phase<KS>::NP], const u4* __restrict__ su, int lane, Phase<KS>& acc) {
  constexpr int STEP = (KS + 3) / 4;
#pragma unroll
  for (int k = a * STEP; k < (a + 1) * STEP && k < KS; ++k) acc.step(xa[k], su + k * Phase<KS>::NP * 64, lane);
}

// The phases of the tile that comes next are formed between the states of the current one: an operand tile is in LDS a tile
// ahead, and no wavefront waits for its chain of matrix instructions before it can start on the states (a launch over 8 x
// 256 pairs of 45 tiles, d = 256: 145 -> 136 us; 128 before two f16 pieces, 115 with them).  The forward kernel, whose states take
// less, runs 10 % slower that way.
#ifndef DROPIN_BWD_WAVES
#define DROPIN_BWD_WAVES 1
#endif
template <int KS, int NW>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(DROPIN_BWD_WAVES, DROPIN_BWD_WAVES))) void dropin_bwd_kernel(const DropinBwdArgs q) {
  typedef Phase<KS> P;
  __shared__ u4 s_u[2][P::REC];
  __shared__ float2 s_yw[2][NW][DT];                   // shares of (sum_j Re(Ct h), sum_j hat w) of the tile (nb > 1)
  const DropinArgs& p = q.f;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
  const int nb = p.nb, ncg = (p.d * nb + NW - 1) / NW;
  const int sg = blockIdx.x / (q.bg * ncg), cell = blockIdx.x - sg * q.bg * ncg;
  const int zb = cell / ncg, b = q.b0 + zb, v = (cell % ncg) * NW + wave;
  const int i = v / nb, sb = v % nb, j0 = 16 * sb;
  const bool iok = i < p.d;
  const int ic = iok ? i : p.d - 1, vc = ic * nb + sb;
  const int l_ = lane & 15, g = lane >> 4;
  const int d = p.d, n = p.n, L = p.L;
  const size_t row = ((size_t)b * d + ic) * L, zrow = (size_t)b * p.zs + (size_t)ic * L;
  const u4* __restrict__ upb = p.up + ((size_t)(b - p.up_b0) * p.up_nt - p.up_t0) * P::TILE;   // + tile * TILE

  u4 xa[KS][P::NP];
  const int* const xe = phase_rows<KS>(p.xp, p.ks, vc, lane, xa);
  // per state: (B_r, 0, Re Ct', Im Ct'), shared by the workgroup, and the bias of this wavefront's channel.
  // They are read from LDS where they are used: in registers they would push the kernel over 256.
  __shared__ f4 s_par[D_MAXN], s_unit[D_MAXN];
  __shared__ float s_xb[NW][16];
  __shared__ int s_ex[NW][16];                         // ... and the exponents of its rows of x
  polar_params<true>(p, s_par, s_unit, tid);
  if (lane < 16) s_xb[wave][lane] = j0 + lane < n ? p.x_bias[(size_t)ic * p.xsi + (size_t)(j0 + lane) * p.xsj] : 0.0f;
  if (P::HALF && lane < 16) s_ex[wave][lane] = xe[lane];
  float hr[4], hi[4], ar[4], ai[4];                    // state at the end of the tile being processed, its adjoint
  float gBr[4], gBi[4], gCr[4], gCi[4], gxb[4];
  int at[4];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int j = j0 + 4 * g + a;
    at[a] = (zb * d + ic) * n + (j < n ? j : 0);
    gBr[a] = gBi[a] = gCr[a] = gCi[a] = gxb[a] = 0.0f;
  }
  if (p.nseg > 1) {
    const ptrdiff_t per = (ptrdiff_t)q.bg * d * n;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const f4 en = q.ent[at[a]];
      hr[a] = en[0]; hi[a] = en[1]; ar[a] = en[2]; ai[a] = en[3];
    }
    seg_enter_row<true>(p.seg + (p.nseg - 1) * per, q.sega + (p.nseg - 1) * per, at, -per, p.nseg - 1 - sg, l_, hr, hi, ar, ai);
  } else {
    const size_t base = (size_t)q.b0 * d * n;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      hr[a] = q.hc_re[base + at[a]];
      hi[a] = q.hc_im[base + at[a]];
      ar[a] = q.dh_re[base + at[a]];
      ai[a] = q.dh_im[base + at[a]];
    }
  }
#pragma unroll
  for (int a = 0; a < 4; ++a)
    if (j0 + 4 * g + a >= n) hr[a] = hi[a] = ar[a] = ai[a] = 0.0f;
  const float Di = p.Dp[ic];
  float gD = 0.0f, gdtb = 0.0f;
  const int t_first = q.t0 + sg * p.sl, t_last = (p.nseg > 1 ? min(t_first + p.sl, q.t1) : q.t1) - 1;
  float* __restrict__ dth = q.dth + ((size_t)zb * d * n + (size_t)ic * p.xsi) * q.lc - (size_t)q.t0 * DT;   // + state j: j xsj rows

  constexpr int NT = NW * 64, NREC = (P::REC + NT - 1) / NT;
  u4 sv[NREC];
  tile_load<NT, NREC, P::REC>(upb + (size_t)t_last * P::TILE, sv, tid);
  tile_store<NT, NREC, P::REC>(sv, s_u[t_last & 1], tid);
  tile_load<NT, NREC, P::REC>(upb + (size_t)max(t_last - 1, t_first) * P::TILE, sv, tid);
  tile_store<NT, NREC, P::REC>(sv, s_u[(t_last + 1) & 1], tid);
  __syncthreads();
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const f4 unit = s_unit[j0 + 4 * g + a];
    turn_in(unit, hr[a], hi[a]);
    turn_in(unit, ar[a], ai[a]);
  }
  P th;
#pragma unroll
  for (int a = 0; a < 4; ++a) phase_part<KS>(a, xa, s_u[t_last & 1], lane, th);
  __syncthreads();                                     // (the first iteration overwrites that tile)
  // the wavefront's own inputs, requested one tile ahead
  float un, dtn, zn, gyn;
  int en = P::HALF ? phase_columns<KS>(upb, t_last)[l_] : 0;   // exponent of the tile's column
  {
    const int l = t_last * DT + l_;
    const bool ok = l < L;
    un = ok ? p.u[row + l] : 0.0f;
    dtn = ok ? p.dt[row + l] : 0.0f;
    zn = ok ? p.z[zrow + l] : 0.0f;
    gyn = ok ? q.gy[row + l] : 0.0f;
  }
  for (int t = t_last; t >= t_first; --t) {
    const int l0 = t * DT, l = l0 + l_;
    const bool lok = l < L;
    const float uv = un, dtv = dtn, zv = zn, gyv = gyn;
    const int eu = en;
    if (t > t_first) {                 // l - DT < L holds
      un = p.u[row + l - DT];
      dtn = p.dt[row + l - DT];
      zn = p.z[zrow + l - DT];
      gyn = q.gy[row + l - DT];
      if (P::HALF) en = phase_columns<KS>(upb, t - 1)[l_];
    }
    tile_load<NT, NREC, P::REC>(upb + (size_t)max(t - 2, t_first) * P::TILE, sv, tid);
    P nx;                                              // the next tile's phases, formed between the states of this one
    const u4* su = s_u[(t + 1) & 1];
    const int lend = min(15, L - 1 - l0);               // the tile's last step that exists
    const float ut = silu_fast(uv), w = dtv * ut, sz = silu_fast(zv), av = gyv * sz;
    const float cnt = (float)(min(l_ + 1, L - l0));      // timesteps of the tile up to this one that exist
    float ysum = 0.0f, wsum = 0.0f, thv[4];
    // GS states side by side, with their share of the next tile's phases.  us by one, two, four of them: 32 x 32 x 64 99, 97, 94; 8 x
    // 180 x 16, 700 steps 111, 103, 101; 8 x 256, 720 steps 128, 118, 119 (there the long phase products stay between the pairs).
    constexpr int GS = KS >= 8 ? 2 : 4;
#pragma unroll
    for (int a0 = 0; a0 < 4; a0 += GS) {
      f4 par[GS];
      float sn[GS], cs[GS], rw[GS], hdr[GS], hdi[GS], Gh[GS];
      float sums[4 * GS];                              // of p, then of conj(E_l) (a conj(Ct))
      float* const pq = sums;
      float* const rh = sums + 2 * GS;
#pragma unroll
      for (int k = 0; k < GS; ++k) {
        const int a = a0 + k;
        phase_part<KS>(a, xa, su, lane, nx);
        par[k] = s_par[j0 + 4 * g + a];
        sincos_any(fmaf(s_xb[wave][4 * g + a], cnt, th.value(a, P::HALF ? s_ex[wave][4 * g + a] + eu : 0)), &sn[k], &cs[k]);
        rw[k] = par[k][0] * w;                                                        // p = conj(E) B_r w = pr - i qi
        pq[2 * k] = cs[k] * rw[k];
        pq[2 * k + 1] = sn[k] * rw[k];
        hdr[k] = av * par[k][2];                                                      // a conj(Ct)
        hdi[k] = -av * par[k][3];
        rh[2 * k] = cs[k] * hdr[k] + sn[k] * hdi[k];
        rh[2 * k + 1] = cs[k] * hdi[k] - sn[k] * hdr[k];
      }
      rows_side_by_side<2 * GS>(sums);
      float phr[GS], phi[GS], hinr[GS], hini[GS];
#pragma unroll
      for (int k = 0; k < GS; ++k) {
        const int a = a0 + k;
        const float csl = row_last(cs[k], lane), snl = row_last(sn[k], lane);
        // forward quantities of the tile from the state at its end
        const float Rer = csl * hr[a] + snl * hi[a], Rei = csl * hi[a] - snl * hr[a];   // conj(E_last) h_out
        hinr[k] = Rer - row_last(pq[2 * k], lane);
        hini[k] = Rei + row_last(pq[2 * k + 1], lane);
        const float Rr = hinr[k] + pq[2 * k], Ri = hini[k] - pq[2 * k + 1];
        const float her = cs[k] * Rr - sn[k] * Ri, hei = cs[k] * Ri + sn[k] * Rr;       // h_l
        ysum = fmaf(par[k][2], her, fmaf(-par[k][3], hei, ysum));
        // adjoints
        const float Kr = csl * ar[a] + snl * ai[a], Ki = csl * ai[a] - snl * ar[a];     // conj(E_last) hat h_out
        phr[k] = rh[2 * k] + Kr;                                                        // hat p_s
        phi[k] = rh[2 * k + 1] + Ki;
        // X = E hat p:  hat w = B_r Re(X),  hat Bt += w X,  Im(conj(hat p) p) = -B_r w Im(X)
        const float Xr = fmaf(cs[k], phr[k], -(sn[k] * phi[k])), Xi = fmaf(cs[k], phi[k], sn[k] * phr[k]);
        wsum = fmaf(par[k][0], Xr, wsum);
        gBr[a] = fmaf(w, Xr, gBr[a]);
        gBi[a] = fmaf(w, Xi, gBi[a]);
        // hat G
        Gh[k] = fmaf(-rw[k], Xi, fmaf(hdi[k], her, -(hdr[k] * hei)));
        if (l_ == lend) Gh[k] -= ar[a] * hi[a] - ai[a] * hr[a];                         // h at the last step is h_out
        gCr[a] = fmaf(av, her, gCr[a]);                                                 // hat Ct += a conj(h)
        gCi[a] = fmaf(-av, hei, gCi[a]);
      }
      rows_side_by_side<0>(Gh);
#pragma unroll
      for (int k = 0; k < GS; ++k) {
        const int a = a0 + k;
        thv[a] = Gh[k];
        gxb[a] += Gh[k];                                                                // (zero past the end)
        // hand over to the previous tile
        hr[a] = hinr[k];
        hi[a] = hini[k];
        ar[a] = row_first(phr[k], lane);
        ai[a] = row_first(phi[k], lane);
      }
      if (KS >= 8) __builtin_amdgcn_sched_barrier(0);
    }
    // Loads and stores share one in-order counter: the wait for the tile, requested in front of the states, comes before this
    // tile's stores, or it would see them out, too (32 x 128, 720 steps: 221 -> 219 us).
    tile_store<NT, NREC, P::REC>(sv, s_u[t & 1], tid);
    // (stored here: a branch inside the loop cuts the four states into blocks that cannot hide each other's latencies)
#pragma unroll
    for (int a = 0; a < 4; ++a)
      if (lok && iok && j0 + 4 * g + a < n) dth[(size_t)(j0 + 4 * g + a) * p.xsj * q.lc + l] = thv[a];
    ysum = rows_sum(ysum);
    wsum = rows_sum(wsum);
    if (nb > 1 && g == 0) s_yw[t & 1][wave][l_] = make_float2(ysum, wsum);
    th = nx;
    if (nb > 1) {                                      // the channel's first wavefront adds the shares up
      __syncthreads();
      for (int k = 1; k < nb; ++k) {
        const float2 o = s_yw[t & 1][(wave + k) & (NW - 1)][l_];
        ysum += o.x;
        wsum += o.y;
      }
    }
    if (iok && lok && g == 0 && sb == 0) {
      const float pre = ysum + Di * ut;
      q.dz[zrow + l] = gyv * pre * dsilu_fast(zv);
      const float ddtv = q.dt_act ? wsum * ut * dsoftplus_of(dtv) : wsum * ut;
      q.ddt[row + l] = ddtv;
      gdtb += ddtv;
      q.du[row + l] = (wsum * dtv + av * Di) * dsilu_fast(uv);
      gD += av * ut;
    }
    if (nb == 1) __syncthreads();
  }
  // ---- reductions over the timesteps (lanes of a row) and hand-off.  The gradients of the 4 n shared
  // parameters are first summed over the workgroup's channels in LDS: every workgroup of the launch adds
  // to the same few addresses.
  // What only this part needs is fetched here: with all arguments at hand from the start the kernel spills scalar registers
  // (d = 256, four launches over 8 batch elements of 45 tiles: 511 us, 504 now).
  const __attribute__((address_space(4))) DropinBwdArgs* e = (const __attribute__((address_space(4))) DropinBwdArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(e));
  __shared__ float s_red[4][D_MAXN];
  if (tid < 4 * D_MAXN) (&s_red[0][0])[tid] = 0.0f;
  __syncthreads();
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    gxb[a] = row_sum(gxb[a]);
    gBr[a] = row_sum(gBr[a]);
    gBi[a] = row_sum(gBi[a]);
    gCr[a] = row_sum(gCr[a]);
    gCi[a] = row_sum(gCi[a]);
  }
  gD = row_sum(gD);
  gdtb = row_sum(gdtb);
  if (iok && l_ == 0) {
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int j = j0 + 4 * g + a;
      if (j < n) {
        const size_t sidx = ((size_t)b * d + i) * n + j;
        if (sg == 0) {
          const float2 dh = turn_out(s_unit[j], ar[a], ai[a]), h = turn_out(s_unit[j], hr[a], hi[a]);
          e->dh_re[sidx] = dh.x;
          e->dh_im[sidx] = dh.y;
          e->hc_re[sidx] = h.x;
          e->hc_im[sidx] = h.y;
        }
        atomicAdd(e->dxb + (size_t)i * e->f.xsi + (size_t)j * e->f.xsj, gxb[a]);
        const f4 par = s_par[j], un_ = s_unit[j];      // polar parameters, turned: B_r itself, Ct' = C_r e^{i (B_theta + C_theta)}
        atomicAdd(&s_red[0][j], gBr[a]);
        atomicAdd(&s_red[1][j], gBi[a] * par[0]);
        atomicAdd(&s_red[2][j], gCr[a] * un_[2] + gCi[a] * un_[3]);
        atomicAdd(&s_red[3][j], gCi[a] * par[2] - gCr[a] * par[3]);
      }
    }
    if (g == 0 && sb == 0) {
      atomicAdd(e->dD + i, gD);
      if (e->ddtb) atomicAdd(e->ddtb + i, e->ddtb_scale * gdtb);
    }
  }
  __syncthreads();
  if (tid < 4 * D_MAXN && (tid & (D_MAXN - 1)) < n) {
    constexpr int SH = 6;                              // log2(D_MAXN)
    float* dst = (tid >> SH) == 0 ? e->dB_r : (tid >> SH) == 1 ? e->dB_th : (tid >> SH) == 2 ? e->dC_r : e->dC_th;
    const int j = tid & (D_MAXN - 1);
    float v = (&s_red[0][0])[tid];
    // (raw radii: through the softplus)
    if (e->f.raw && !((tid >> SH) & 1)) v *= sigmoidf_(((tid >> SH) == 0 ? e->f.B_r : e->f.C_r)[(size_t)j * e->f.bcs]);
    atomicAdd(dst + (size_t)j * e->f.bcs, v);
  }
}

// A buffer set, FILL_BLOCK floats by one workgroup of 256, 16 bytes a lane where both sides allow it.
__device__ __forceinline__ void fill_block(const FillArgs& a, int i, size_t block) {
  float* __restrict__ dst = a.dst[i];
  const float* __restrict__ src = a.src[i];
  const size_t at = block * FILL_BLOCK, end = min((size_t)a.n[i], at + FILL_BLOCK);
  const bool vec = ((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src)) & 15) == 0;
  for (size_t j = at + 4 * threadIdx.x; j < end; j += 1024) {
    if (vec && j + 4 <= end) {
      *reinterpret_cast<f4*>(dst + j) = src ? *reinterpret_cast<const f4*>(src + j) : f4{0, 0, 0, 0};
    } else {
      for (size_t k = j; k < end && k < j + 4; ++k) dst[k] = src ? src[k] : 0.0f;
    }
  }
}
// Several buffers in one launch (blockIdx.y picks the buffer)
__global__ __launch_bounds__(256) void fill_kernel(const FillArgs a) { fill_block(a, blockIdx.y, blockIdx.x); }

// What a call prepares, in one launch: the records of x, the tiles of u, the buffers that start from zero or from a copy.  Each
// alone takes 4 us, nearly all of it the launch; a call of 64 pairs and 256 steps spent 20 of 85 us (both directions) on five of them.
__global__ __launch_bounds__(256) void dropin_prep_kernel(const DropinPrepArgs a, const FillArgs f) {
  unsigned blk = blockIdx.x;
  if (blk < a.xblocks) { xprep_block(a, blk); return; }
  blk -= a.xblocks;
  if (blk < a.ublocks) { uprep_block(a, blk); return; }
  blk -= a.ublocks;
  for (int i = 0; i < f.count; ++i) {
    const unsigned own = (unsigned)((f.n[i] + FILL_BLOCK - 1) / FILL_BLOCK);
    if (blk < own) { fill_block(f, i, blk); return; }
    blk -= own;
  }
}

}  // namespace aussm
