// Unitary forward scan in chunked matrix form on the bf16 matrix cores, fp32-accurate (N <= 16).
//
// Inside a chunk of XT = 32 timesteps starting from the state H (h at the end of the previous
// chunk), with Theta_t the running sum of theta over the chunk, P_t = exp(i Theta_t),
// w_s = delta_s u_s and V_s = conj(P_s) w_s (per channel):
//     h_t[n]  = P_t ( H[n] + sum_{s<=t} B_s[n] V_s )
//     y_t     = Re( P_t S_t ) + D u_t,     S_t = sum_{s<=t} G[t,s] V_s + sum_n C_t[n] H[n],
//     G[t,s]  = sum_n C_t[n] B_s[n]        (channel independent, masked to s <= t)
//     H'[n]   = P_last ( H[n] + sum_s B_s[n] V_s ).
// Every sum is a small complex GEMM whose free dimension is the channel, so the per-(channel,
// timestep) vector work is one sincos and a handful of products, independent of N.
//
// Arithmetic.  The fp32 matrix instructions share the vector ALU, the bf16 ones (XDL) run beside
// it, so the GEMMs use v_mfma_f32_16x16x32_bf16 on operands split EXACTLY into NP bf16 pieces
// (x = p1 + p2 + p3, each piece the bf16 rounding of what the previous ones left: three pieces
// carry 27 significand bits, more than fp32 holds).  A product keeps the partial products
// p_i q_j with i + j <= NP + 1, accumulated in fp32: with NP = 3 what is dropped is below 2^-26
// relative, i.e. the GEMMs are fp32-accurate; NP = 2 (2^-17) is there for measurements.
//
// Work split: a workgroup owns (batch b, 64 channels) and runs the chunks in order; each of its
// four wavefronts owns 16 channels end to end.  Lane l = (dl = l % 16, g = l / 16) is channel dl
// and owns the eight timesteps e = 0..7 -> t(g, e) = 16*(e/4) + 4*g + e%4 of every chunk.  That is
// the K order of the matrix instruction's B operand (lane group g holds K slots 8g..8g+7) under
// the permutation slot (g, e) <-> timestep t(g, e), and also the C/D layout of the result tiles
// (tile e/4, rows 4*g + e%4), so u/delta/theta go from global memory to matrix operands and the
// results go back to global memory as 16-byte vectors without passing through LDS.
// The channel-independent A operands (B_t, C_t and G in the orders each product needs, already
// split into pieces) are staged once per workgroup in LDS as 16-byte records [row][g].
#pragma once
#include "scan_common.h"
#include <type_traits>

namespace aussm {

typedef float f2v __attribute__((ext_vector_type(2)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));


// State (ADJ: adjoint) that enters segment sg of batch element bb of a split call: lane (dl, g) holds n = 4 g + i of channel d.
// part of parts: the entries in as many runs; part 0 applies the first to (hr, hi), any other starts from zero and
// composes its run, whose product goes to (pr, pi).
template <bool ADJ, typename Args>
__device__ __forceinline__ void seg_enter(const Args& p, int bb, int sg, int d, int g, f4& hr, f4& hi, int part = 0, int parts = 1,
                                          float* pr = nullptr, float* pi = nullptr) {
  const int own = (sg + (ADJ ? 1 : 0)) * p.hs;
  const int all = ADJ ? (p.nf > own ? p.nf - own : 0) : own, per = (all + parts - 1) / parts, from = part * per;
  const int cnt = all - from < per ? all - from : per;
  const size_t e = ((size_t)bb * p.nf + (ADJ ? p.nf - 1 : 0)) * p.D + d;
  const ptrdiff_t st = ADJ ? -(ptrdiff_t)p.D : (ptrdiff_t)p.D;
  const float* z = p.seg + e * p.N * 2 + from * st * p.N * 2;
  const float* q = p.segq + e * 2 + from * st * 2;
  const ptrdiff_t zs = st * p.N * 2, qs = st * 2;
  float xr = 1.0f, xi = 0.0f;
  constexpr int U = 4;
#pragma unroll 1
  for (int j = 0; j < cnt; j += U) {
    f4 za[U], zb[U];
    float2 qq[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const ptrdiff_t o = j + i < cnt ? j + i : cnt - 1;
      qq[i] = *reinterpret_cast<const float2*>(q + o * qs);
      if (p.N == XN) {                                       // (uniform; the entries lie on 16 bytes)
        const f4* zz = reinterpret_cast<const f4*>(z + o * zs + 8 * g);
        za[i] = zz[0]; zb[i] = zz[1];
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int n = 4 * g + k < p.N ? 4 * g + k : p.N - 1;
          const float2 v = *reinterpret_cast<const float2*>(z + o * zs + 2 * n);
          (k < 2 ? za : zb)[i][2 * (k & 1)] = v.x;
          (k < 2 ? za : zb)[i][2 * (k & 1) + 1] = v.y;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      if (j + i < cnt) {                                     // uniform
        const float x = qq[i].x, y = ADJ ? -qq[i].y : qq[i].y, t = fmaf(x, xr, -y * xi);
        xi = fmaf(x, xi, y * xr);
        xr = t;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const f4& v = k < 2 ? za[i] : zb[i];
          const float nr = fmaf(x, hr[k], fmaf(-y, hi[k], v[2 * (k & 1)]));
          hi[k] = fmaf(x, hi[k], fmaf(y, hr[k], v[2 * (k & 1) + 1]));
          hr[k] = nr;
        }
      }
    }
  }
  if (pr) { *pr = xr; *pi = xi; }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (4 * g + i >= p.N) { hr[i] = 0.f; hi[i] = 0.f; }
}

__device__ __forceinline__ f4 xdl(const u4& a, const u4& b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8v, a), __builtin_bit_cast(bf8v, b), c, 0, 0, 0);
}
// two fp32 -> packed bf16 pair (round to nearest even), low half = a
__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
  const f2v v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf2v));
}
// Split the pair (a, b) into NP packed bf16 pieces.  The residuals are exact in fp32: they are
// taken with the bf16 dot instruction, r = x + (-1) * piece (one instruction per value instead of
// an unpack and a subtract).
// The multipliers (-1, 0) and (0, -1) are kept in registers the compiler cannot see through: as
// literal operands of this instruction they do not encode the intended packed pair.
struct SplitK { uint32_t lo, hi; };
__device__ __forceinline__ SplitK make_splitk() {
  SplitK k{0x0000bf80u, 0xbf800000u};
  asm volatile("" : "+v"(k.lo), "+v"(k.hi));
  return k;
}
template <int NP>
__device__ __forceinline__ void split2(const SplitK& sk, float a, float b, uint32_t (&out)[NP]) {
  const bf2v m_lo = __builtin_bit_cast(bf2v, sk.lo), m_hi = __builtin_bit_cast(bf2v, sk.hi);
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const f2v v = {a, b};
    const bf2v pk = __builtin_convertvector(v, bf2v);
    out[p] = __builtin_bit_cast(uint32_t, pk);
    if (p + 1 < NP) {
      a = __builtin_amdgcn_fdot2_f32_bf16(pk, m_lo, a, false);
      b = __builtin_amdgcn_fdot2_f32_bf16(pk, m_hi, b, false);
    }
  }
}
// eight values -> NP operand registers quads (K slots 0..7 of one lane group)
template <int NP>
__device__ __forceinline__ void split8(const SplitK& sk, const float (&x)[8], u4 (&out)[NP]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t pc[NP];
    split2<NP>(sk, x[2 * q], x[2 * q + 1], pc);
#pragma unroll
    for (int p = 0; p < NP; ++p) out[p][q] = pc[p];
  }
}
// c += a . b over the kept partial products (small terms first)
template <int NP>
__device__ __forceinline__ f4 xmm(const u4 (&a)[NP], const u4 (&b)[NP], f4 c) {
#pragma unroll
  for (int s = NP - 1; s >= 0; --s)
#pragma unroll
    for (int i = 0; i <= s; ++i) c = xdl(a[i], b[s - i], c);
  return c;
}
// The same when only the first NPA pieces of a (and, for xmm_pp, of b too) can be non-zero: operands
// that came from bf16 inputs are a single exact piece, the products with their other pieces vanish.
template <int NP, int NPA>
__device__ __forceinline__ f4 xmm_p(const u4 (&a)[NP], const u4 (&b)[NP], f4 c) {
#pragma unroll
  for (int s = NP - 1; s >= 0; --s)
#pragma unroll
    for (int i = 0; i <= s; ++i)
      if (i < NPA) c = xdl(a[i], b[s - i], c);
  return c;
}
template <int NP, int NPA>
__device__ __forceinline__ f4 xmm_pp(const u4 (&a)[NP], const u4 (&b)[NP], f4 c) {
#pragma unroll
  for (int s = NP - 1; s >= 0; --s)
#pragma unroll
    for (int i = 0; i <= s; ++i)
      if (i < NPA && s - i < NPA) c = xdl(a[i], b[s - i], c);
  return c;
}
// ... and when it is the second operand whose pieces >= NPB vanish
template <int NP, int NPB>
__device__ __forceinline__ f4 xmm_q(const u4 (&a)[NP], const u4 (&b)[NP], f4 c) {
#pragma unroll
  for (int s = NP - 1; s >= 0; --s)
#pragma unroll
    for (int i = 0; i <= s; ++i)
      if (s - i < NPB) c = xdl(a[i], b[s - i], c);
  return c;
}
// the K-th matrix instruction of xmm (same order); skipped when it involves a piece >= NPA of a
template <int NP, int K, int NPA = NP>
__device__ __forceinline__ f4 xmm_k(const u4 (&a)[NP], const u4 (&b)[NP], f4 c) {
  constexpr int s0 = NP - 1;
  // products are visited with s = NP-1 .. 0 and i = 0 .. s: find (s, i) of index K
  constexpr int s = (NP == 3) ? (K < 3 ? 2 : (K < 5 ? 1 : 0)) : (NP == 2 ? (K < 2 ? 1 : 0) : 0);
  constexpr int base = (NP == 3) ? (K < 3 ? 0 : (K < 5 ? 3 : 5)) : (NP == 2 ? (K < 2 ? 0 : 2) : 0);
  constexpr int i = K - base;
  static_assert(s <= s0 && i <= s, "bad product index");
  if constexpr (i >= NPA) return c;
  else return xdl(a[i], b[s - i], c);
}
__device__ __forceinline__ u4 neg_bf16x8(const u4& v) { return v ^ u4{0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u}; }

// LDS records: 8 bf16 (16 bytes) per (row, lane group g), stored [g][row] so that the 16 lanes of a
// group read consecutive records (no bank conflicts); one plane per piece.
__device__ __forceinline__ constexpr int xrec(int row, int g, int rows) { return g * rows + row; }
template <int NP>
struct XdlBC {
  u4 cs_r[NP][XT * 4];   // row t: [ Cr[4g..4g+3], -Ci[4g..4g+3] ]   (real part of C.x)
  u4 cs_i[NP][XT * 4];   // row t: [ Ci[4g..4g+3],  Cr[4g..4g+3] ]   (imaginary part of C.x)
  u4 bs[NP][XT * 4];     // row s: [ Br[4g..4g+3],  Bi[4g..4g+3] ]
  u4 bs_c[NP][XT * 4];   // row s: [-Bi[4g..4g+3],  Br[4g..4g+3] ]   (written by the same code path as cs_i)
  u4 bt_r[NP][XN * 4];   // row n: Br[t(g, e)][n], e = 0..7
  u4 bt_i[NP][XN * 4];   //        Bi
};
template <int NP>
struct XdlG {
  u4 re[NP][XT * 4];     // row t: G[t][t(g, e)], e = 0..7 (zero where s > t)
  u4 im[NP][XT * 4];
};

// Inputs as they lie in memory, kept raw in registers from the (early) load to the use: float
// tensors as they are, bf16 tensors as packed words that are widened where they are consumed
// (a bf16 value is the upper half of the float of the same value).
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
// four consecutive real inputs of a channel
template <typename Tin> struct Raw4;
template <> struct Raw4<float> {
  f4 v;
  __device__ __forceinline__ void load(const float* p) { v = *reinterpret_cast<const f4*>(p); }
  __device__ __forceinline__ float get(int i) const { return v[i]; }
  __device__ __forceinline__ void touch() const { touch_vgpr(v[0]); touch_vgpr(v[1]); touch_vgpr(v[2]); touch_vgpr(v[3]); }
};
template <> struct Raw4<bf16_t> {
  u2 v;
  __device__ __forceinline__ void load(const bf16_t* p) { v = *reinterpret_cast<const u2*>(p); }
  __device__ __forceinline__ float get(int i) const { return (i & 1) ? bf16_hi(v[i >> 1]) : bf16_lo(v[i >> 1]); }
  __device__ __forceinline__ void touch() const { touch_vgpr(__uint_as_float(v[0])); touch_vgpr(__uint_as_float(v[1])); }
};
// one complex input (re, im)
template <typename Tin> struct RawC;
template <> struct RawC<float> {
  float2 v;
  __device__ __forceinline__ void load(const float* p) { v = *reinterpret_cast<const float2*>(p); }
  __device__ __forceinline__ float re() const { return v.x; }
  __device__ __forceinline__ float im() const { return v.y; }
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(v.x), "+v"(v.y)); }
};
template <> struct RawC<bf16_t> {
  uint32_t v;
  __device__ __forceinline__ void load(const bf16_t* p) { v = *reinterpret_cast<const uint32_t*>(p); }
  __device__ __forceinline__ float re() const { return bf16_lo(v); }
  __device__ __forceinline__ float im() const { return bf16_hi(v); }
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(v)); }
};
// four consecutive complex inputs of a state row
template <typename Tin> struct RawC4;
template <> struct RawC4<float> {
  f4 a, b;
  __device__ __forceinline__ void load(const float* p) {
    a = *reinterpret_cast<const f4*>(p);
    b = *reinterpret_cast<const f4*>(p + 4);
  }
  __device__ __forceinline__ float re(int j) const { return j < 2 ? a[2 * j] : b[2 * j - 4]; }
  __device__ __forceinline__ float im(int j) const { return j < 2 ? a[2 * j + 1] : b[2 * j - 3]; }
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(a), "+v"(b)); }
};
template <> struct RawC4<bf16_t> {
  u4 a;
  __device__ __forceinline__ void load(const bf16_t* p) { a = *reinterpret_cast<const u4*>(p); }
  __device__ __forceinline__ float re(int j) const { return bf16_lo(a[j]); }
  __device__ __forceinline__ float im(int j) const { return bf16_hi(a[j]); }
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(a)); }
};

// Requires: N <= 16, L % 4 == 0, u/delta/theta/z/y 16-byte aligned, B/C 16-byte aligned,
// ck % 32 == 0.  Tin: float or bf16_t (u, delta, B, C).  The launcher checks these and otherwise
// takes the generic kernel.
template <int NP, bool GATED, typename Tin = float>
__global__ __launch_bounds__(256) void unitary_fwd_xdl_kernel(const FwdArgs p) {
  __shared__ XdlBC<NP> s_bc[3];
  __shared__ XdlG<NP> s_g[2];

  const int wg = xcd_remap(blockIdx.x, gridDim.x);
  const int b = wg / p.ncg, d0 = (wg % p.ncg) * CH;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
  const int dl = lane & 15, g = lane >> 4;
  const int D = p.D, N = p.N;
  const int d = d0 + wave * 16 + dl;
  const bool dok = d < D;
  const int dc = dok ? d : D - 1;
  // b counts (batch element, segment of p.L steps) pairs when the launcher has split the sequence; the last segment may
  // be shorter
  const int bb = b / p.ns, sg = b - bb * p.ns;
  const size_t so = (size_t)sg * p.L;
  const int L = p.ld - (int)so < p.L ? p.ld - (int)so : p.L;
  const size_t row = ((size_t)bb * D + dc) * p.ld + so;
  const Tin* __restrict__ gu = static_cast<const Tin*>(p.u) + row;
  const Tin* __restrict__ gdl = static_cast<const Tin*>(p.delta) + row;
  const float* __restrict__ gth = p.theta + row;
  const float* __restrict__ gz = GATED ? p.z + row : nullptr;
  const Tin* __restrict__ gB = static_cast<const Tin*>(p.Bm);
  const Tin* __restrict__ gC = static_cast<const Tin*>(p.Cm);
  const float dsk = (p.Dskip && dok) ? p.Dskip[dc] : 0.0f;
  const int nchunks = (L + XT - 1) / XT;
  const SplitK sk = make_splitk();
  constexpr int NPA = sizeof(Tin) == 2 ? 1 : NP;   // non-zero pieces of the staged B / C records

  // G tiles above the block diagonal are read (as zeros) but never written
  for (int i = tid; i < (int)(sizeof(s_g) / 16); i += 256) reinterpret_cast<u4*>(s_g)[i] = u4{0, 0, 0, 0};

  // ---- B/C staging, first mapping: thread (t = tid % 32, g1 = (tid / 32) % 4) of C (tid < 128) or
  // B (tid >= 128) builds the record [row t][g1] from the four state rows 4 g1 .. 4 g1 + 3.
  const int m1_t = tid & 31, m1_g = (tid >> 5) & 3;
  const bool m1_isB = tid >= 128;
  const Tin* __restrict__ m1_src = m1_isB ? gB : gC;
  RawC<Tin> m1_raw[4];
  // second mapping: thread (n = tid % 16, g2 = (tid / 16) % 4, half = (tid / 64) % 2) reads the four
  // timesteps 16 half + 4 g2 .. + 3 of row n of B; tid < 128 writes the Br half-record, the
  // others the Bi and -Bi half-records.
  const int m2_n = tid & 15, m2_g = (tid >> 4) & 3, m2_half = (tid >> 6) & 1;
  const bool m2_im = tid >= 128;
  RawC4<Tin> m2_raw;
  auto bc_load = [&](int c) {
    const int l = c * XT + m1_t;
    const int lc = l < L ? l : 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int n = 4 * m1_g + k;
      const size_t o = (((size_t)bb * N + (n < N ? n : 0)) * p.ld + so + lc) * 2;
      m1_raw[k].load(m1_src + o);
    }
    const int l2 = c * XT + 16 * m2_half + 4 * m2_g;
    const int l2c = l2 < L ? l2 : 0;
    const size_t o2 = (((size_t)bb * N + (m2_n < N ? m2_n : 0)) * p.ld + so + l2c) * 2;
    m2_raw.load(gB + o2);
  };
  // Branch-free: C threads write [re, -im] -> cs_r and [im, re] -> cs_i, B threads [re, im] -> bs and
  // [-im, re] -> bs_c; real-part threads of the second mapping write bt_r, the others bt_i.
  const uint32_t m1_s1 = m1_isB ? 0u : 0x80008000u, m1_s2 = m1_isB ? 0x80008000u : 0u;
  // (only the NPA pieces that can be non-zero are formed and stored; the others are never read)
  auto bc_store = [&](int c, XdlBC<NP>& s) {
    {
      const bool tok = c * XT + m1_t < L;
      float x[8];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bool ok = tok && (4 * m1_g + k < N);
        x[k] = ok ? m1_raw[k].re() : 0.0f;
        x[4 + k] = ok ? m1_raw[k].im() : 0.0f;
      }
      u4 pc[NPA];
      split8<NPA>(sk, x, pc);
      const int o = xrec(m1_t, m1_g, XT);
      u4* d1 = m1_isB ? &s.bs[0][0] : &s.cs_r[0][0];
      u4* d2 = m1_isB ? &s.bs_c[0][0] : &s.cs_i[0][0];
#pragma unroll
      for (int q = 0; q < NPA; ++q) {
        d1[q * (XT * 4) + o] = u4{pc[q][0], pc[q][1], pc[q][2] ^ m1_s1, pc[q][3] ^ m1_s1};
        d2[q * (XT * 4) + o] = u4{pc[q][2] ^ m1_s2, pc[q][3] ^ m1_s2, pc[q][0], pc[q][1]};
      }
    }
    {
      const bool ok = (m2_n < N) && (c * XT + 16 * m2_half + 4 * m2_g < L);
      const float v0 = ok ? (m2_im ? m2_raw.im(0) : m2_raw.re(0)) : 0.0f, v1 = ok ? (m2_im ? m2_raw.im(1) : m2_raw.re(1)) : 0.0f;
      const float v2 = ok ? (m2_im ? m2_raw.im(2) : m2_raw.re(2)) : 0.0f, v3 = ok ? (m2_im ? m2_raw.im(3) : m2_raw.re(3)) : 0.0f;
      uint32_t a[NPA], c2[NPA];
      split2<NPA>(sk, v0, v1, a);
      split2<NPA>(sk, v2, v3, c2);
      const int o = xrec(m2_n, m2_g, XN) * 2 + m2_half;   // 8-byte half-record index
      u2* d1 = reinterpret_cast<u2*>(m2_im ? &s.bt_i[0][0] : &s.bt_r[0][0]);
#pragma unroll
      for (int q = 0; q < NPA; ++q) d1[q * (XN * 4 * 2) + o] = u2{a[q], c2[q]};
    }
  };

  // ---- G^T tile of one wavefront (rows s of tile st, columns t of tile tt): wave 0 -> (tt 0,
  // st 0), 1 -> (1, 0), 2 and 3 -> (1, 1) (the same values twice: cheaper than a branch).
  // A lane ends up with G[t = 16 tt + dl][s = 16 st + 4 g + i], i = 0..3: half a record of row t.
  const int gtt = wave >= 1 ? 1 : 0, gst = wave >= 2 ? 1 : 0;
  const int g_lim = (gtt == gst) ? dl : 64;   // diagonal tiles keep s <= t (a per-lane bound: no branch)
  auto make_g = [&](const XdlBC<NP>& s, XdlG<NP>& o) {
    u4 a[NP], br[NP], bi[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      a[q] = s.bs[q][xrec(16 * gst + dl, g, XT)];
      br[q] = s.cs_r[q][xrec(16 * gtt + dl, g, XT)];
      bi[q] = s.cs_i[q][xrec(16 * gtt + dl, g, XT)];
    }
    f4 gr = xmm_pp<NP, NPA>(a, br, f4{0, 0, 0, 0});
    f4 gi = xmm_pp<NP, NPA>(a, bi, f4{0, 0, 0, 0});
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool keep = 4 * g + i <= g_lim;
      gr[i] = keep ? gr[i] : 0.0f;
      gi[i] = keep ? gi[i] : 0.0f;
    }
    uint32_t r0[NP], r1[NP], i0[NP], i1[NP];
    split2<NP>(sk, gr[0], gr[1], r0);
    split2<NP>(sk, gr[2], gr[3], r1);
    split2<NP>(sk, gi[0], gi[1], i0);
    split2<NP>(sk, gi[2], gi[3], i1);
    const int h = xrec(16 * gtt + dl, g, XT) * 2 + gst;   // 8-byte half-record index
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      reinterpret_cast<u2*>(o.re[q])[h] = u2{r0[q], r1[q]};
      reinterpret_cast<u2*>(o.im[q])[h] = u2{i0[q], i1[q]};
    }
  };

  // ---- channel data of one chunk: two runs of four timesteps per lane.  Loads are unconditional
  // from a clamped address; out-of-range runs are zeroed where they are used.
  struct In { Raw4<Tin> u[2], de[2]; f4 th[2], z[2]; };
  auto in_load = [&](In& r, int c) {
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const int l = c * XT + 16 * st + 4 * g;
      const int lc = l < L ? l : 0;
      r.u[st].load(gu + lc);
      r.de[st].load(gdl + lc);
      r.th[st] = *reinterpret_cast<const f4*>(gth + lc);
      if (GATED) r.z[st] = *reinterpret_cast<const f4*>(gz + lc);
    }
  };
  auto in_touch = [&](const In& r) {
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      r.u[st].touch(); r.de[st].touch(); touch4(r.th[st]);
      if (GATED) touch4(r.z[st]);
    }
  };

  // ---- per-channel vector work of one chunk: phases, rotations, rotated inputs (split)
  struct Prep {
    float cs[2][4], sn[2][4];
    u4 vr[NP], vi[NP], nvi[NP];
    f4 u[2], z[2];
    float cT, sT;
  };
  // first half: phases of the chunk, reduced to (-pi, pi] when any of them is large so that the
  // running sums stay small enough for sincos_small and for fp32 sums of 32 terms
  auto prep_phase = [&](const In& r, int c, float (&th)[2][4]) {
    bool big = false;
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const bool ok = c * XT + 16 * st + 4 * g < L;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        th[st][i] = ok ? r.th[st][i] : 0.0f;
        big |= fabsf(th[st][i]) > 4.0f;
      }
    }
    if (__builtin_expect(__any(big), 0)) {
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int i = 0; i < 4; ++i) th[st][i] = (float)remainder((double)th[st][i], 6.283185307179586476925);
    }
  };
  auto prep_rest = [&](const In& r, int c, float (&th)[2][4], Prep& o) {
    float w[2][4];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const bool ok = c * XT + 16 * st + 4 * g < L;
#pragma unroll
      for (int i = 0; i < 4; ++i) { o.u[st][i] = r.u[st].get(i); w[st][i] = ok ? r.de[st].get(i) * o.u[st][i] : 0.0f; }
      th[st][1] += th[st][0]; th[st][2] += th[st][1]; th[st][3] += th[st][2];
      if (GATED) o.z[st] = r.z[st];
    }
    // exclusive offsets over the order (st 0: g 0..3), (st 1: g 0..3)
    float sa = th[0][3], sb = th[1][3];
    {
      float ta = __shfl_up(sa, 16), tb = __shfl_up(sb, 16);
      if (g >= 1) { sa += ta; sb += tb; }
      ta = __shfl_up(sa, 32); tb = __shfl_up(sb, 32);
      if (g >= 2) { sa += ta; sb += tb; }
    }
    const float tot_a = __shfl(sa, 48 + dl);
    const float off_a = sa - th[0][3];
    const float off_b = tot_a + sb - th[1][3];
    float vr[8], vi[8];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float ph = th[st][i] + (st ? off_b : off_a);
        sincos_small(ph, &o.sn[st][i], &o.cs[st][i]);
        vr[4 * st + i] = o.cs[st][i] * w[st][i];
        vi[4 * st + i] = -o.sn[st][i] * w[st][i];
      }
    }
    split8<NP>(sk, vr, o.vr);
    split8<NP>(sk, vi, o.vi);
#pragma unroll
    for (int q = 0; q < NP; ++q) o.nvi[q] = neg_bf16x8(o.vi[q]);
    // rotation over the whole chunk: the element (st 1, g 3, i 3) is timestep 31
    o.cT = __shfl(o.cs[1][3], 48 + dl);
    o.sT = __shfl(o.sn[1][3], 48 + dl);
  };

  // ---- state: lane (dl, g) holds H[n = 4 g + i][channel dl]
  f4 Hr = {0, 0, 0, 0}, Hi = {0, 0, 0, 0};
  if (p.h0 && dok) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = 4 * g + i;
      if (n < N) {
        const size_t o = (((size_t)bb * D + d) * N + n) * 2;
        Hr[i] = p.h0[o];
        Hi[i] = p.h0[o + 1];
      }
    }
  }

  if (p.seg) seg_enter<false>(p, bb, sg, dc, g, Hr, Hi);

  int i0 = 0, i1 = 1, i2 = 2;   // LDS slots of chunks c, c+1, c+2
  const int ck_chunks = p.ck / XT;
  int ck_left = ck_chunks;           // chunks to the next checkpoint
  // this lane's rows n = 4 g .. 4 g + 3 of checkpoint 0; one checkpoint further = N * 2 * D floats
  float* __restrict__ hck_ptr = p.hck ? p.hck + ((((size_t)bb * p.nck + sg * (p.L / p.ck)) * N + 4 * g) * 2) * D + dc : nullptr;
  const size_t hck_stride = (size_t)N * 2 * D;

  // One chunk.  pc: vector work of chunk c (ready); pn: receives that of chunk c + 1, computed from
  // in1 while the matrix pipe works; in2 receives the loads of chunk c + 2.
  //
  // Issue order.  The matrix pipe and the vector ALU run side by side only if their instructions
  // alternate in the wavefront's (in-order) stream.  The step is therefore cut into regions: each
  // holds the matrix instructions of one group of products plus independent vector work, and ends
  // with a scheduling fence.  Inside a region the group barriers ask for one matrix instruction
  // followed by a few vector ones.  Pure arithmetic is not ordered by a fence, so the inputs of a
  // region's vector work pass through pin() after the previous fence and its results through
  // touch_vgpr() before the next one.
#define XDL_REGION(NMFMA, NVALU)                                  \
  _Pragma("unroll") for (int k_ = 0; k_ < (NMFMA); ++k_) {        \
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);            \
    __builtin_amdgcn_sched_group_barrier(0x002, (NVALU), 0);      \
  }                                                               \
  __builtin_amdgcn_sched_barrier(0)
  constexpr int NPP = NP * (NP + 1) / 2;   // matrix instructions per product
  auto pin = [](float& v) { asm volatile("" : "+v"(v)); };
  auto step = [&](int c, In& in1, In& in2, Prep& pc, Prep& pn) {
    const int l0 = c * XT;
    float th[2][4];
    prep_phase(in1, c + 1, th);     // (holds the only branch of the step)
    __builtin_amdgcn_sched_barrier(0);

    const XdlBC<NP>& s = s_bc[i0];
    const XdlBC<NP>& s1 = s_bc[i1];
    const XdlG<NP>& G = s_g[c & 1];
    XdlG<NP>& Gn = s_g[(c + 1) & 1];
    // ---- region 0: operands of the first products, global loads of chunk c + 2
    u4 hk[NP], ga[NP], gbr[NP], gbi[NP], c_r[2][NP], c_i[2][NP];
    {
      const float x[8] = {Hr[0], Hr[1], Hr[2], Hr[3], Hi[0], Hi[1], Hi[2], Hi[3]};
      split8<NP>(sk, x, hk);
    }
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      ga[q] = s1.bs[q][xrec(16 * gst + dl, g, XT)];
      gbr[q] = s1.cs_r[q][xrec(16 * gtt + dl, g, XT)];
      gbi[q] = s1.cs_i[q][xrec(16 * gtt + dl, g, XT)];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        c_r[tt][q] = s.cs_r[q][xrec(16 * tt + dl, g, XT)];
        c_i[tt][q] = s.cs_i[q][xrec(16 * tt + dl, g, XT)];
      }
    }
    in_load(in2, c + 2);
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int k = 0; k < 4; ++k) touch_vgpr(__uint_as_float(hk[q][k]));
    __builtin_amdgcn_sched_barrier(0);

    // ---- region 1: G^T tile of chunk c + 1  |  staging of B/C of chunk c + 2
#pragma unroll
    for (int k = 0; k < 4; ++k) m1_raw[k].pin();
    m2_raw.pin();
    f4 ggr = xmm_pp<NP, NPA>(ga, gbr, f4{0, 0, 0, 0});
    f4 ggi = xmm_pp<NP, NPA>(ga, gbi, f4{0, 0, 0, 0});
    bc_store(c + 2, s_bc[i2]);
    XDL_REGION(2 * NPP, 12);
    bc_load(c + 3);

    // ---- region 2: S = C.H  |  G tile to LDS, phases and the first rotations of chunk c + 1
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int i = 0; i < 4; ++i) pin(th[st][i]);
    f4 Sr[2], Si[2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      Sr[tt] = xmm_p<NP, NPA>(c_r[tt], hk, f4{0, 0, 0, 0});
      Si[tt] = xmm_p<NP, NPA>(c_i[tt], hk, f4{0, 0, 0, 0});
    }
    {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool keep = 4 * g + i <= g_lim;
        ggr[i] = keep ? ggr[i] : 0.0f;
        ggi[i] = keep ? ggi[i] : 0.0f;
      }
      uint32_t r0[NP], r1[NP], j0[NP], j1[NP];
      split2<NP>(sk, ggr[0], ggr[1], r0);
      split2<NP>(sk, ggr[2], ggr[3], r1);
      split2<NP>(sk, ggi[0], ggi[1], j0);
      split2<NP>(sk, ggi[2], ggi[3], j1);
      const int h = xrec(16 * gtt + dl, g, XT) * 2 + gst;   // 8-byte half-record index
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        reinterpret_cast<u2*>(Gn.re[q])[h] = u2{r0[q], r1[q]};
        reinterpret_cast<u2*>(Gn.im[q])[h] = u2{j0[q], j1[q]};
      }
    }
    float w[8], ph[8];
    {
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const bool ok = (c + 1) * XT + 16 * st + 4 * g < L;
#pragma unroll
        for (int i = 0; i < 4; ++i) { pn.u[st][i] = in1.u[st].get(i); w[4 * st + i] = ok ? in1.de[st].get(i) * pn.u[st][i] : 0.0f; }
        th[st][1] += th[st][0]; th[st][2] += th[st][1]; th[st][3] += th[st][2];
        if (GATED) pn.z[st] = in1.z[st];
      }
      // exclusive offsets over the order (st 0: g 0..3), (st 1: g 0..3)
      float sa = th[0][3], sb = th[1][3];
      float ta = __shfl_up(sa, 16), tb = __shfl_up(sb, 16);
      if (g >= 1) { sa += ta; sb += tb; }
      ta = __shfl_up(sa, 32); tb = __shfl_up(sb, 32);
      if (g >= 2) { sa += ta; sb += tb; }
      const float tot_a = __shfl(sa, 48 + dl);
      const float off_a = sa - th[0][3];
      const float off_b = tot_a + sb - th[1][3];
#pragma unroll
      for (int e = 0; e < 8; ++e) ph[e] = th[e >> 2][e & 3] + ((e >> 2) ? off_b : off_a);
    }
    float* pcs = &pn.cs[0][0];
    float* psn = &pn.sn[0][0];
#pragma unroll
    for (int e = 0; e < 2; ++e) { sincos_small(ph[e], &psn[e], &pcs[e]); touch_vgpr(psn[e]); touch_vgpr(pcs[e]); }
    u4 b_r[NP], b_i[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      b_r[q] = s.bt_r[q][xrec(dl, g, XN)];
      b_i[q] = s.bt_i[q][xrec(dl, g, XN)];
    }
    XDL_REGION(4 * NPP, 7);

    // ---- region 3: H += B^T V  |  remaining rotations of chunk c + 1
#pragma unroll
    for (int e = 2; e < 8; ++e) pin(ph[e]);
    {
      auto quantum = [&](auto ec) {
        constexpr int e = decltype(ec)::value;          // 2..7
        constexpr int k = e - 2;                        // product index 0..5 (NP = 3), clipped below
        sincos_small(ph[e], &psn[e], &pcs[e]);
        touch_vgpr(psn[e]); touch_vgpr(pcs[e]);
        if constexpr (k < NPP) {
          Hr = xmm_k<NP, k, NPA>(b_r, pc.vr, Hr);
          Hi = xmm_k<NP, k, NPA>(b_r, pc.vi, Hi);
          Hr = xmm_k<NP, k, NPA>(b_i, pc.nvi, Hr);
          Hi = xmm_k<NP, k, NPA>(b_i, pc.vr, Hi);
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      quantum(std::integral_constant<int, 2>{}); quantum(std::integral_constant<int, 3>{});
      quantum(std::integral_constant<int, 4>{}); quantum(std::integral_constant<int, 5>{});
      quantum(std::integral_constant<int, 6>{}); quantum(std::integral_constant<int, 7>{});
    }
    u4 g_r[2][NP], g_i[2][NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) {
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        g_r[tt][q] = G.re[q][xrec(16 * tt + dl, g, XT)];
        g_i[tt][q] = G.im[q][xrec(16 * tt + dl, g, XT)];
      }
    }
    XDL_REGION(4 * NPP, 6);

    // ---- region 4: S += G.V  |  rotated inputs of chunk c + 1 (split), state rotation
#pragma unroll
    for (int e = 0; e < 8; ++e) pin(w[e]);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      Sr[tt] = xmm<NP>(g_r[tt], pc.vr, Sr[tt]);
      Si[tt] = xmm<NP>(g_r[tt], pc.vi, Si[tt]);
      Sr[tt] = xmm<NP>(g_i[tt], pc.nvi, Sr[tt]);
      Si[tt] = xmm<NP>(g_i[tt], pc.vr, Si[tt]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float xr = Hr[i], xi = Hi[i];
      Hr[i] = pc.cT * xr - pc.sT * xi;
      Hi[i] = fmaf(pc.cT, xi, pc.sT * xr);
    }
    {
      float vr[8], vi[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        vr[e] = pcs[e] * w[e];
        vi[e] = -psn[e] * w[e];
      }
      split8<NP>(sk, vr, pn.vr);
      split8<NP>(sk, vi, pn.vi);
#pragma unroll
      for (int q = 0; q < NP; ++q) pn.nvi[q] = neg_bf16x8(pn.vi[q]);
      // rotation over the whole chunk: the element (st 1, g 3, i 3) is timestep 31
      pn.cT = __shfl(pcs[7], 48 + dl);
      pn.sT = __shfl(psn[7], 48 + dl);
#pragma unroll
      for (int q = 0; q < NP; ++q)
#pragma unroll
        for (int k = 0; k < 4; ++k) { touch_vgpr(__uint_as_float(pn.vr[q][k])); touch_vgpr(__uint_as_float(pn.nvi[q][k])); }
    }
    XDL_REGION(8 * NPP, 3);

    // ---- outputs: rows 16 tt + 4 g + i of channel dl are this lane's own timesteps
    f4 yo[2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v = pc.cs[tt][i] * Sr[tt][i] - pc.sn[tt][i] * Si[tt][i];
        v = fmaf(dsk, pc.u[tt][i], v);
        if (GATED) v *= siluf_(pc.z[tt][i]);
        yo[tt][i] = v;
      }
    }
    if (p.y && dok) {
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        const int l = l0 + 16 * tt + 4 * g;
        if (l < L) *reinterpret_cast<f4*>(p.y + row + l) = yo[tt];
      }
    }
    // optional: Im(P_t S_t), which the backward pass would otherwise recompute
    if (p.aux && dok) {
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        const int l = l0 + 16 * tt + 4 * g;
        if (l < L) {
          f4 ph;
#pragma unroll
          for (int i = 0; i < 4; ++i) ph[i] = pc.cs[tt][i] * Si[tt][i] + pc.sn[tt][i] * Sr[tt][i];
          *reinterpret_cast<f4*>(p.aux + row + l) = ph;
        }
      }
    }
    // ---- checkpoint: state at the end of every ck-step block and at the end of the sequence
    const bool ck_now = l0 < L && (--ck_left == 0 || l0 + XT >= L);
    if (p.hck && dok && ck_now) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (4 * g + i < N) {
          hck_ptr[(size_t)i * 2 * D] = Hr[i];
          hck_ptr[(size_t)i * 2 * D + D] = Hi[i];
        }
      }
    }
    if (ck_now) { ck_left = ck_chunks; hck_ptr += hck_stride; }
    const int tmp = i0; i0 = i1; i1 = i2; i2 = tmp;
    __syncthreads();
  };
#undef XDL_REGION

  // ---- prologue
  In inA, inB;
  Prep P0, P1;
  bc_load(0);
  in_load(inB, 0);
  in_load(inA, 1);
  bc_store(0, s_bc[0]);
  bc_load(1);
  bc_store(1, s_bc[1]);
  bc_load(2);
  {
    float th[2][4];
    prep_phase(inB, 0, th);
    prep_rest(inB, 0, th, P0);
  }
  __syncthreads();
  make_g(s_bc[0], s_g[0]);
  __syncthreads();

  // Two chunks per trip so that the register sets alternate without copies.  With an odd number of
  // chunks the last half-trip runs on an all-padding chunk: zero input, zero phase, no stores, and
  // the state passes through unchanged.
  for (int c = 0; c < nchunks; c += 2) {
    step(c, inA, inB, P0, P1);
    step(c + 1, inB, inA, P1, P0);
  }

  if (p.aux && blockIdx.x == 0 && tid == 0) p.aux[(size_t)(p.B / p.ns) * D * p.ld] = __uint_as_float(p.auxtag);
  if (p.hL && dok && sg == p.ns - 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = 4 * g + i;
      if (n < N) {
        const size_t o = (((size_t)bb * D + d) * N + n) * 2;
        p.hL[o] = Hr[i];
        p.hL[o + 1] = Hi[i];
      }
    }
  }
}

}  // namespace aussm
