// Splitting the sequence of a unitary scan over workgroups (few (batch, channel) pairs, long L).
//
// The recurrence is linear in the state, so a segment [l0, l0 + Ls) of the sequence acts on the
// state that enters it as  H_out = P H_in + Z  with P = exp(i sum theta) the segment's rotation
// and Z its end state from a zero start; the adjoint runs the other way, A_in = conj(P) A_out + Y
// with Y the adjoint at the segment start from a zero adjoint at its end.  The launcher therefore
//   1. computes (P, Z) or (P, Y) of every segment with unitary_seg_state_kernel (all segments in
//      parallel; only the sums  Z = P sum_s conj(P_s) delta_s u_s B_s,  Y = sum_t conj(P_t) dy_t conj(C_t)
//      are formed: per chunk one product with the channel as free index, on the matrix cores in
//      the layout of the scan kernels),
//   2. runs the scan kernel proper with (batch, segment) pairs as its batch index, every segment
//      starting from what the segments before it make of the state (seg_chain).
#pragma once
#include <type_traits>

#include "scan_fwd_xdl.h"

namespace aussm {


// ADJ = false: Z of each segment, chunks in forward order,  H <- P_T (H + B^T V).
// ADJ = true:  Y of each segment, chunks in reverse order,  A <- conj(P_T) A + conj(C)^T Q.
// Requires N <= 16, L % 4 == 0, 16-byte aligned tensors.  Tin: float or bf16_t (u, delta, B, C).
// mem: SEG_STATE_LDS bytes of LDS; block of blocks: the workgroup's index in this part of the launch.
constexpr int SEG_STATE_LDS = 2 * 2 * 3 * XN * 4 * 16;
template <int NP, bool ADJ, typename Tin = float>
__device__ __forceinline__ void seg_state_body(const SegArgs& p, char* mem, int block, int blocks) {
  // row n: M[t(g, e)][n], real and imaginary parts (the imaginary part negated for ADJ: conj(C))
  static_assert(NP <= 3, "LDS is sized for three pieces");
  u4 (*s_mr)[NP][XN * 4] = reinterpret_cast<u4 (*)[NP][XN * 4]>(mem);
  u4 (*s_mi)[NP][XN * 4] = s_mr + 2;

  const int wg = xcd_remap(block, blocks);
  const int vb = wg / p.ncg, d0 = (wg % p.ncg) * CH;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
  const int dl = lane & 15, g = lane >> 4;
  const int D = p.D, N = p.N;
  const int d = d0 + wave * 16 + dl;
  const bool dok = d < D;
  const int dc = dok ? d : D - 1;
  const int bb = vb / p.ns;
  const size_t so = (size_t)(vb - bb * p.ns) * p.L;
  const int L = p.ld - (int)so < p.L ? p.ld - (int)so : p.L;   // (the last segment may be shorter)
  const size_t row = ((size_t)bb * D + dc) * p.ld + so;
  using TA = typename std::conditional<ADJ, float, Tin>::type;   // dy is always float
  const TA* __restrict__ gx1 = static_cast<const TA*>(p.x1) + row;
  const Tin* __restrict__ gx2 = ADJ ? nullptr : static_cast<const Tin*>(p.x2) + row;
  const Tin* __restrict__ gM = static_cast<const Tin*>(p.M);
  const float* __restrict__ gth = p.theta + row;
  const int nchunks = (L + XT - 1) / XT;
  const SplitK sk = make_splitk();

  // staging: thread (n = tid % 16, g2 = (tid / 16) % 4, half = (tid / 64) % 2) reads the four
  // timesteps 16 half + 4 g2 .. + 3 of row n; tid < 128 writes the real half-record, the others
  // the imaginary one
  const int m2_n = tid & 15, m2_g = (tid >> 4) & 3, m2_half = (tid >> 6) & 1;
  const bool m2_im = tid >= 128;
  RawC4<Tin> m2_raw;
  auto m_load = [&](int c) {
    const int cc = c < 0 ? 0 : (c >= nchunks ? nchunks - 1 : c);
    const int l2 = cc * XT + 16 * m2_half + 4 * m2_g;
    const int l2c = l2 < L ? l2 : 0;
    const size_t o2 = (((size_t)bb * N + (m2_n < N ? m2_n : 0)) * p.ld + so + l2c) * 2;
    m2_raw.load(gM + o2);
  };
  auto m_store = [&](int c, int slot) {
    const bool ok = (m2_n < N) && (c * XT + 16 * m2_half + 4 * m2_g < L);
    const float sg = (ADJ && m2_im) ? -1.0f : 1.0f;
    float v0 = m2_im ? m2_raw.im(0) : m2_raw.re(0), v1 = m2_im ? m2_raw.im(1) : m2_raw.re(1);
    float v2 = m2_im ? m2_raw.im(2) : m2_raw.re(2), v3 = m2_im ? m2_raw.im(3) : m2_raw.re(3);
    v0 = ok ? sg * v0 : 0.0f; v1 = ok ? sg * v1 : 0.0f; v2 = ok ? sg * v2 : 0.0f; v3 = ok ? sg * v3 : 0.0f;
    constexpr int NPS = sizeof(Tin) == 2 ? 1 : NP;   // bf16 values are a single exact piece
    uint32_t a0[NPS], a1[NPS];
    split2<NPS>(sk, v0, v1, a0);
    split2<NPS>(sk, v2, v3, a1);
    const int o = xrec(m2_n, m2_g, XN) * 2 + m2_half;   // 8-byte half-record index
    u4 (*dst)[XN * 4] = m2_im ? s_mi[slot] : s_mr[slot];
#pragma unroll
    for (int q = 0; q < NPS; ++q) reinterpret_cast<u2*>(dst[q])[o] = u2{a0[q], a1[q]};
  };

  struct In { f4 th[2]; Raw4<TA> a[2]; Raw4<Tin> b[2]; };
  auto in_load = [&](In& r, int c) {
    const int cc = c < 0 ? 0 : (c >= nchunks ? nchunks - 1 : c);
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const int l = cc * XT + 16 * st + 4 * g;
      const int lc = l < L ? l : 0;
      r.th[st] = *reinterpret_cast<const f4*>(gth + lc);
      r.a[st].load(gx1 + lc);
      if (!ADJ) r.b[st].load(gx2 + lc);
    }
  };

  // lane (dl, g) holds the state (or adjoint) rows n = 4 g + i of channel dl
  f4 Sr = {0, 0, 0, 0}, Si = {0, 0, 0, 0};
  float pr = 1.0f, pi = 0.0f;   // rotation of the chunks done so far

  In cur;
  const int c_first = ADJ ? nchunks - 1 : 0, c_step = ADJ ? -1 : 1;
  m_load(c_first);
  in_load(cur, c_first);

  for (int k = 0; k < nchunks; ++k) {
    const int c = c_first + k * c_step;
    const int slot = k & 1;
    const int l0 = c * XT;
    m_store(c, slot);
    In nxt;
    m_load(c + c_step);
    in_load(nxt, c + c_step);
    __syncthreads();   // planes of this chunk visible; the other slot was last read one barrier ago

    float th[2][4], x[8];
    bool big = false;
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const bool ok = dok && (l0 + 16 * st + 4 * g < L);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        th[st][i] = ok ? cur.th[st][i] : 0.0f;
        big |= fabsf(th[st][i]) > 4.0f;
        const float v = ADJ ? cur.a[st].get(i) : cur.a[st].get(i) * cur.b[st].get(i);
        x[4 * st + i] = ok ? v : 0.0f;
      }
    }
    if (__builtin_expect(__any(big), 0)) {
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int i = 0; i < 4; ++i) th[st][i] = (float)remainder((double)th[st][i], 6.283185307179586476925);
    }
    // running phase inside the chunk: the lane's two runs of four steps, then across the lane groups
#pragma unroll
    for (int st = 0; st < 2; ++st) { th[st][1] += th[st][0]; th[st][2] += th[st][1]; th[st][3] += th[st][2]; }
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
    float xr[8], xi[8], c7 = 0.0f, s7 = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float ph = th[e >> 2][e & 3] + ((e >> 2) ? off_b : off_a);
      float sn, cs;
      if (e == 7) sincos_small(ph, &sn, &cs);       // (in lane group 3 the rotation of the whole chunk: it accumulates)
      else sincos_small_hw(ph, &sn, &cs);
      xr[e] = cs * x[e];        // x conj(P)
      xi[e] = -sn * x[e];
      if (e == 7) { c7 = cs; s7 = sn; }
    }
    const float cT = __shfl(c7, 48 + dl), sT = __shfl(s7, 48 + dl);   // rotation of the whole chunk
    u4 Xr[NP], Xi[NP], nXi[NP];
    split8<NP>(sk, xr, Xr);
    split8<NP>(sk, xi, Xi);
#pragma unroll
    for (int q = 0; q < NP; ++q) nXi[q] = neg_bf16x8(Xi[q]);
    u4 mr[NP], mi[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) { mr[q] = s_mr[slot][q][xrec(dl, g, XN)]; mi[q] = s_mi[slot][q][xrec(dl, g, XN)]; }
    if (ADJ) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float ar = Sr[i], ai = Si[i];
        Sr[i] = cT * ar + sT * ai;
        Si[i] = cT * ai - sT * ar;
      }
    }
    constexpr int NPA = sizeof(Tin) == 2 ? 1 : NP;   // bf16 B / C: a single exact piece
    Sr = xmm_p<NP, NPA>(mr, Xr, Sr);  Sr = xmm_p<NP, NPA>(mi, nXi, Sr);
    Si = xmm_p<NP, NPA>(mr, Xi, Si);  Si = xmm_p<NP, NPA>(mi, Xr, Si);
    if (!ADJ) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float hr = Sr[i], hi = Si[i];
        Sr[i] = cT * hr - sT * hi;
        Si[i] = cT * hi + sT * hr;
      }
    }
    {
      const float nr = pr * cT - pi * sT, ni = pr * sT + pi * cT;
      pr = nr; pi = ni;
    }
    cur = nxt;
  }

  if (dok) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = 4 * g + i;
      if (n < N) {
        const size_t o = (((size_t)vb * D + d) * N + n) * 2;
        p.out[o] = Sr[i];
        p.out[o + 1] = Si[i];
      }
    }
    if (g == 0) {
      p.ptot[((size_t)vb * D + d) * 2] = pr;
      p.ptot[((size_t)vb * D + d) * 2 + 1] = pi;
    }
  }
}

// Four wavefronts per SIMD (128 registers): the launch of a split call (1024 light workgroups for 64 fine segments
// of a batch of 4 x 4 channel groups) then fits the chip in one round instead of one and a third.
template <int NP, bool ADJ, typename Tin = float>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) void unitary_seg_state_kernel(const SegArgs p) {
  __shared__ __align__(16) char s_mem[SEG_STATE_LDS];
  seg_state_body<NP, ADJ, Tin>(p, s_mem, blockIdx.x, gridDim.x);
}

}  // namespace aussm
