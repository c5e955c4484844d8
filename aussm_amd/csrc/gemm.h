// fp32-accurate matrix products on the bf16 matrix cores: the linear layers of the blocks and the two products with
// the phase adjoints of the fused operator.
//
// Both operands are fp32 in memory and split EXACTLY into three bf16 pieces while they are staged into LDS (scan_fwd_xdl.h:
// split8, xmm<3>): what a product drops is below 2^-26 of it, the sums are fp32; infinities and NaN come out as fp32 sums
// give them (xg_plain).  Workgroup tile 128 x (32 EN), four wavefronts of 64 x (16 EN), 32 of k per step; the values of the
// next step are requested before the products of the current one, and two workgroups per compute unit cover each
// other's barriers.
//
// Operands may be contiguous along k or along their other index (AK1 / BK1), so no transposed copy is ever made:
//   along k: four neighbouring lanes fetch the 32 values of a row (one 128-byte line), 16 bytes at a time;
//   else:    a wavefront fetches all rows' values of one k (up to 512 bytes), eight k in turn.
// TR: the operands change places in the matrix instruction, so that the lanes of a result register run along m,
// for a C that is contiguous along m: the stores and atomics of 16 lanes cover one 64-byte piece either way.
#pragma once
#include "gemm_args.h"
#include "scan_fwd_xdl.h"

#include <type_traits>

namespace aussm {

// Record slot of (row r of a 16-row tile, k group g = 8 values): 16 g + (r + 4 g) % 16.  The rotation keeps the
// 16-byte writes of the along-k mapping (four neighbouring lanes = the four g of one row) and the reads (16
// neighbouring lanes = 16 rows of one g) both free of bank conflicts.
__device__ __forceinline__ int xg_slot(int r, int g) { return 16 * g + ((r + 4 * g) & 15); }

typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));

// split8<3> with the residuals taken by an unpack and a subtract instead of the dot instruction: the same pieces.  Beside
// a busy matrix pipe the dot instruction costs more than the two (256 x 23040, K = 4096 382 us with it, 331 us without).
// (Values that are not finite, or round to infinity in bf16, have no such pieces: xg_plain.)
__device__ __forceinline__ void split8_sub(const float (&x)[8], u4 (&out)[3]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float a = x[2 * q], b = x[2 * q + 1];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const uint32_t pk = pk_bf16(a, b);
      out[p][q] = pk;
      if (p < 2) {
        a -= __uint_as_float(pk << 16);
        b -= __uint_as_float(pk & 0xffff0000u);
      }
    }
  }
}

// One thread's share of an operand tile of H NT / 4 rows x 32 k (NT threads): H records of 8 k each.
//   K1:  row tid / 4 (+ NT / 4), k group tid % 4
//   else rows H lane .. H lane + H - 1 (one load for two rows) of the wavefront's 64 H rows, k group = wavefront % 4: the
//        k index, its bound and the stride along k are scalars, and a load instruction is a scalar base plus the row's offset
// Loads are unconditional (no branch may hide from the compiler how many are in flight): in the last, partial step
// along k they repeat valid elements, and stage() clears what lies past K.  QUAD: K is a multiple of four.
template <bool K1, bool QUAD, int H, int NT>
struct XgOperand {
  const float* row[H];       // K1: this thread's rows; else row[0]: its first row (the second one is next to it)
  long sk;
  int r0, kq;
  struct Vals { float v[H][8]; };
  __device__ __forceinline__ void place(int tid) {
    r0 = K1 ? tid >> 2 : H * (tid & 63) + 64 * H * (wave_index() >> 2);
    kq = 8 * (K1 ? tid & 3 : wave_index() & 3);
  }
  __device__ __forceinline__ int local_row(int h) const { return K1 ? r0 + (NT / 4) * h : r0 + h; }
  __device__ __forceinline__ int slot(int h) const {
    const int r = local_row(h);
    return (r >> 4) * (3 * 64) + xg_slot(r & 15, kq >> 3);
  }
  // pair: (not K1, H == 2) the thread's two rows are neighbours in memory
  __device__ __forceinline__ void fetch(Vals& x, long zoff, int k0, int K, bool pair) const {
    const int k = k0 + kq;
    if constexpr (K1 && QUAD) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int kk = min(k + 4 * q, K - 4);
#pragma unroll
        for (int h = 0; h < H; ++h) {
          const f4u t = *reinterpret_cast<const f4u*>(row[h] + (zoff + kk));
#pragma unroll
          for (int c = 0; c < 4; ++c) x.v[h][4 * q + c] = t[c];
        }
      }
    } else if (!K1 && H == 2 && pair) {                 // uniform
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const f2u t = *reinterpret_cast<const f2u*>(row[0] + (zoff + (long)min(k + c, K - 1) * sk));
        x.v[0][c] = t[0]; x.v[H - 1][c] = t[1];
      }
    } else {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const long o = zoff + (long)min(k + c, K - 1) * (K1 ? 1 : sk);
#pragma unroll
        for (int h = 0; h < H; ++h) x.v[h][c] = row[h][o];
      }
    }
  }
  __device__ __forceinline__ void stage(Vals& x, int k0, int K, u4* __restrict__ lds) const {
    if (k0 + 32 > K) {                                  // uniform
#pragma unroll
      for (int c = 0; c < 8; ++c)
#pragma unroll
        for (int h = 0; h < H; ++h) x.v[h][c] = k0 + kq + c < K ? x.v[h][c] : 0.0f;
    }
#pragma unroll
    for (int h = 0; h < H; ++h) {
      u4 pc[3];
      split8_sub(x.v[h], pc);
#pragma unroll
      for (int c = 0; c < 3; ++c) lds[slot(h) + c * 64] = pc[c];
    }
  }
};

// An infinity, and a finite value that rounds to one in bf16, leaves a NaN in its pieces (inf - inf) and in every sum that it
// enters.  Sums that came out as an infinity or a NaN are formed again here from the values themselves, in fp32 steps: of a
// wavefront's slice `sw` (rows mw .., columns nw ..) those of the steps of its slice of the sum.  64 results at a time: few that
// are not finite one after the other by all lanes, four terms a lane and turn, else one by each lane, which ends
// early where its sum has become a NaN.  256 x 23040, K = 1024, 77 us of finite values: 257 us with one infinity (one lane to
// a sum: 3.3 ms), 114 us of NaN, 11 ms with an infinity in every sum.
// (The arguments are read again: kept in scalar registers across the main loop for this they cost every product.)
template <bool TR, int TM, int TN, int WR, int WN, int LD>
__device__ __forceinline__ void xg_plain(float* __restrict__ sw, int mw, int nw, int lane) {
  typedef const __attribute__((address_space(4))) XGemmArgs* Args;
  Args p = (Args)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  const int tiles = ((p->M + TM - 1) / TM) * ((p->N + TN - 1) / TN), sl = xcd_remap(blockIdx.x, gridDim.x) / tiles;
  const int nk = (p->K + 31) / 32, steps = nk * p->Z, per = (steps + p->slices - 1) / p->slices;
  const int s0 = sl * per, s1 = s0 + per < steps ? s0 + per : steps;
  const long terms = 32l * (s1 - s0);
#pragma unroll 1
  for (int base = 0; base < WR * WN; base += 64) {
    auto row = [](int i) { return TR ? i % WR : i / WN; };
    auto col = [](int i) { return TR ? i / WR : i % WN; };
    auto at = [&](int i) { return sw + (TR ? col(i) * LD + row(i) : row(i) * LD + col(i)); };
    const int own = base + lane;
    const bool bad = mw + row(own) < p->M && nw + col(own) < p->N && !(*at(own) * 0.0f == 0.0f);
    unsigned long long left = __ballot(bad);
    const bool few = __popcll(left) <= 8;
#pragma unroll 1
    while (left) {                                          // (uniform; at most eight turns)
      const int i = few ? base + __ffsll(left) - 1 : own, step = few ? 256 : 4;
      left = few ? left & (left - 1) : 0;
      const int m = min(mw + row(i), p->M - 1), n = min(nw + col(i), p->N - 1), nb = n / p->nper;
      const float* a = p->A + (long)m * p->sam;
      const float* b = p->B + ((long)nb * p->sbb + (long)(n - nb * p->nper) * p->sbn);
      float sum = 0.0f;
#pragma unroll 1
      for (long t = few ? 4 * lane : bad ? 0 : terms; t < terms && sum == sum; t += step) {
        const int s = s0 + (int)(t >> 5), z = s / nk, k = (s - z * nk) * 32 + (int)(t & 31);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const long kk = min(k + j, p->K - 1);
          const float f = fmaf(a[z * p->saz + kk * p->sak], b[z * p->sbz + kk * p->sbk], sum);
          sum = k + j < p->K ? f : sum;
        }
      }
      if (few) {
#pragma unroll
        for (int o = 32; o; o >>= 1) sum += __shfl_xor(sum, o);
        if (lane == 0) *at(i) = sum;
      } else if (bad) {
        *at(i) = sum;
      }
    }
  }
}

// The results go through LDS to the memory: 64 registers written with fixed offsets, then rolled loops over the rows
// along the contiguous index of C - 16 bytes a lane for whole, aligned tiles, else one element a lane (bounds, batch
// borders, atomics).  Unrolled stores straight from the registers, each with its own bounds and offset, made the
// code several times the size of the main loop and covered 64 bytes at a time: 32 x 720 columns, 256 rows, K = 16
// 19.5 us, now 13 us.
//
// WIDE: eight wavefronts on a tile of 256 x (32 EN), both operand tiles twice in LDS, the values two steps ahead.  While the
// wavefronts multiply step s they also split the values of step s + 1 into the other pair of tiles: one barrier a step, and
// a value is split for twice as many products as in the narrow tile.  The first four wavefronts split before they
// multiply, the others after it.  256 x 23040, K = 1024: 94 us narrow, 80 us wide (96 columns: see run_xgemm); of these,
// the matrix instructions alone take 55 us and everything but them 58 us: the two overlap by half.
template <bool AK1, bool BK1, bool TR, int WM, int EM, int EN, bool QUAD, bool WIDE>
__global__ __launch_bounds__(WIDE ? 512 : 256, WIDE ? 1 : 2) void xgemm_kernel(const XGemmArgs p) {
  constexpr int NT = WIDE ? 512 : 256, NWN = NT / 64 / WM;  // wavefronts: WM along the rows, NWN along the columns
  constexpr int TM = 16 * EM * WM, TN = 16 * EN * NWN;      // EM, EN: 16-wide row and column tiles per wavefront
  constexpr int HA = TM > NT / 4 ? 2 : 1, HB = TN > NT / 4 ? 2 : 1;    // records of A and B per thread
  static_assert(TM <= HA * NT / 4 && TN <= HB * NT / 4, "a thread stages at most two records of an operand");
  constexpr int NP = 3;
  constexpr int WN = 16 * EN;                               // columns of a wavefront's block
  constexpr int WR = 16 * EM;                               // ... and rows
  constexpr int LD = (TR ? WR : WN) + 4;                    // row stride of its slice in LDS: WR rows x WN columns, or transposed
  constexpr int SLICE = (TR ? WN : WR) * LD;
  constexpr int ATILE = HA * (NT / 64) * NP * 64, TILES = ATILE + HB * (NT / 64) * NP * 64;   // records of both operand tiles
  constexpr int SLICES = (NT / 256) * SLICE;                // (four slices of SLICE floats = SLICE 16-byte records)
  constexpr int LDS16 = (WIDE ? 2 : 1) * TILES > SLICES ? (WIDE ? 2 : 1) * TILES : SLICES;
  __shared__ u4 s_mem[LDS16];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
  // consecutive logical workgroups share their columns (B is the large operand) and an XCD
  const int tm = (p.M + TM - 1) / TM, tn = (p.N + TN - 1) / TN;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);
  const int m0 = (wg % tm) * TM, n0 = (wg / tm % tn) * TN, sl = wg / (tm * tn);
  const int wm = (wave / NWN) * EM, wn = (wave % NWN) * EN;     // this wavefront's first 16-wide tiles
  f4 acc[EM][EN];
#pragma unroll
  for (int e = 0; e < EM; ++e)
#pragma unroll
    for (int f = 0; f < EN; ++f) acc[e][f] = f4{0, 0, 0, 0};
  // batch and position of the tile's first column; most tiles lie in one batch (no division per column)
  const int nb0 = n0 / p.nper, np0 = n0 - nb0 * p.nper;
  const bool one = np0 + TN <= p.nper || p.nper >= p.N;
  // rows past M / N are fetched from the last valid one (they only reach results that are not stored)
  XgOperand<AK1, QUAD, HA, NT> oa;
  XgOperand<BK1, QUAD, HB, NT> ob;
  oa.place(tid); ob.place(tid);
  oa.sk = p.sak; ob.sk = p.sbk;
#pragma unroll
  for (int h = 0; h < HA; ++h) oa.row[h] = p.A + (long)min(m0 + oa.local_row(h), p.M - 1) * p.sam;
#pragma unroll
  for (int h = 0; h < HB; ++h) {
    const int dn = min(min(ob.local_row(h), TN - 1), p.N - 1 - n0) + np0, nb = one ? 0 : dn / p.nper;
    ob.row[h] = p.B + ((long)(nb0 + nb) * p.sbb + (long)(dn - nb * p.nper) * p.sbn);
  }
  // two neighbouring rows in one load: every pair of the tile exists and lies in one batch (uniform)
  const bool pa = m0 + HA * NT / 4 <= p.M, pb = one && n0 + TN <= p.N;
  const int nk = (p.K + 31) / 32, steps = nk * p.Z, per = (steps + p.slices - 1) / p.slices;
  const int s0 = sl * per, s1 = s0 + per < steps ? s0 + per : steps;
  int fz = s0 / nk, fit = s0 - fz * nk;                     // (z, k step) of the next fetch
  typename XgOperand<AK1, QUAD, HA, NT>::Vals va[2];
  typename XgOperand<BK1, QUAD, HB, NT>::Vals vb[2];
  int sfit = fit;
  const int rslot = xg_slot(lane & 15, lane >> 4);          // the record of (row lane % 16, g lane / 16)
  auto fetch = [&](auto st) {
    constexpr int S = decltype(st)::value;
    oa.fetch(va[S], (long)fz * p.saz, fit * 32, p.K, pa);
    ob.fetch(vb[S], (long)fz * p.sbz, fit * 32, p.K, pb);
    if (++fit == nk) { fit = 0; ++fz; }
  };
  auto stage = [&](auto st, int buf) {
    constexpr int S = decltype(st)::value;
    oa.stage(va[S], sfit * 32, p.K, s_mem + buf * TILES);
    ob.stage(vb[S], sfit * 32, p.K, s_mem + buf * TILES + ATILE);
    if (++sfit == nk) sfit = 0;
  };
  typedef std::integral_constant<int, 0> I0;
  typedef std::integral_constant<int, 1> I1;
  auto multiply = [&](int buf) {
    const u4* const s_a = s_mem + buf * TILES;
    const u4* const s_b = s_a + ATILE;
    u4 rB[EN][NP];
#pragma unroll
    for (int f = 0; f < EN; ++f)
#pragma unroll
      for (int c = 0; c < NP; ++c) rB[f][c] = s_b[((wn + f) * NP + c) * 64 + rslot];
#pragma unroll
    for (int e = 0; e < EM; ++e) {
      u4 rA[NP];
#pragma unroll
      for (int c = 0; c < NP; ++c) rA[c] = s_a[((wm + e) * NP + c) * 64 + rslot];
#pragma unroll
      for (int f = 0; f < EN; ++f) acc[e][f] = xmm<NP>(rA, rB[f], acc[e][f]);
    }
  };
  if (s0 < s1) fetch(I0{});
  if constexpr (WIDE) {
    if (s0 + 1 < s1) fetch(I1{});
    if (s0 < s1) stage(I0{}, 0);
    if (s0 + 2 < s1) fetch(I0{});
    __syncthreads();
    auto run = [&](auto first_tag) {
      constexpr bool FIRST = decltype(first_tag)::value;
      auto step = [&](int s, auto q) {
        constexpr int Q = decltype(q)::value;
        typedef std::integral_constant<int, Q ^ 1> O;
        auto next = [&]() {
          if (s + 1 < s1) {
            stage(O{}, Q ^ 1);
            if (s + 3 < s1) fetch(O{});
          }
        };
        if constexpr (FIRST) next();
        multiply(Q);
        if constexpr (!FIRST) next();
        __syncthreads();
      };
#pragma unroll 1
      for (int s = s0; s < s1; s += 2) {
        step(s, I0{});
        if (s + 1 < s1) step(s + 1, I1{});
      }
    };
    if (wave < 4) run(std::true_type{});
    else run(std::false_type{});
  } else {
#pragma unroll 1
    for (int s = s0; s < s1; ++s) {
      if (s > s0) __syncthreads();
      stage(I0{}, 0);
      __syncthreads();
      if (s + 1 < s1) fetch(I0{});
      multiply(0);
    }
    __syncthreads();
  }
  // result tile (e, f), register a: row 16 e + 4 (lane / 16) + a, column 16 f + lane % 16 of the wavefront's block
  float* const sw = reinterpret_cast<float*>(s_mem) + wave * SLICE;
  const int c = lane & 15, g = lane >> 4;
  float probe[2] = {0.0f, 0.0f};                            // a NaN if a result is one
#pragma unroll
  for (int e = 0; e < EM; ++e)
#pragma unroll
    for (int f = 0; f < EN; ++f) {
#pragma unroll
      for (int a = 0; a < 2; ++a) probe[a] = fmaf(acc[e][f][a], acc[e][f][a + 2], probe[a]);
      if constexpr (TR) *reinterpret_cast<f4*>(sw + (16 * f + c) * LD + 16 * e + 4 * g) = acc[e][f];
      else {
#pragma unroll
        for (int a = 0; a < 4; ++a) sw[(16 * e + 4 * g + a) * LD + 16 * f + c] = acc[e][f][a];
      }
    }
  __builtin_amdgcn_wave_barrier();                          // (a slice belongs to one wavefront)
  const int mw = m0 + 16 * wm, nw = n0 + 16 * wn;
  if (__builtin_expect(__ballot(probe[0] + probe[1] != probe[0] + probe[1]) != 0, 0)) {
    xg_plain<TR, TM, TN, WR, WN, LD>(sw, mw, nw, lane);
    __builtin_amdgcn_wave_barrier();
  }
  const float* const add = p.add ? p.add : p.reduce ? p.C : nullptr;
  constexpr int ROWS = TR ? WN : WR, COLS = TR ? WR : WN;   // rows of the slice run along the contiguous index of C
  if (p.slices > 1) {                                       // uniform: summed into C (TR: one batch, nper = N)
    constexpr int RA = 64 / COLS;                           // lane = column (two rows at a time where 32 fill the row)
    const int q = lane % COLS;
    const bool cok = lane < RA * COLS && (TR ? mw + q < p.M : nw + q < p.N);
    const int dq = nw + q - n0 + np0, bq = (TR || one) ? 0 : dq / p.nper;
    float* const dst = p.C + (TR ? (long)(mw + q) * p.scm : (long)(nb0 + bq) * p.scb + (long)(dq - bq * p.nper) * p.scn);
#pragma unroll 4
    for (int r = lane / COLS; r < ROWS; r += RA) {
      const int o = (TR ? nw : mw) + r;
      if (cok && o < (TR ? p.N : p.M)) atomicAdd(dst + (long)o * (TR ? p.scn : p.scm), p.alpha * sw[r * LD + q]);
    }
    return;
  }
  constexpr int PR = COLS / 4, RR = 64 / PR;                // lanes per row, rows per iteration
  const int q = 4 * (lane % PR);
  // the other index's bounds and strides; four elements that exist, in one batch and aligned, leave as 16 bytes
  const int cnt = lane < RR * PR ? min(4, TR ? p.M - (mw + q) : p.N - (nw + q)) : 0;
  const int dnq = nw + q - n0 + np0, nbq = (TR || one) ? 0 : dnq / p.nper, npq = dnq - nbq * p.nper;
  const bool ptr16 = ((reinterpret_cast<uintptr_t>(p.C) | (add ? reinterpret_cast<uintptr_t>(add) : 0)) & 15) == 0;
  const bool quad = cnt == 4 && (TR || one || npq + 4 <= p.nper);
#pragma unroll 2
  for (int r = lane / PR; r < ROWS; r += RR) {
    if (cnt <= 0 || (TR ? nw : mw) + r >= (TR ? p.N : p.M)) continue;
    f4 v = *reinterpret_cast<const f4*>(sw + r * LD + q) * p.alpha;
    long o;
    if constexpr (TR) {
      const int dn = nw + r - n0 + np0, nb = one ? 0 : dn / p.nper;
      o = (long)(nb0 + nb) * p.scb + (long)(dn - nb * p.nper) * p.scn + (mw + q);
    } else {
      o = (long)(nb0 + nbq) * p.scb + npq + (long)(mw + r) * p.scm;
    }
    if (p.bias) {
#pragma unroll
      for (int a = 0; a < 4; ++a) v[a] = fmaf(p.bias_scale, p.bias[TR ? min(mw + q + a, p.M - 1) : mw + r], v[a]);
    }
    if (quad && ptr16 && (o & 3) == 0) {
      if (add) v += *reinterpret_cast<const f4*>(add + o);
      if (p.act == 1) {
#pragma unroll
        for (int a = 0; a < 4; ++a) v[a] = softplusf_(v[a]);
      }
      *reinterpret_cast<f4*>(p.C + o) = v;
    } else {
      const float x[4] = {v[0], v[1], v[2], v[3]};
#pragma unroll 1
      for (int a = 0; a < cnt; ++a) {
        long oa_ = o + a;
        if (!quad && !TR && !one) {                         // the four may lie in more than one batch
          const int nb = (dnq + a) / p.nper;
          oa_ = (long)(nb0 + nb) * p.scb + (dnq + a - nb * p.nper) + (long)(mw + r) * p.scm;
        }
        float t = a == 0 ? x[0] : a == 1 ? x[1] : a == 2 ? x[2] : x[3];
        if (add) t += add[oa_];
        p.C[oa_] = p.act == 1 ? softplusf_(t) : t;
      }
    }
  }
}

}  // namespace aussm
