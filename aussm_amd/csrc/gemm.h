// fp32-accurate matrix products on the 16-bit matrix cores: the linear layers of the blocks and the two products with
// the phase adjoints of the fused operator.
//
// Both operands are fp32 in memory and split while they are staged into LDS, 32 of k per step.  Two ways (run_xgemm has the rule):
//   bf16: exactly, into three pieces (scan_fwd_xdl.h: split8, xmm<3>), six partial products; what a product drops is below 2^-26
//         of it.  For short sums: one tile of operands, two barriers a step.
//   HALF: each row of A and column of B, scaled by a power of two, into two f16 pieces (split_half.h), three partial products in two
//         accumulators.  Half the matrix instructions, two thirds of the LDS traffic and fewer vector instructions a value (6 cycles a
//         lane against 7); operand tiles twice in LDS, one barrier a step; sums closer to 64 bits because there are half as many
//         additions (relative error of N(0, 1) sums, bf16 / HALF: K = 128 1.52e-7 / 1.10e-7, 512 3.4e-7 / 1.7e-7, 1024 4.8e-7 / 2.2e-7).
// Sums are fp32; infinities and NaN come out as fp32 sums give them (xg_plain).
//
// Operands may be contiguous along k or along their other index (AK1 / BK1), so no transposed copy is ever made:
//   along k: four neighbouring lanes fetch the 32 values of a row (one 128-byte line), 16 bytes at a time;
//   else:    a wavefront fetches all rows' values of one k (up to 512 bytes), eight k in turn.
// TR: the operands change places in the matrix instruction, so that the lanes of a result register run along m,
// for a C that is contiguous along m: the stores and atomics of 16 lanes cover one 64-byte piece either way.
#pragma once
#include "gemm_args.h"
#include "scan_fwd_xdl.h"
#include "split_half.h"

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

// HALF: the scales come from the first step's values, with room for 2048 times the largest of a row and two whole pieces down to
// 2^-17 of it (smaller ones to 2^-40 of it).  Where a value outgrows its scale its first piece is an infinity and the sums
// come out as NaN: the workgroup starts again with scales from all values; so it does at once if a row's first 32 values are
// zeros, which say nothing.  (The operator's phase adjoints grow up to 120-fold along a sequence of 720; with room for 128 its products
// took 1.5 times as long.)  Values of XG_HUGE or more take no part and leave NaN, as an infinity does.
constexpr float XG_HUGE = 8.5070592e37f;   // 2^126
constexpr int XG_ROOM = 10;

// what lies past K, in a step that is not whole
template <int H>
__device__ __forceinline__ void xg_clear(float (&v)[H][8], int k0, int kq, int K) {
  if (k0 + 32 > K) {                                    // uniform
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int h = 0; h < H; ++h) v[h][c] = k0 + kq + c < K ? v[h][c] : 0.0f;
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
  static constexpr int NP = 3, ROWS = H * NT / 4;
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
  __device__ __forceinline__ void clear(Vals& x, int k0, int K) const { xg_clear(x.v, k0, kq, K); }
  __device__ __forceinline__ void stage(const Vals& x, u4* __restrict__ lds) const {
#pragma unroll
    for (int h = 0; h < H; ++h) {
      u4 pc[NP];
      split8_sub(x.v[h], pc);
#pragma unroll
      for (int c = 0; c < NP; ++c) lds[slot(h) + c * 64] = pc[c];
    }
  }
};

// The same for f16 pieces.  A load is a scalar base, 32 bits a thread and (not K1) a scalar offset along k, with no branch on its way: the
// compiler counts the loads that are on their way, and where their number depends on a branch it waits for all.  So the tile's
// rows and a step of z lie within 2 GiB each (run_xgemm), and a fetch that is not `real` reads nothing.
template <bool K1, bool QUAD, int H, int NT>
struct XgHalfOperand {
  static constexpr int NP = 2, ROWS = H * NT / 4;
  const float* base;         // of the tile (uniform)
  uint32_t off[H];           // bytes from there to the thread's rows
  float scale[H];            // of the thread's rows
  int st, r0, kq;
  struct Vals { float v[H][8]; };
  __device__ __forceinline__ void place(int tid) {
    r0 = K1 ? tid >> 2 : (tid & 63) + 64 * H * (wave_index() >> 2);
    kq = 8 * (K1 ? tid & 3 : wave_index() & 3);
  }
  __device__ __forceinline__ int local_row(int h) const { return K1 ? r0 + (NT / 4) * h : r0 + 64 * h; }
  __device__ __forceinline__ int slot(int h) const {
    const int r = local_row(h);
    return (r >> 4) * (NP * 64) + xg_slot(r & 15, kq >> 3);
  }
  __device__ __forceinline__ void fetch(Vals& x, long zoff, int k0, int K, bool real) const {
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base + zoff), 0, __builtin_amdgcn_readfirstlane(real ? -1 : 0), 0x27000);
    if constexpr (K1 && QUAD) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const uint32_t o = 4 * (uint32_t)min(k0 + kq + 4 * q, K - 4);
#pragma unroll
        for (int h = 0; h < H; ++h) {
          const f4 t = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off[h] + o, 0, 0));
#pragma unroll
          for (int c = 0; c < 4; ++c) x.v[h][c + 4 * q] = t[c];
        }
      }
    } else {
      int so = (k0 + kq) * st;                          // (not K1: scalar)
      const int last = (K - 1) * st;
#pragma unroll
      for (int c = 0; c < 8; ++c, so += st) {
        const int o = min(so, last);
#pragma unroll
        for (int h = 0; h < H; ++h)
          x.v[h][c] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, K1 ? off[h] + (uint32_t)o : off[h], K1 ? 0 : o, 0));
      }
    }
  }
  __device__ __forceinline__ void clear(Vals& x, int k0, int K) const { xg_clear(x.v, k0, kq, K); }
  __device__ __forceinline__ void stage(const Vals& x, u4* __restrict__ lds) const {
#pragma unroll
    for (int h = 0; h < H; ++h) {
      u4 pc[NP];
      split8_half<true>(x.v[h], scale[h], pc);
#pragma unroll
      for (int c = 0; c < NP; ++c) lds[slot(h) + c * 64] = pc[c];
    }
  }
  __device__ __forceinline__ void largest(const Vals& x, float (&m)[H]) const {
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const float v = fabsf(x.v[h][c]);
        m[h] = fmaxf(m[h], v < XG_HUGE ? v : 0.0f);
      }
  }
  __device__ __forceinline__ void largest_to(const float (&m)[H], uint32_t* s_most) const {
#pragma unroll
    for (int h = 0; h < H; ++h) atomicMax(s_most + local_row(h), __float_as_uint(m[h]));
  }
  __device__ __forceinline__ void scales(const int* s_exp) {
#pragma unroll
    for (int h = 0; h < H; ++h) scale[h] = exp2_of(s_exp[local_row(h)]);
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
// NW wavefronts, WM of them along the rows.  HALF with eight: one workgroup a compute unit, whose first four wavefronts split the values of
// the next step before they multiply and the others after it, so that either kind of work has half of the chip's wavefronts.
//
// What bounds it, at 256 x 23040, K = 1024 with 256 x 96 (57 us; with six bf16 products 77): without the loads 47, without the matrix
// instructions 47, without the split 49, split and writes to LDS alone 30.  Of the way there: half the matrix instructions 77 -> 72,
// pieces by packed conversions (v_fma_mixlo takes 10 cycles) 61, loads with scalar offsets and two steps ahead 57.
template <bool AK1, bool BK1, bool TR, int NW, int WM, int EM, int EN, bool QUAD, bool HALF>
__global__ __launch_bounds__(64 * NW, HALF && EM * EN <= 4 ? 4 : 2) void xgemm_kernel(const XGemmArgs p) {
  constexpr int NT = 64 * NW, NWN = NW / WM;  // wavefronts: WM along the rows, NWN along the columns
  constexpr int TM = 16 * EM * WM, TN = 16 * EN * NWN;      // EM, EN: 16-wide row and column tiles per wavefront
  constexpr int HA = TM > NT / 4 ? 2 : 1, HB = TN > NT / 4 ? 2 : 1;    // records of A and B per thread
  static_assert(TM <= HA * NT / 4 && TN <= HB * NT / 4, "a thread stages at most two records of an operand");
  typedef std::conditional_t<HALF, XgHalfOperand<AK1, QUAD, HA, NT>, XgOperand<AK1, QUAD, HA, NT>> OpA;
  typedef std::conditional_t<HALF, XgHalfOperand<BK1, QUAD, HB, NT>, XgOperand<BK1, QUAD, HB, NT>> OpB;
  constexpr int NP = HALF ? 2 : 3, NBUF = HALF ? 2 : 1;
  constexpr int WN = 16 * EN;                               // columns of a wavefront's block
  constexpr int WR = 16 * EM;                               // ... and rows
  constexpr int LD = (TR ? WR : WN) + 4;                    // row stride of its slice in LDS: WR rows x WN columns, or transposed
  constexpr int SLICE = (TR ? WN : WR) * LD;
  constexpr int ATILE = OpA::ROWS * 4 * NP, TILES = ATILE + OpB::ROWS * 4 * NP;   // records of both operand tiles
  constexpr int SLICES = (NT / 256) * SLICE;                // (four slices of SLICE floats = SLICE 16-byte records)
  constexpr int LDS16 = NBUF * TILES > SLICES ? NBUF * TILES : SLICES;
  __shared__ u4 s_mem[LDS16];
  constexpr int ROWS_ = OpA::ROWS + OpB::ROWS;              // HALF: rows of A, then of B: largest value, exponent
  __shared__ uint32_t s_most[HALF ? ROWS_ : 1];
  __shared__ int s_exp[HALF ? ROWS_ : 1], s_blank, s_bad;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index();
  // consecutive logical workgroups share their columns (B is the large operand) and an XCD
  const int tm = (p.M + TM - 1) / TM, tn = (p.N + TN - 1) / TN;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);
  const int m0 = (wg % tm) * TM, n0 = (wg / tm % tn) * TN, sl = wg / (tm * tn);
  const int wm = (wave / NWN) * EM, wn = (wave % NWN) * EN;     // this wavefront's first 16-wide tiles
  f4 acc[EM][EN], low[HALF ? EM : 1][HALF ? EN : 1];
  auto zero = [&]() {
#pragma unroll
    for (int e = 0; e < EM; ++e)
#pragma unroll
      for (int f = 0; f < EN; ++f) {
        acc[e][f] = f4{0, 0, 0, 0};
        if constexpr (HALF) low[e][f] = f4{0, 0, 0, 0};
      }
  };
  // batch and position of the tile's first column; most tiles lie in one batch (no division per column)
  const int nb0 = n0 / p.nper, np0 = n0 - nb0 * p.nper;
  const bool one = np0 + TN <= p.nper || p.nper >= p.N;
  // rows past M / N are fetched from the last valid one (they only reach results that are not stored)
  OpA oa;
  OpB ob;
  oa.place(tid); ob.place(tid);
  auto row_a = [&](int h) { return (long)min(m0 + oa.local_row(h), p.M - 1) * p.sam; };
  auto row_b = [&](int h) {
    const int dn = min(min(ob.local_row(h), TN - 1), p.N - 1 - n0) + np0, nb = one ? 0 : dn / p.nper;
    return (long)(nb0 + nb) * p.sbb + (long)(dn - nb * p.nper) * p.sbn;
  };
  if constexpr (HALF) {
    const long fa = (long)m0 * p.sam, fb = (long)nb0 * p.sbb + (one ? (long)np0 * p.sbn : 0);
    oa.base = p.A + fa; ob.base = p.B + fb;
    oa.st = 4 * (int)p.sak; ob.st = 4 * (int)p.sbk;
#pragma unroll
    for (int h = 0; h < HA; ++h) oa.off[h] = 4 * (uint32_t)(row_a(h) - fa);
#pragma unroll
    for (int h = 0; h < HB; ++h) ob.off[h] = 4 * (uint32_t)(row_b(h) - fb);
  } else {
    oa.sk = p.sak; ob.sk = p.sbk;
#pragma unroll
    for (int h = 0; h < HA; ++h) oa.row[h] = p.A + row_a(h);
#pragma unroll
    for (int h = 0; h < HB; ++h) ob.row[h] = p.B + row_b(h);
  }
  // two neighbouring rows in one load: every pair of the tile exists and lies in one batch (uniform)
  const bool pa = m0 + OpA::ROWS <= p.M, pb = one && n0 + TN <= p.N;
  const int nk = (p.K + 31) / 32, steps = nk * p.Z, per = (steps + p.slices - 1) / p.slices;
  const int s0 = sl * per, s1 = s0 + per < steps ? s0 + per : steps;
  int fs, fz, fit, sfit;                                    // next fetch: step and its (z, k step); k step of the next values
  constexpr int AHEAD = HALF && EM * EN <= 12 ? 2 : 1;      // steps whose values are on their way
  typename OpA::Vals va[AHEAD];
  typename OpB::Vals vb[AHEAD];
  auto start = [&]() { fs = s0; fz = s0 / nk; sfit = fit = s0 - fz * nk; };
  const int rslot = xg_slot(lane & 15, lane >> 4);          // the record of (row lane % 16, g lane / 16)
  auto fetch = [&](auto st) {
    constexpr int S = decltype(st)::value % AHEAD;
    if constexpr (HALF) {
      oa.fetch(va[S], (long)fz * p.saz, fit * 32, p.K, fs < s1);
      ob.fetch(vb[S], (long)fz * p.sbz, fit * 32, p.K, fs < s1);
    } else {
      oa.fetch(va[S], (long)fz * p.saz, fit * 32, p.K, pa);
      ob.fetch(vb[S], (long)fz * p.sbz, fit * 32, p.K, pb);
    }
    fs = __builtin_amdgcn_readfirstlane(fs + 1);
    const int k1 = fit + 1 == nk ? 0 : fit + 1;
    fz = __builtin_amdgcn_readfirstlane(fs < s1 && k1 == 0 ? fz + 1 : fz);
    fit = __builtin_amdgcn_readfirstlane(fs < s1 ? k1 : fit);
  };
  typedef std::integral_constant<int, 0> I0;
  typedef std::integral_constant<int, 1> I1;
  auto clear = [&](auto st) {
    constexpr int S = decltype(st)::value % AHEAD;
    oa.clear(va[S], sfit * 32, p.K);
    ob.clear(vb[S], sfit * 32, p.K);
    if (++sfit == nk) sfit = 0;
  };
  auto split = [&](auto st, int buf) {
    constexpr int S = decltype(st)::value % AHEAD;
    oa.stage(va[S], s_mem + buf * TILES);
    ob.stage(vb[S], s_mem + buf * TILES + ATILE);
  };
  auto multiply = [&](int buf) {
    const u4* const s_a = s_mem + buf * TILES;
    const u4* const s_b = s_a + ATILE;
    u4 rB[EN][NP];
#pragma unroll
    for (int f = 0; f < EN; ++f)
#pragma unroll
      for (int c = 0; c < NP; ++c) rB[f][c] = s_b[((wn + f) * NP + c) * 64 + rslot];
    if constexpr (HALF) {
      // rows a tile ahead where registers are left; the two instructions on one sum of mixed pieces far apart
      constexpr int RB = AHEAD == 1 ? 2 : 1;
      u4 rA[RB][NP];
      auto rows = [&](int e) {
#pragma unroll
        for (int c = 0; c < NP; ++c) rA[e % RB][c] = s_a[((wm + e) * NP + c) * 64 + rslot];
      };
      if (RB == 2) rows(0);
#pragma unroll
      for (int e = 0; e < EM; ++e) {
        if (RB == 1 || e + 1 < EM) rows(e + RB - 1);
        const u4 (&a)[NP] = rA[e % RB];
#pragma unroll
        for (int f = 0; f < EN; ++f) low[e][f] = xdl_half(a[1], rB[f][0], low[e][f]);
#pragma unroll
        for (int f = 0; f < EN; ++f) acc[e][f] = xdl_half(a[0], rB[f][0], acc[e][f]);
#pragma unroll
        for (int f = 0; f < EN; ++f) low[e][f] = xdl_half(a[0], rB[f][1], low[e][f]);
      }
      if constexpr (RB == 2) {
        __builtin_amdgcn_sched_group_barrier(0x100, EN * NP + 2 * NP, 0);
#pragma unroll
        for (int e = 0; e < EM; ++e) {
          __builtin_amdgcn_sched_group_barrier(0x008, 3 * EN, 0);
          if (e + 2 < EM) __builtin_amdgcn_sched_group_barrier(0x100, NP, 0);
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < EM; ++e) {
        u4 rA[NP];
#pragma unroll
        for (int c = 0; c < NP; ++c) rA[c] = s_a[((wm + e) * NP + c) * 64 + rslot];
#pragma unroll
        for (int f = 0; f < EN; ++f) acc[e][f] = xmm<NP>(rA, rB[f], acc[e][f]);
      }
    }
  };
  const int c = lane & 15, g = lane >> 4;                   // result tile (e, f), register a: row 16 e + 4 g + a, column 16 f + c
  float probe[2];                                           // a NaN if a result is one
  auto probe_results = [&]() {
    probe[0] = probe[1] = 0.0f;
#pragma unroll
    for (int e = 0; e < EM; ++e)
#pragma unroll
      for (int f = 0; f < EN; ++f)
#pragma unroll
        for (int a = 0; a < 2; ++a) probe[a] = fmaf(acc[e][f][a], acc[e][f][a + 2], probe[a]);
    return __ballot(probe[0] + probe[1] != probe[0] + probe[1]) != 0;
  };
  bool bad;
  if constexpr (HALF) {
    if (tid == 0) s_blank = s_bad = 0;                      // (read behind barriers of the first pass, never cleared)
#pragma unroll 1
    for (int pass = 0;; ++pass) {
      if (tid < ROWS_) s_most[tid] = 0;
      __syncthreads();
      float ma[HA], mb[HB];
#pragma unroll
      for (int h = 0; h < HA; ++h) ma[h] = 0.0f;
#pragma unroll
      for (int h = 0; h < HB; ++h) mb[h] = 0.0f;
      start();
#pragma unroll 1
      for (int s = s0; s < (pass ? s1 : s0 + 1); ++s) {
        fetch(I0{});
        clear(I0{});
        oa.largest(va[0], ma);
        ob.largest(vb[0], mb);
      }
      oa.largest_to(ma, s_most);
      ob.largest_to(mb, s_most + OpA::ROWS);
      __syncthreads();
      if (tid < ROWS_) {
        const float m = __uint_as_float(s_most[tid]);
        s_exp[tid] = half_exponent(m > 0.0f ? m : 1.0f) - (pass ? 0 : XG_ROOM);
        if (!(m > 0.0f)) s_blank = 1;
      }
      __syncthreads();
      if (!pass && __builtin_amdgcn_readfirstlane(s_blank)) continue;
      oa.scales(s_exp);
      ob.scales(s_exp + OpA::ROWS);
      if (pass) {
        start();
        fetch(I0{});
        clear(I0{});
      }
      zero();
      if constexpr (AHEAD == 2) fetch(I1{});
      split(I0{}, 0);
      __builtin_amdgcn_sched_barrier(0);
      fetch(I0{});
      __syncthreads();
      // One step and whole turns of two: what lies past the last step is zeros, and its loads read nothing but are made.  (The compiler
      // counts the loads on their way and waits for all where their number depends on a branch; a way out of the loop between two
      // steps moves the sums to other registers.)
      auto run = [&](auto first_tag) {
        constexpr bool FIRST = decltype(first_tag)::value;
        auto step = [&](auto i) {
          constexpr int Q = decltype(i)::value;
          typedef std::integral_constant<int, Q ^ 1> Next;
          auto next = [&]() {
            clear(Next{});
            split(Next{}, Q ^ 1);
            __builtin_amdgcn_sched_barrier(0);              // (loads moved up would take registers of their own)
            fetch(Next{});
          };
          if constexpr (FIRST) {
            next();
            __builtin_amdgcn_sched_barrier(0);
          }
          multiply(Q);
          if constexpr (!FIRST) {
            __builtin_amdgcn_sched_barrier(0);
            next();
          }
          __syncthreads();
        };
#pragma unroll 1
        for (int r = (s1 - s0) / 2; r > 0; --r) {
          step(I0{});
          step(I1{});
        }
        multiply(0);
      };
      if (NT == 256 || wave < 4) run(std::true_type{});
      else run(std::false_type{});
#pragma unroll
      for (int e = 0; e < EM; ++e)
#pragma unroll
        for (int f = 0; f < EN; ++f)
#pragma unroll
          for (int a = 0; a < 4; ++a)
            acc[e][f][a] = __builtin_amdgcn_ldexpf(fmaf(low[e][f][a], HALF_LO_INV, acc[e][f][a]),
                                                   -(s_exp[16 * (wm + e) + 4 * g + a] + s_exp[OpA::ROWS + 16 * (wn + f) + c]));
      bad = probe_results();
      if (bad && lane == 0) s_bad = 1;
      __syncthreads();                                      // (s_mem has been read, too)
      if (pass || !__builtin_amdgcn_readfirstlane(s_bad)) break;
    }
  } else {
    zero();
    start();
    fetch(I0{});
#pragma unroll 1
    for (int s = s0; s < s1; ++s) {
      if (s > s0) __syncthreads();
      clear(I0{});
      split(I0{}, 0);
      __syncthreads();
      if (s + 1 < s1) fetch(I0{});
      multiply(0);
    }
    bad = probe_results();
    __syncthreads();
  }
  float* const sw = reinterpret_cast<float*>(s_mem) + wave * SLICE;
#pragma unroll
  for (int e = 0; e < EM; ++e)
#pragma unroll
    for (int f = 0; f < EN; ++f) {
      if constexpr (TR) *reinterpret_cast<f4*>(sw + (16 * f + c) * LD + 16 * e + 4 * g) = acc[e][f];
      else {
#pragma unroll
        for (int a = 0; a < 4; ++a) sw[(16 * e + 4 * g + a) * LD + 16 * f + c] = acc[e][f][a];
      }
    }
  __builtin_amdgcn_wave_barrier();                          // (a slice belongs to one wavefront)
  const int mw = m0 + 16 * wm, nw = n0 + 16 * wn;
  if (__builtin_expect(bad, 0)) {
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
