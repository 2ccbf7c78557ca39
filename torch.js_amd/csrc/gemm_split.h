// fp32 GEMM on the CDNA4 bf16 matrix cores: products of floats split into
// three bf16 parts.  Serves the products that no gradient is taken through
// and the weight gradients of vocabulary tables (tjh_gemm_split); gemm.hip's
// float matrix cores serve the other recorded ones, whose roundings a
// training run depends on: AdamW's g / (|g| + eps) amplifies a change of all
// of them to 2e-5 in the second step's gradients of GPT-2, in which the float
// path itself is 1.6e-5 from 64 bits.  A result under no_grad therefore
// differs from the recorded one by roundings.
//
// Stands for matmul.wgsl:17-50 behind Tensor.matmul / mm and nn.Linear
// (Tensor.ts:2132-2331, src/nn/linear.ts:43-66) under no_grad.
//
// C = alpha * op(A) op(B) + beta * C (+ bias), row-major.
//
// Products.  v_mfma_f32_32x32x2_f32 does 64 FLOP per cycle and SIMD, the
// bf16 32x32x16 form 1024.  Each float is split into three bf16 parts that
// sum to it exactly (split2 below) and six of the nine part products are
// added up in float, 2.67 times the float rate.
//
// Sums.  A running sum in the matrix cores is rounded at every instruction:
// at every second k in the float form, six times in 16 k's here.  So there
// are two running sums, one of the product of the leading parts, and one of
// the five others, 2^-7 and less of it, whose roundings do not count: one
// rounding in 16 k's.  Against 64 bits, single slices, normal values: 768
// terms 1.6e-7 (float 5.0e-7, one sum of all six 4.2e-7), 4096 terms 4.0e-7
// (float 1.1e-6); products of positive values or of a constant and values in
// [0, 1) alike (768 terms 1.2e-7 and 1.4e-7, float 3.5e-7 and 3.7e-7, one sum
// 4.0e-7 and 6.2e-7).  The instruction also loses the low bits of its small
// terms to one side, downwards: the mean error of 8192 x 3072 x 768 is 6
// standard errors from zero.  Every second row of A and column of B is
// negated, so that neighbouring elements lose to opposite sides (under 1).
//
// 8192 x 3072 x 768 takes 317-350 us on the float cores and 209-228 us here,
// 50257 x 768 x 8192 (A^T B) 4.8 and 3.6 ms, 777 x 2304 x 768 50 and 34 us.
// What bounds the large ones is power: with random operands the clock falls
// to 1.9 GHz, so data moved per product counts as much as issue slots.
//
// Tiling (a workgroup of WR x WC waves): block tile BM x BN, K step 16; each
// wave owns a (BM / WR) x (BN / WC) sub-tile of 32x32 MFMA blocks, at most 64
// x 64, whose two sums take 128 registers.  Operand tiles are loaded as floats
// into registers one step ahead (two steps on the smaller wave tiles; on 64 x
// 64 the second set is no gain: 8192 x 3072 x 768 226 us with, 213 without),
// split there once per workgroup, and stored as three planes of bf16 in one
// of two LDS buffers.
//   256 x 128, 8 waves of 64 x 64, one workgroup per CU
//   128 x 128, 4 waves of 64 x 64, two per CU
//   128 x 64, 4 waves of 64 x 32, three per CU
//   64 x 64, 4 waves of 32 x 32, four per CU
// Small outputs with long K are split over K; partials are summed by a
// second pass in a fixed order (deterministic).
// MFMA operand layout (32x32x16 bf16): lane l feeds A[m = l%32][k = 8*(l/32)
//   + 0..7] and B[the same k][n = l%32]; accumulator register r of lane l
//   holds C[8*(r/4) + 4*(l/32) + r%4][l%32].
// Operand loads are 128-bit along k, or a wave's 256 consecutive bytes and
// more along the outer index, at any 4-byte alignment (HSA runs the GPU in
// unaligned-access mode; the compiler itself emits such loads for packed
// data), so odd row strides need nothing of their own.  Tiles over the edge
// of the product repeat its last row or column and do not store it; a last K
// step of fewer than 16 is loaded float by float.
// Workgroup order: tiles are grouped 8 M-tiles at a time so neighbouring
// tiles share B columns, and each XCD receives a contiguous run of that
// order so the sharing happens inside one L2.

#pragma once

#include "gemm_args.h"
#include "kahan.h"

namespace tjh {

// ------------------------------------------------------- the operand split

// A float as three bfloat16 parts: x = h + m + l, each part the nearest
// bfloat16 of what is left.  Three times eight significant bits hold the 24
// of a float: the sum is exact while the parts stay above the smallest
// bfloat16 (2^-133; the matrix cores keep subnormal operands), so for |x| >=
// 2^-109; below, an absolute error of at most 2^-134 remains (kTinySum).
// For 1 <= |x| < 2, |m| <= 2^-8 and |l| <= 2^-17, so
// of the nine products of two split numbers the three not formed (m l, l m,
// l l) are at most 2^-24 + 2^-34 of the product, one float rounding of it
// (a tenth of that in the root mean square over normal values).
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx2u __attribute__((ext_vector_type(2), aligned(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{a, b}, bf16x2));
}
__device__ __forceinline__ float bf16_lo(unsigned u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf16_hi(unsigned u) { return __uint_as_float(u & 0xffff0000u); }
// the parts of sign * a and sign * b, packed (the differences are exact)
__device__ __forceinline__ void split2(float a, float b, float sign, unsigned& h, unsigned& m,
                                       unsigned& l) {
  h = pack_bf16(a, b) ^ (sign < 0.f ? 0x80008000u : 0u);
  const float ra = __builtin_fmaf(a, sign, -bf16_lo(h)), rb = __builtin_fmaf(b, sign, -bf16_hi(h));
  m = pack_bf16(ra, rb);
  l = pack_bf16(ra - bf16_lo(m), rb - bf16_hi(m));
}

// LDS layout of one part of an operand tile: per 32 outer indices (m or n)
// a kBlk-byte block of 16-byte chunks (8 k values of one outer index), in
// the order the MFMA reads them: lane l takes outer index l % 32, k = 8
// (l / 32) .. + 7, so a fragment is one contiguous 1 KB read.  The chunks of
// the second k half are rotated by four so that a wave storing both halves
// of neighbouring rows does not meet itself in the LDS banks.
constexpr int kBlk = BK * 32 * 2;
__device__ __forceinline__ int chunk_at(int o, int kq) {
  return (o >> 5) * kBlk + kq * 512 + ((o & 31) ^ (kq << 2)) * 16;
}

// An operand tile of OUTER x BK floats in the registers of T lanes, as items
// of 8 k values x W outer indices.  KC: the operand is stored [outer][k]
// (k contiguous); otherwise [k][outer], and a wave's items share their k
// rows, so a row's address is uniform.  The last pass over the lanes may
// cover part of the workgroup's waves.
// EDGE: outer indices past the end repeat the last one (their products are
// never stored), one at a time.
template <bool KC, int OUTER, int T, bool EDGE>
struct Tile {
  static constexpr int W = !KC && !EDGE && OUTER * BK / 8 / T >= 2 ? 2 : 1;
  static constexpr int NI = OUTER * BK / 8 / W;  // items of the tile
  static constexpr int I = (NI + T - 1) / T;     // items per lane
  static_assert(BK == 16 && NI % 64 == 0 && (KC || OUTER / W % 64 == 0), "whole waves");
  float r[I][W][8];

  __device__ __forceinline__ static bool has(int i) {
    return NI % T == 0 || (int)threadIdx.x + T * i < NI;
  }
  __device__ __forceinline__ static void at(int i, int& o, int& kq) {
    const int f = threadIdx.x + T * i;
    if (KC) {
      o = f >> 1;
      kq = f & 1;
    } else {
      constexpr int Q = OUTER / W;
      kq = __builtin_amdgcn_readfirstlane(f / Q);
      o = (f % Q) * W;
    }
  }
  // Loads the whole K tile at outer index o0, k index k0 of P (row stride
  // ld, `rows` outer indices).
  __device__ __forceinline__ void load(const float* __restrict__ P, int64_t ld, int64_t rows,
                                       int64_t o0, int64_t k0) {
#pragma unroll
    for (int i = 0; i < I; ++i) {
      if (!has(i)) continue;
      int o, kq;
      at(i, o, kq);
      if (EDGE && o0 + o >= rows) o = (int)(rows - 1 - o0);
      if (KC) {
        const float* __restrict__ p = P + (o0 + o) * ld + k0 + kq * 8;
        const floatx4 a = *reinterpret_cast<const floatx4u*>(p);
        const floatx4 b = *reinterpret_cast<const floatx4u*>(p + 4);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          r[i][0][k] = a[k];
          r[i][0][4 + k] = b[k];
        }
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float* __restrict__ p = P + (k0 + kq * 8 + k) * ld + o0;
          if (W == 2) {
            const floatx2 v = *reinterpret_cast<const floatx2u*>(p + (unsigned)o);
            r[i][0][k] = v.x;
            r[i][W - 1][k] = v.y;
          } else {
            r[i][0][k] = p[(unsigned)o];
          }
        }
      }
    }
  }
  // The same float by float, with 0 for k past kend.
  __device__ __forceinline__ void load_tail(const float* __restrict__ P, int64_t ld, int64_t rows,
                                            int64_t kend, int64_t o0, int64_t k0) {
#pragma unroll
    for (int i = 0; i < I; ++i) {
      if (!has(i)) continue;
      int o, kq;
      at(i, o, kq);
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const int64_t go = o0 + o + w < rows ? o0 + o + w : rows - 1;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int64_t gk = k0 + kq * 8 + k;
          r[i][w][k] = gk < kend ? (KC ? P[go * ld + gk] : P[gk * ld + go]) : 0.f;
        }
      }
    }
  }
  // Adds the tile's k values of each outer index to its running sum.
  __device__ __forceinline__ void sum(Kahan (&s)[I][W]) const {
#pragma unroll
    for (int i = 0; i < I; ++i) {
      if (!has(i)) continue;
#pragma unroll
      for (int w = 0; w < W; ++w) {
#pragma unroll
        for (int k = 0; k < 8; ++k) s[i][w].add(r[i][w][k]);
      }
    }
  }
  // Splits the tile and stores its parts in LDS, `part` bytes apart, outer
  // index o negated where it is odd.
  __device__ __forceinline__ void store(char* __restrict__ S, int part) const {
#pragma unroll
    for (int i = 0; i < I; ++i) {
      if (!has(i)) continue;
      int o, kq;
      at(i, o, kq);
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const float sign = (o + w) & 1 ? -1.f : 1.f;
        uintx4 h, m, l;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          unsigned a, b, c;
          split2(r[i][w][2 * q], r[i][w][2 * q + 1], sign, a, b, c);
          h[q] = a;
          m[q] = b;
          l[q] = c;
        }
        char* d = S + chunk_at(o + w, kq);
        *reinterpret_cast<uintx4*>(d) = h;
        *reinterpret_cast<uintx4*>(d + part) = m;
        *reinterpret_cast<uintx4*>(d + 2 * part) = l;
      }
    }
  }
};

// Wave tiles that keep 96 accumulator registers or more run two waves per
// SIMD (256 registers each), smaller ones three or more.
constexpr int gemm_waves_per_simd(int wm, int wn) {
  return wm * wn >= 64 * 64 ? 2 : wm * wn >= 64 * 32 ? 3 : 4;
}

// A sum other than zero of less than this magnitude (as the bits of a float
// shifted left, less one, so that zero is the largest), 2^-75, can show what
// operands under 2^-109 lost.
constexpr unsigned kTinySum = ((127u - 75) << 24) - 1;

// The 32 x 32 block of products over [kbeg, kend) that holds row `row` (of
// this lane's A value) and column `col` (of its B value; both clamped to the
// product) on the float matrix cores, in the accumulator layout above.  Lane
// half h takes k = 8 h .. + 7 of each 16, so a lane's values of an operand
// with k contiguous are two 128-bit loads.
template <bool TA, bool TB>
__device__ __forceinline__ floatx16 float_block(const GemmArgs& g, int64_t row, int64_t col, int h,
                                                int64_t kbeg, int64_t kend) {
  if (row >= g.M) row = g.M - 1;
  if (col >= g.N) col = g.N - 1;
  const float* __restrict__ a = TA ? g.A + row : g.A + row * g.lda;
  const float* __restrict__ b = TB ? g.B + col * g.ldb : g.B + col;
  floatx16 s;
#pragma unroll
  for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll 1
  for (int64_t k0 = kbeg; k0 < kend; k0 += 16) {
    const int64_t k = k0 + 8 * h;
    float x[8], y[8];
    if (k0 + 16 <= kend) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        x[q] = TA ? a[(k + q) * g.lda] : a[k + q];
        y[q] = TB ? b[k + q] : b[(k + q) * g.ldb];
      }
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        x[q] = k + q < kend ? (TA ? a[(k + q) * g.lda] : a[k + q]) : 0.f;
        y[q] = k + q < kend ? (TB ? b[k + q] : b[(k + q) * g.ldb]) : 0.f;
      }
    }
#pragma unroll
    for (int q = 0; q < 8; ++q)
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(x[q], y[q], s, 0, 0, 0);
  }
  return s;
}

template <int BM, int BN, int WR, int WC, bool TA, bool TB, bool EDGE>
__global__ __launch_bounds__(WR * WC * 64, gemm_waves_per_simd(BM / WR, BN / WC)) void k_gemm_split(
    GemmArgs g) {
  constexpr int T = WR * WC * 64;
  constexpr int WM = BM / WR, WN = BN / WC;  // wave tile
  constexpr int FM = WM / 32, FN = WN / 32;  // MFMA blocks per wave
  constexpr int PA = BM * BK * 2, PB = BN * BK * 2, BUF = 3 * (PA + PB);
  static_assert(FM >= 1 && FN >= 1 && FM * 32 == WM && FN * 32 == WN, "tile");
  __shared__ __attribute__((aligned(16))) char lds[2 * BUF];

  // Wave priority: the prologue and the epilogue run at raised priority.
  // Where two workgroups share a CU, at equal priority the one in its
  // epilogue (address arithmetic and stores) barely advances while the
  // other issues MFMAs, and its successor cannot start.
  __builtin_amdgcn_s_setprio(3);
  // ---- tile coordinates (grouped ordering for L2 reuse)
  const int tiles_m = g.tiles_m, tiles_n = g.tiles_n;
  int bid = xcd_tile(blockIdx.x, gridDim.x);
  constexpr int GROUP = 8;
  int group_size = GROUP * tiles_n;
  int group = bid / group_size;
  int first_m = group * GROUP;
  int gm = tiles_m - first_m < GROUP ? tiles_m - first_m : GROUP;
  int in_group = bid % group_size;
  int tm = first_m + in_group % gm;
  int tn = in_group / gm;
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;

  const float* __restrict__ A = g.A;
  const float* __restrict__ B = g.B;
  float* __restrict__ C = g.C;
  // split-K: this workgroup covers K range [kbeg, kend)
  const int64_t kbeg = (int64_t)blockIdx.y * g.kchunk;
  const int64_t kend = kbeg + g.kchunk < g.K ? kbeg + g.kchunk : g.K;

  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const int wm = wid / WC, wn = wid % WC;
  const int l32 = lane & 31, h = lane >> 5;

  floatx16 acc[FM][FN], low[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[i][j][r] = 0.f;
        low[i][j][r] = 0.f;
      }

  // A: logical [M][K]; stored [M][K] (!TA) or [K][M] (TA)
  // B: logical [K][N]; as an "outer = n" tile it is stored [N][K] when TB
  //    (k contiguous, like !TA) and [K][N] when !TB (n contiguous, like TA).
  // `ktiles` whole K tiles; the rest (fewer than BK k values, or all of them
  // where the operands are not 4-byte aligned) is loaded float by float
  const int64_t ktiles = kend > kbeg && (!EDGE || (g.vecA && g.vecB)) ? (kend - kbeg) / BK : 0;
  using TileA = Tile<!TA, BM, T, EDGE>;
  using TileB = Tile<TB, BN, T, EDGE>;
  TileA ta, ta2;
  TileB tb, tb2;
  // bias_mode 3: the workgroups of the first column tile also sum the rows
  // of op(A) over their K range (the bias gradient of a weight gradient),
  // from the floats in flight to LDS
  const bool row_sums = TA && g.bias_mode == 3 && tn == 0;
  Kahan rsum[TileA::I][TileA::W];
  auto fetch = [&](int64_t t, TileA& xa, TileB& xb) {
    const int64_t k0 = kbeg + t * BK;
    xa.load(A, g.lda, g.M, m0, k0);
    xb.load(B, g.ldb, g.N, n0, k0);
  };
  auto stage = [&](int64_t t, TileA& xa, TileB& xb) {
    char* S = lds + (t & 1) * BUF;
    if (TA && row_sums) xa.sum(rsum);
    xa.store(S, PA);
    xb.store(S + 3 * PA, PB);
  };
  // the six products of a K tile, the smallest terms first
  auto compute = [&](int64_t t) {
    const char* S = lds + (t & 1) * BUF;
    const int at = (h << 9) + ((l32 ^ (h << 2)) << 4);
    const char* as = S + wm * FM * kBlk + at;
    const char* bs = S + 3 * PA + wn * FN * kBlk + at;
    constexpr int PI[6] = {2, 1, 0, 1, 0, 0}, PJ[6] = {0, 1, 2, 0, 1, 0};
    bf16x8 bf[FN][3];
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        bf[j][p] = *reinterpret_cast<const bf16x8*>(bs + p * PB + j * kBlk);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      bf16x8 af[3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
        af[p] = *reinterpret_cast<const bf16x8*>(as + p * PA + i * kBlk);
#pragma unroll
      for (int u = 0; u < 6; ++u)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          floatx16& to = u < 5 ? low[i][j] : acc[i][j];
          to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[PI[u]], bf[j][PJ[u]], to, 0, 0, 0);
        }
    }
  };

  // PF2: two K tiles in flight in registers (tile t + 2 is fetched while
  // tile t's MFMAs run), for the wave tiles whose registers allow it
  constexpr bool PF2 = gemm_waves_per_simd(WM, WN) > 2;
  if (ktiles > 0) {
    fetch(0, ta, tb);
    if (PF2 && ktiles > 1) fetch(1, ta2, tb2);
    stage(0, ta, tb);
  }
  __syncthreads();
  __builtin_amdgcn_s_setprio(0);
  // The scheduling barriers keep the loads ahead of the MFMAs (the
  // scheduler sinks them to shorten their registers' lifetimes).
  if constexpr (PF2) {
    const int64_t last = ktiles - 1;
    int64_t t = 0;
    for (; t + 1 < ktiles; t += 2) {  // two steps per pass keep the sets static
      fetch(t + 2 < last ? t + 2 : last, ta, tb);
      __builtin_amdgcn_sched_barrier(0);
      compute(t);
      stage(t + 1, ta2, tb2);
      __syncthreads();
      fetch(t + 3 < last ? t + 3 : last, ta2, tb2);
      __builtin_amdgcn_sched_barrier(0);
      compute(t + 1);
      if (t + 2 < ktiles) stage(t + 2, ta, tb);
      __syncthreads();
    }
    if (t < ktiles) {
      compute(t);
      __syncthreads();
    }
  } else {
    for (int64_t t = 0; t < ktiles; ++t) {
      const bool more = t + 1 < ktiles;
      if (more) fetch(t + 1, ta, tb);
      __builtin_amdgcn_sched_barrier(0);
      compute(t);
      if (more) stage(t + 1, ta, tb);
      __syncthreads();
    }
  }

  if constexpr (EDGE) {
    for (int64_t t = ktiles; kbeg + t * BK < kend; ++t) {
      const int64_t k0 = kbeg + t * BK;
      ta.load_tail(A, g.lda, g.M, kend, m0, k0);
      tb.load_tail(B, g.ldb, g.N, kend, n0, k0);
      stage(t, ta, tb);
      __syncthreads();
      compute(t);
      __syncthreads();
    }
  }

  __builtin_amdgcn_s_setprio(3);
  if (TA && row_sums) {
    // the two k halves of a row are in two lanes, added with what their
    // compensations hold (50257 rows over 8192: 3.9e-8 off 64 bits, 5.6e-8 by
    // plain adds); the operand tiles are free here (the K loop ended on a
    // barrier)
    Kahan(*rp)[BM] = reinterpret_cast<Kahan(*)[BM]>(lds);
#pragma unroll
    for (int i = 0; i < TileA::I; ++i) {
      if (!TileA::has(i)) continue;
      int o, kq;
      TileA::at(i, o, kq);
#pragma unroll
      for (int w = 0; w < TileA::W; ++w) rp[kq][o + w] = rsum[i][w];
    }
    __syncthreads();
    for (int o = threadIdx.x; o < BM && m0 + o < g.M; o += T) {
      Kahan k = rp[0][o];
      const Kahan k1 = rp[1][o];
      const float plain = k.s + k1.s;
      k.add(k1.s);
      k.add(-k1.c);
      // an infinity has no compensation
      const bool fin = plain - plain == 0.f;
      const float sum = fin ? k.s - k.c : plain;
      if (g.rsw) {
        float* w = g.rsw + 2 * blockIdx.y * g.M + m0 + o;
        w[0] = sum;
        w[g.M] = fin ? (k.s - sum) - k.c : 0.f;
      } else {
        const_cast<float*>(g.bias)[m0 + o] = sum;
      }
    }
  }

  // ---- epilogue
  // Element (i, j, r) of this wave sits at row r0 + ro(i, r), column
  // c0 + 32 j, with ro = 32 i + 8 (r / 4) + r % 4.  Addresses are one base
  // per lane plus a uniform row offset (ro x ld, scalar arithmetic), and
  // the beta / bias / activation choice is made once, not per element:
  // the epilogue runs beside the other workgroup's MFMAs, where every
  // vector instruction it issues is slow.
  const int64_t r0 = m0 + wm * WM + 4 * h, c0 = n0 + wn * WN + l32;
  const bool nobias = g.bias_mode == 0 || g.bias_mode == 3;
  float* __restrict__ Wp =
      g.ws ? g.ws + blockIdx.y * g.M * g.N : nullptr;
  // the general case of one element: its sum a at (row, col)
  auto finish = [&](int64_t row, int64_t col, float a) {
    if (Wp) {
      Wp[row * g.N + col] = a;
      return;
    }
    float v = g.alpha * a;
    float* cp = C + row * g.ldc + col;
    if (g.beta != 0.f) v += g.beta * *cp;
    if (g.bias_mode == 1) v += g.bias[col];
    else if (g.bias_mode == 2) v += g.bias[row];
    *cp = epilogue_act(g, row, col, v);
  };
  // The sign of this lane's column; odd rows carry the other one.  It is
  // taken back by a multiply-add with +0, which a sum that is exactly zero
  // leaves as +0, as the float cores do.
  const float sign = l32 & 1 ? -1.f : 1.f, alpha = g.alpha;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] += low[i][j];
  // An infinity or NaN among the operands (or a finite value that rounds to
  // infinity in bfloat16) makes parts of the split NaN: the 32 x 32 blocks
  // whose sums are not all finite are formed again from the floats
  // themselves, on the float matrix cores, with the infinities and NaNs of
  // float arithmetic.  0 * x is 0 for finite x and NaN otherwise.  2048 x
  // 3072 x 768 takes 75 us, with a NaN in every row 243 us (11.3 ms by
  // multiply-adds one after the other, 89 us on gemm.hip's tiles).
  // So are blocks with a sum under 2^-75 but not zero: what the parts lose of
  // operands under 2^-109 is 2^-134 a term times the other operand, which
  // larger sums show nothing of unless that operand times the number of terms
  // exceeds 2^33.  (2048 x 3072 x 768 with operands of 1e-12 takes 225 us.
  // Following the largest operand through the K steps, to know, took 1 to 4%;
  // looking for tiny operands took longer than the block.)
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      float z0 = 0.f, z1 = 0.f;
      unsigned low_sum = ~0u;
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        z0 = __builtin_fmaf(acc[i][j][r], 0.f, z0);
        z1 = __builtin_fmaf(acc[i][j][r + 1], 0.f, z1);
        low_sum = min(low_sum, min((__float_as_uint(acc[i][j][r]) << 1) - 1,
                                   (__float_as_uint(acc[i][j][r + 1]) << 1) - 1));
      }
      const bool again = !(z0 + z1 == 0.f) || low_sum < kTinySum;
      const int64_t row = m0 + wm * WM + i * 32 + l32, col = n0 + wn * WN + j * 32 + l32;
      if (__any(again)) {
        acc[i][j] = float_block<TA, TB>(g, row, col, h, kbeg, kend);
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] *= r & 1 ? -sign : sign;
      }
    }
  auto each = [&](auto&& put) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        if (EDGE && c0 + j * 32 >= g.N) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int ro = i * 32 + 8 * (r >> 2) + (r & 3);
          if (!EDGE || r0 + ro < g.M)
            put(__builtin_fmaf(acc[i][j][r], r & 1 ? -sign : sign, 0.f), ro, j * 32);
        }
      }
  };
  if (Wp) {
    // raw partial sums; the reduce kernel applies alpha / beta / bias
    float* __restrict__ W = Wp + r0 * g.N + c0;
    const int64_t ld = g.N;
    each([&](float a, int ro, int co) { W[ro * ld + co] = a; });
    return;
  }
  float* __restrict__ Cb = C + r0 * g.ldc + c0;
  const int64_t ldc = g.ldc, ldx = g.ldaux;
  float* __restrict__ Xb = g.aux ? g.aux + r0 * ldx + c0 : nullptr;
  if (g.beta == 0.f && nobias && g.act == 0) {
    each([&](float a, int ro, int co) { Cb[ro * ldc + co] = alpha * a; });
    return;
  }
  if (g.beta == 0.f && g.bias_mode == 1 && (g.act == 0 || g.act == 1 || g.act == 3)) {
    // bias per column (+ GELU or + residual)
    const float* __restrict__ bb = g.bias + c0;
    const int act = g.act;
    auto run = [&](auto ACT) {
      constexpr int A_ = decltype(ACT)::value;
      each([&](float a, int ro, int co) {
        float v = alpha * a + bb[co];
        if (A_ == 1) {
          v = gelu_f(v);
        } else if (A_ == 3) {
          v += Xb[ro * ldx + co];
        }
        Cb[ro * ldc + co] = v;
      });
    };
    if (act == 0) run(IConst<0>());
    else if (act == 1) run(IConst<1>());
    else run(IConst<3>());
  } else {
    each([&](float a, int ro, int co) { finish(r0 + ro, c0 + co, a); });
  }
}

struct TileCfg {
  int bm, bn, wr, wc;  // block tile, wave rows and columns
};
constexpr TileCfg kTiles[] = {{256, 128, 4, 2}, {128, 128, 2, 2}, {128, 64, 2, 2}, {64, 64, 2, 2}};
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);

template <int BM, int BN, int WR, int WC, bool EDGE>
void launch_split_e(const GemmArgs& g, dim3 grid, int ta, int tb) {
  const dim3 block(WR * WC * 64);
  if (!ta && !tb)
    tjh_launch((k_gemm_split<BM, BN, WR, WC, false, false, EDGE>), grid, block, 0, stream(), g);
  else if (!ta && tb)
    tjh_launch((k_gemm_split<BM, BN, WR, WC, false, true, EDGE>), grid, block, 0, stream(), g);
  else
    tjh_launch((k_gemm_split<BM, BN, WR, WC, true, false, EDGE>), grid, block, 0, stream(), g);
}

// One launch of tile I.  Each tile's kernels are compiled in a source file
// of their own (gemm_split_*.hip).
template <int I>
void launch_split(const GemmArgs& g, dim3 grid, int ta, int tb, bool edge) {
  constexpr TileCfg t = kTiles[I];
  if (edge) launch_split_e<t.bm, t.bn, t.wr, t.wc, true>(g, grid, ta, tb);
  else launch_split_e<t.bm, t.bn, t.wr, t.wc, false>(g, grid, ta, tb);
}

}  // namespace tjh
