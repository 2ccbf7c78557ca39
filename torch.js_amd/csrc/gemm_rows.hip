// C = alpha * A B^T (+ beta C, bias, GELU or a residual) for up to 8 rows of
// A: the Linear layers of a decoding step, one token for each sequence
// (nn.Linear, src/nn/linear.ts:43-66).
//
// Bound by reading B once: 9.4 MB take 1.5 us at the 6 TB/s of a large copy,
// so the latency of the loads and the last round count.  A wave owns R rows
// of B and holds every product with the rows of A, lanes striding K in 16
// bytes, so each row of B is read once, contiguously, by the whole chip at
// any N; A (at most 8 rows) comes from the L1.  A 64 x 64 matrix-core tile
// multiplies 60 rows of padding instead and needs K slices and a second
// launch to fill the CUs with N / 64 tiles.  Four rows: 2304 and 3072 x 768
// 5.7 us, 768 x 768 and 768 x 3072 4.8 us (tile and sum of slices: 9.8 + 4.9
// on average), 50257 x 768 30 us or 5.1 TB/s (70 us).
#include "gemm_rows.h"

namespace tjh {
namespace {

constexpr int kWaves = 4;

// KS: the waves of a workgroup split K (few columns, long K) and add up
// through LDS; otherwise each wave has R columns of its own.
template <int MR, int R, bool KS>
__global__ __launch_bounds__(64 * kWaves) void k_gemm_rows(GemmArgs g) {
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t n0 = KS ? (int64_t)blockIdx.x * R : ((int64_t)blockIdx.x * kWaves + w) * R;
  __shared__ float part[KS ? kWaves : 1][MR * R];
  if (!KS && n0 >= g.N) return;
  const float* __restrict__ a[MR];
  const float* __restrict__ b[R];
#pragma unroll
  for (int m = 0; m < MR; ++m) a[m] = g.A + (m < g.M ? m : g.M - 1) * g.lda;
#pragma unroll
  for (int r = 0; r < R; ++r) b[r] = g.B + (n0 + r < g.N ? n0 + r : g.N - 1) * g.ldb;
  float acc[MR][R];
#pragma unroll
  for (int m = 0; m < MR; ++m)
#pragma unroll
    for (int r = 0; r < R; ++r) acc[m][r] = 0.f;
  constexpr int kStep = 256;  // k values of a wave's 128-bit load
  const int64_t K4 = g.K & ~(int64_t)3;
#pragma unroll 4
  for (int64_t k = 4 * lane + (KS ? w * kStep : 0); k < K4; k += KS ? kWaves * kStep : kStep) {
    floatx4 bv[R];
#pragma unroll
    for (int r = 0; r < R; ++r) bv[r] = *reinterpret_cast<const floatx4u*>(b[r] + k);
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const floatx4 av = *reinterpret_cast<const floatx4u*>(a[m] + k);
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[m][r] = __builtin_fmaf(av[q], bv[r][q], acc[m][r]);
    }
  }
  if (K4 + lane < g.K && (!KS || w == 0)) {
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r)
        acc[m][r] = __builtin_fmaf(a[m][K4 + lane], b[r][K4 + lane], acc[m][r]);
  }
  // lane m * R + r keeps the sum of (m, r)
  float s = 0.f;
#pragma unroll
  for (int m = 0; m < MR; ++m)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float t = wave_sum(acc[m][r]);
      s = lane == m * R + r ? t : s;
    }
  if (KS) {
    if (lane < MR * R) part[w][lane] = s;
    __syncthreads();
    if (w != 0) return;
    s = 0.f;
    if (lane < MR * R)
      for (int q = 0; q < kWaves; ++q) s += part[q][lane];
  }
  const int64_t row = lane / R, col = n0 + lane % R;
  if (lane >= MR * R || row >= g.M || col >= g.N) return;
  float v = g.alpha * s;
  float* cp = g.C + row * g.ldc + col;
  if (g.beta != 0.f) v += g.beta * *cp;
  if (g.bias_mode == 1) v += g.bias[col];
  else if (g.bias_mode == 2) v += g.bias[row];
  *cp = epilogue_act(g, row, col, v);
}

template <int MR>
void launch_rows(const GemmArgs& g, int cus) {
  const dim3 block(64 * kWaves);
  // four columns a wave where that still gives every SIMD two waves: A is
  // read from the L1 a quarter as often (50257 x 768, four rows).  Fewer
  // columns than two waves a SIMD and more than one load each: the waves of
  // a workgroup share a column's K.
  if (g.N >= 32LL * cus)
    tjh_launch((k_gemm_rows<MR, 4, false>), dim3((unsigned)cdiv(g.N, 4 * kWaves)), block, 0,
               stream(), g);
  else if (g.N >= 8LL * cus || g.K <= 256)
    tjh_launch((k_gemm_rows<MR, 1, false>), dim3((unsigned)cdiv(g.N, kWaves)), block, 0, stream(),
               g);
  else
    tjh_launch((k_gemm_rows<MR, 1, true>), dim3((unsigned)g.N), block, 0, stream(), g);
}

}  // namespace

int gemm_rows(const GemmArgs& g, int cus) {
  if (g.M <= 1) launch_rows<1>(g, cus);
  else if (g.M <= 2) launch_rows<2>(g, cus);
  else if (g.M <= 4) launch_rows<4>(g, cus);
  else launch_rows<8>(g, cus);
  return check_launch("gemm_rows");
}

}  // namespace tjh
