// The host side of the split-product GEMM (gemm_split.h): tile choice,
// split-K and the C entry point.

#include "gemm_split.h"
#include "gemm_rows.h"

#include <stdio.h>
#include <stdlib.h>
#include <string.h>

namespace tjh {

extern template void launch_split<0>(const GemmArgs&, dim3, int, int, bool);
extern template void launch_split<1>(const GemmArgs&, dim3, int, int, bool);
extern template void launch_split<2>(const GemmArgs&, dim3, int, int, bool);
extern template void launch_split<3>(const GemmArgs&, dim3, int, int, bool);
extern template void launch_split<4>(const GemmArgs&, dim3, int, int, bool);
extern template void launch_split<5>(const GemmArgs&, dim3, int, int, bool);

namespace {

struct Plan {
  int tile;
  int64_t splits;
};

// Picks the tile and the K slices of least estimated time, the sum of, in
// microseconds:
//   the larger of (a) the products at the tile's full rate, stretched by
//   how unevenly the workgroups fill the CUs and (b) one workgroup's K steps
//   at the pace of a workgroup alone on its CU, which is fetch latency for
//   the small tiles;
//   a fixed cost (first fetch, epilogue);
//   with slices, writing and adding the partials (5 TB/s) in one launch more.
// Rates are TFLOP/s with the CUs full, as measured on GPT-2's products
// (8192 tokens, 768 to 50257 wide; the chip's power limit holds the clock
// near 1.9 GHz there, where the six bf16 products allow 320): the larger
// the wave tile the fewer LDS bytes and operand splits per product.  The
// steps alone are from products of 8192 x 768 x 768 (96 to 192 of the large
// tiles) and 777 x 768 x 768 (42 to 156 of the small ones).  A CU that runs
// two or three small workgroups hides most of an uneven last round (8192 x
// 2304 x 768 in 4.5 tiles of 128 x 128 per CU: 157 us, 152 at the full
// rate), one or two large ones hide little (256 x 128, 2.25 per CU: 184).
//
// The rounding of a sum grows with the terms of its slice, and the float
// cores split what cannot fill the CUs into slices of 256 k's and more: here
// slices are kept to 400 where the output has fewer 128 x 128 tiles than
// there are CUs, and to 3200 where it has fewer than twice as many, which
// keeps the error at the float products' (logits of GPT-2 over 777 tokens,
// 64-bit reference: 8.2e-7 off in single slices, 7.1e-7 so, 7.1e-7 in float).
//
// TJH_SPLIT_TILE=BMxBN forces a tile (read on every call, so a test can
// sweep the tiles in one process).
//
// With A transposed (a weight gradient, K the tokens) outputs that fill the
// CUs take at least the slices the float cores cut them into: 50257 x 768 x
// 8192 in 2730 (error against 64 bits 7.8e-7, in float 9.1e-7), x 2048 in
// 1024 (5.0e-7, in one slice 6.9e-7; in float 5.9e-7).
Plan choose_plan(int64_t M, int64_t N, int64_t K, int cus, bool wgrad) {
  int forced = -1;
  if (const char* e = getenv("TJH_SPLIT_TILE")) {
    for (int i = 0; i < kNumTiles; ++i) {
      char buf[32];
      snprintf(buf, sizeof(buf), "%dx%d", kTiles[i].bm, kTiles[i].bn);
      if (strncmp(buf, e, strlen(buf)) == 0) forced = i;
    }
  }
  static const double rate[kNumTiles] = {212, 200, 203, 190, 160, 125};
  static const double step[kNumTiles] = {1.84, 1.5, 1.2, 0.62, 0.55, 0.5};
  static const double uneven[kNumTiles] = {0.8, 0.8, 0.8, 0.3, 0.3, 0.3};
  static const double fixed[kNumTiles] = {9, 8, 7, 6, 5, 5};
  const int64_t blocks = cdiv(M, 128) * cdiv(N, 128);
  int64_t slice = blocks >= 2 * cus ? K + 1 : blocks >= cus ? 3200 : 400;
  if (wgrad && blocks >= cus) {
    slice = cdiv(K, 3) < 3200 ? cdiv(K, 3) : 3200;
    if (slice < 1024) slice = 1024;
  }
  int64_t smax = K / 64 < 64 ? K / 64 : 64;
  if (smax < 1) smax = 1;
  int64_t smin = cdiv(K, slice) < smax ? cdiv(K, slice) : smax;
  if (smin < 1) smin = 1;
  Plan best{kNumTiles - 1, 1};
  double best_t = 1e300;
  for (int i = 0; i < kNumTiles; ++i) {
    if (forced >= 0 && i != forced) continue;
    const TileCfg& t = kTiles[i];
    const int64_t tiles = cdiv(M, t.bm) * cdiv(N, t.bn);
    const double work = 2e-6 * tiles * t.bm * t.bn * K / rate[i];
    // slices that make whole rounds of the CUs
    for (int64_t rounds = 0; rounds <= 6; ++rounds) {
      int64_t s = rounds * cus / tiles;
      s = s < smin ? smin : s > smax ? smax : s;
      const double n = (double)tiles * s / cus;
      const double most = (double)cdiv(tiles * s, cus);
      const double full = work * (n < 1 ? 1 : 1 + uneven[i] * (most / n - 1));
      const double alone = cdiv(cdiv(K, s), BK) * step[i];
      double us = full > alone ? full : alone;
      us += fixed[i];
      if (s > 1) us += 5 + 8e-6 * s * M * N / 5;
      if (us < best_t) {
        best_t = us;
        best = Plan{i, s};
      }
    }
  }
  return best;
}

void launch_tile(int ti, const GemmArgs& g, dim3 grid, int ta, int tb, bool edge) {
  switch (ti) {
    case 0: launch_split<0>(g, grid, ta, tb, edge); break;
    case 1: launch_split<1>(g, grid, ta, tb, edge); break;
    case 2: launch_split<2>(g, grid, ta, tb, edge); break;
    case 3: launch_split<3>(g, grid, ta, tb, edge); break;
    case 4: launch_split<4>(g, grid, ta, tb, edge); break;
    default: launch_split<5>(g, grid, ta, tb, edge); break;
  }
}

}  // namespace
}  // namespace tjh

using namespace tjh;

extern "C" int tjh_gemm_split(int transA, int transB, int64_t M, int64_t N, int64_t K, float alpha,
                              const float* A, int64_t lda, const float* B, int64_t ldb, float beta,
                              float* C, int64_t ldc, const float* bias, int bias_mode,
                              const float* residual, int64_t ldr, int act) {
  TJH_REQUIRE_INIT();
  TJH_ARG(M >= 0 && N >= 0 && K >= 0, "tjh_gemm_split: negative size");
  TJH_ARG(bias_mode >= 0 && bias_mode <= 3, "tjh_gemm_split: bad bias_mode %d", bias_mode);
  TJH_ARG(bias_mode != 3 || act == 0, "tjh_gemm_split: bias_mode 3 takes no activation");
  TJH_ARG(bias_mode == 0 || bias, "tjh_gemm_split: bias_mode %d needs a bias pointer", bias_mode);
  TJH_ARG(act == 0 || act == 1 || act == 3, "tjh_gemm_split: bad activation %d", act);
  TJH_ARG(act != 3 || (residual && ldr >= N), "tjh_gemm_split: activation 3 needs residual (ld >= N)");
  if (M == 0 || N == 0) return TJH_OK;
  // row strides must cover the contiguous extent
  TJH_ARG(lda >= (transA ? M : K) || (transA ? M : K) <= 1, "tjh_gemm_split: lda too small");
  TJH_ARG(ldb >= (transB ? K : N) || (transB ? K : N) <= 1, "tjh_gemm_split: ldb too small");
  TJH_ARG(ldc >= N, "tjh_gemm_split: ldc too small");
  // A^T . B^T and row sums of an A stored [M][K] have no kernel here, and
  // sums of fewer than two K steps nothing to gain: the float cores
  if ((transA && transB) || (bias_mode == 3 && !transA) || K < 32) {
    if (act == 1) {  // which keep the pre-activation
      Scratch keep((size_t)(M * N) * sizeof(float));
      if (!keep.ok()) return set_error(TJH_ERR_OOM, "tjh_gemm_split: no scratch");
      return gemm("gemm", transA, transB, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1,
                  bias, bias_mode, keep.as<float>(), N, 1);
    }
    return gemm("gemm", transA, transB, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1,
                bias, bias_mode, const_cast<float*>(residual), ldr, act);
  }
  const int cus = num_cus() > 0 ? num_cus() : 256;
  GemmArgs g{};
  g.A = A; g.B = B; g.C = C; g.bias = bias;
  g.M = M; g.N = N; g.K = K;
  g.lda = lda; g.ldb = ldb; g.ldc = ldc;
  g.alpha = alpha; g.beta = beta; g.bias_mode = bias_mode;
  g.vecA = ((uintptr_t)A & 3) == 0;
  g.vecB = ((uintptr_t)B & 3) == 0;
  g.aux = act == 3 ? const_cast<float*>(residual) : nullptr;
  g.ldaux = ldr;
  g.act = act;
  KernelScope ks("gemm");
  // few rows: nothing to gain from the matrix cores
  if (!transA && transB && M <= kFewRows && g.vecA && g.vecB && cdiv(N, 4) < (int64_t(1) << 31))
    return gemm_rows(g, cus);
  const Plan plan = choose_plan(M, N, K, cus, transA);
  const TileCfg& tc = kTiles[plan.tile];
  g.tiles_m = (int)cdiv(M, tc.bm);
  g.tiles_n = (int)cdiv(N, tc.bn);
  TJH_ARG((int64_t)g.tiles_m * g.tiles_n < (int64_t(1) << 31), "tjh_gemm_split: too many tiles");
  // the sum of partials indexes elements in 32 bits; without scratch for
  // them the product runs in one slice
  int64_t splits = M * N < (int64_t(1) << 32) ? plan.splits : 1;
  g.kchunk = cdiv(cdiv(K, splits), BK) * BK;
  splits = cdiv(K, g.kchunk);
  // K slices: the products' partials, then the row sums'
  const int64_t sums = bias_mode == 3 ? splits * M : 0;
  Scratch ws(splits > 1 ? (size_t)(splits * M * N + sums) * sizeof(float) : 0);
  if (splits > 1 && !ws.ok()) {
    splits = 1;
    g.kchunk = cdiv(K, BK) * BK;
  }
  g.ws = splits > 1 ? ws.as<float>() : nullptr;
  g.rsw = splits > 1 && sums ? g.ws + splits * M * N : nullptr;
  // tiles, K steps or loads that need a guard
  const bool edge = M % tc.bm || N % tc.bn || K % BK || !g.vecA || !g.vecB;
  launch_tile(plan.tile, g, dim3((unsigned)(g.tiles_m * g.tiles_n), (unsigned)splits), transA,
              transB, edge);
  const int rc = check_launch("gemm_split");
  if (rc != TJH_OK || splits == 1) return rc;
  return gemm_splitk_sum(g, splits, 1, cus);
}
