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

namespace {

struct Plan {
  int tile;
  int64_t splits;
};

// Picks the tile and the K slices of least estimated time, the sum of, in
// microseconds:
//   the larger of (a) the products at the tile's full rate, stretched by
//   how unevenly the workgroups fill the CUs, and (b) one workgroup's K steps
//   at the pace of a workgroup alone on its CU, which is fetch latency for
//   the small tiles;
//   a fixed cost (first fetch, epilogue);
//   with slices, writing and adding the partials in one launch more.
// The constants are a least-squares fit to 2433 times of 111 products (12 to
// 8192 rows, 10 to 50257 columns, 40 to 9000 terms, every tile, 1 to 48
// slices), 8% root mean square; its choices are 3.5% off the fastest on
// average.  Rates are TFLOP/s with the CUs full (the chip's power limit holds
// the clock near 1.9 GHz there, where the six bf16 products allow 320).  A
// first round in which every CU holds at least one workgroup, but not its
// fill of `cap`, loses `part` of the idle share, later rounds `uneven`.
// With A transposed the widest tile, which reads the tall operand least, is
// 4% faster than the others (50257 x 768 x 8192: 3.59 ms, 3.79 in 128 x 128).
//
// The rounding of a sum grows with the root of its slice's terms.  The float
// cores cut what cannot fill half the CUs with 128 x 128 tiles into slices of
// 64 k's and more, and what cannot fill them twice into 256 and more.  The two
// sums here round an eighth as often, so slices of eight times that length
// err no more: 512 and 2048 (777 x 768 x 768: 1.1e-7 off 64 bits in two
// slices, 1.6e-7 in one, 1.6e-7 in float; 777 x 1536 x 384 in one: 1.1e-7,
// in float 1.5e-7).
//
// TJH_SPLIT_TILE=BMxBN forces a tile and BMxBN:S its slices (read on every
// call, so a test can sweep them in one process).
Plan choose_plan(int64_t M, int64_t N, int64_t K, int cus, bool ta) {
  int forced = -1;
  int64_t slices = 0;
  if (const char* e = getenv("TJH_SPLIT_TILE")) {
    for (int i = 0; i < kNumTiles; ++i) {
      char buf[32];
      snprintf(buf, sizeof(buf), "%dx%d", kTiles[i].bm, kTiles[i].bn);
      const size_t n = strlen(buf);
      if (strncmp(buf, e, n) == 0 && (e[n] == 0 || e[n] == ':')) {
        forced = i;
        if (e[n] == ':') slices = atoi(e + n + 1);
      }
    }
  }
  static const double rate[kNumTiles] = {201, 200, 155, 120};
  static const double step[kNumTiles] = {1.11, 0.82, 0.61, 0.51};
  static const double fixed[kNumTiles] = {8, 7.8, 6.8, 6.7};
  static const double part[kNumTiles] = {1.2, 0.64, 0.97, 1.2};
  static const double uneven[kNumTiles] = {0.75, 0.59, 0.29, 0.41};
  static const int cap[kNumTiles] = {1, 2, 3, 4};
  const int64_t blocks = cdiv(M, 128) * cdiv(N, 128);
  const int64_t slice = 2 * blocks < cus ? 512 : blocks < 2 * cus ? 2048 : K + 1;
  int64_t smax = K / 64 < 64 ? K / 64 : 64;
  if (smax < 1) smax = 1;
  int64_t smin = cdiv(K, slice) < smax ? cdiv(K, slice) : smax;
  // no more than the float cores' most for an output that fills the CUs: the
  // partials of 4100 x 1024 over 65536 terms stay at 134 MB (32 slices: 537)
  if (blocks >= cus && smin > 8) smin = 8;
  Plan best{kNumTiles - 1, 1};
  double best_t = 1e300;
  for (int i = 0; i < kNumTiles; ++i) {
    if (forced >= 0 && i != forced) continue;
    const TileCfg& t = kTiles[i];
    const int64_t tiles = cdiv(M, t.bm) * cdiv(N, t.bn);
    const double work = 2e-6 * tiles * t.bm * t.bn * K / (ta && i == 0 ? 1.04 * rate[i] : rate[i]);
    // slices that make whole rounds of the CUs
    for (int64_t rounds = 0; rounds <= 6; ++rounds) {
      int64_t s = rounds * cus / tiles;
      s = s < smin ? smin : s > smax ? smax : s;
      if (slices > 0) s = slices;
      const double n = (double)tiles * s / cus;  // workgroups a CU
      const double idle = n <= cap[i] ? part[i] * (cdiv(tiles * s, cus) / n - 1)
                                      : uneven[i] * (cdiv(tiles * s, cap[i] * cus) * cap[i] / n - 1);
      const double full = n < 1 ? work : work * (1 + idle);
      const double alone = cdiv(cdiv(K, s), BK) * step[i];
      double us = (full > alone ? full : alone) + fixed[i];
      if (s > 1) us += 1.8 + 8e-6 * s * M * N / 5.6;
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
    default: launch_split<3>(g, grid, ta, tb, edge); break;
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
  const int cus = num_cus() > 0 ? num_cus() : 256;
  const bool aligned = (((uintptr_t)A | (uintptr_t)B) & 3) == 0;
  // Few rows of A are multiplied where they are (gemm_rows.hip).  More than 4
  // are more to read than B's rows once they leave the L1 (8 x 256 x 65536:
  // 127 us, 47 on the float cores; x 8192: 10 and 16), and with short rows
  // the sums over the lanes are most of the work (8 x 50257 x 64: 18 and 14).
  const bool rows = !transA && transB && M <= kFewRows && K >= 32 && aligned && bias_mode != 3 &&
                    cdiv(N, 4) < (int64_t(1) << 31) && (M <= 4 || (K >= 256 && K < 16384));
  // An output of a few tiles is bound by the latency of its K steps, which
  // are shorter on the float cores (64 x 256: 3 to 9% less time at 256 to
  // 8192 terms, 9 x 256 x 32768 29 us and 35 to 41), except where they cut a
  // ragged one into strips (64 x 1000: a third more).
  const bool small = !rows && cdiv(M, 64) * cdiv(N, 64) < 32 && (M < 64 || M % 64 == 0) &&
                     (N < 64 || N % 64 == 0) && K % BK == 0 && !getenv("TJH_SPLIT_TILE");
  // A^T . B^T and row sums of an A stored [M][K] have no kernel here, and
  // sums of fewer than two K steps nothing to gain: the float cores
  if (small || (transA && transB) || (bias_mode == 3 && !transA) || K < 32) {
    if (act == 1) {  // which keep the pre-activation
      Scratch keep((size_t)(M * N) * sizeof(float));
      if (!keep.ok()) return set_error(TJH_ERR_OOM, "tjh_gemm_split: no scratch");
      return gemm("gemm", transA, transB, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1,
                  bias, bias_mode, keep.as<float>(), N, 1);
    }
    return gemm("gemm", transA, transB, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1,
                bias, bias_mode, const_cast<float*>(residual), ldr, act);
  }
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
  KernelScope ks(rows ? "gemm_rows" : "gemm_split");
  if (rows) return gemm_rows(g, cus);
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
  const int64_t sums = bias_mode == 3 ? 2 * splits * M : 0;
  Scratch ws(splits > 1 ? (size_t)(splits * M * N + sums) * sizeof(float) : 0);
  if (splits > 1 && !ws.ok()) {
    splits = 1;
    g.kchunk = cdiv(K, BK) * BK;
  }
  g.ws = splits > 1 ? ws.as<float>() : nullptr;
  g.rsw = splits > 1 && sums ? g.ws + splits * M * N : nullptr;
  g.rs_pairs = 1;
  // tiles, K steps or loads that need a guard
  const bool edge = M % tc.bm || N % tc.bn || K % BK || !g.vecA || !g.vecB;
  launch_tile(plan.tile, g, dim3((unsigned)(g.tiles_m * g.tiles_n), (unsigned)splits), transA,
              transB, edge);
  const int rc = check_launch("gemm_split");
  if (rc != TJH_OK || splits == 1) return rc;
  return gemm_splitk_sum(g, splits, 1, cus);
}
