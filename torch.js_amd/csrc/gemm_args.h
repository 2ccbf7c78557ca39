// What the GEMM kernels of gemm.hip (float products) and gemm_split.h (split
// products) share: their arguments, the order of the tiles, the activation
// epilogue and the sum of split-K partials.
#pragma once

#include "common.h"
#include "ops_math.h"

namespace tjh {

constexpr int BK = 16;

typedef float floatx16 __attribute__((ext_vector_type(16)));
// Staging registers are native 4-wide vectors: a struct float4 copied out
// of a reinterpret_cast load is not always split into registers by the
// compiler and then lives in scratch memory.
typedef float floatx4 __attribute__((ext_vector_type(4)));
// The same vector at 4-byte alignment: operand rows start wherever the row
// stride puts them.
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

struct GemmArgs {
  const float* A;
  const float* B;
  float* C;
  const float* bias;
  int64_t M, N, K;
  int64_t lda, ldb, ldc;
  int64_t sA, sB, sC;
  float alpha, beta;
  int bias_mode;
  int vecA, vecB;  // 128-bit loads allowed for the operand
  int tiles_m, tiles_n;
  int64_t kchunk;  // K range per split (multiple of BK); splits = gridDim.y
  float* ws;       // split-K partials [batch][split][M][N] (nullptr: none)
  float* rsw;      // split-K partials of the row sums (bias_mode 3/4) [split][M]
  int rs_pairs;    // 1: rsw is [split][2][M], each sum and what it rounds off
  // epilogue activation on the final C values (after alpha, beta, bias):
  // 1: aux (if any) <- v, C <- GELU(v);  2: C <- v * GELU'(aux);  3: C <- aux + v
  float* aux;
  int64_t ldaux;
  int act;
  // A formed on load from logits (k_gemm<..., XF>): A's element at logits
  // row r, class c is (exp(logits[r][c] - lse_r) - (c == t_r)) * s_r, the
  // cross-entropy gradient, with xrow[r] = {lse_r, s_r, t_r (int bits), 0};
  // xm0 / xk0 locate this (sub-)product in the logits (rows = m without
  // TA, k with TA)
  const floatx4* xrow;
  int64_t xm0, xk0;
};

// A compile-time int carried by a value (dispatch into generic lambdas).
template <int V>
struct IConst {
  static constexpr int value = V;
};

// Workgroups are dispatched to the 8 XCDs round-robin (workgroup w runs on
// XCD w % 8), and each XCD has its own L2.  Renumbering so that XCD x
// receives the contiguous run [x*n/8, (x+1)*n/8) of the grouped tile order
// keeps the tiles that share A rows and B columns on one L2.  A bijection on
// [0, n): ids past the last multiple of 8 keep their number.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_tile(int bid, int n) {
  const int full = n - n % kXcds;
  if (bid >= full) return bid;
  return (bid % kXcds) * (full / kXcds) + bid / kXcds;
}

// The activation epilogue, shared by the GEMM and the split-K sum.
__device__ __forceinline__ float epilogue_act(const GemmArgs& g, int64_t row, int64_t col,
                                              float v) {
  if (g.act == 1) {
    if (g.aux) g.aux[row * g.ldaux + col] = v;
    return gelu_f(v);
  }
  if (g.act == 2) return v * gelu_grad(g.aux[row * g.ldaux + col]);
  if (g.act == 3) return g.aux[row * g.ldaux + col] + v;
  return v;
}

// C = alpha * (the sum of `splits` partials in g.ws) + beta C + bias, with
// the activation: the pass that ends a product split over K.
int gemm_splitk_sum(const GemmArgs& g, int64_t splits, int64_t batch, int cus);

}  // namespace tjh
