// A pre-LayerNorm transformer block without gradients in one call: the
// launches of nn.LayerNorm, the qkv projection, the key / value cache,
// F.scaled_dot_product_attention, the output projection and the MLP
// (src/nn/layernorm.ts:25-119, linear.ts:43-66, functional.ts:866-890), in
// that order on the library stream, with the values those calls give one by
// one.  A decoding step is eight launches of a few microseconds a block;
// issued from Python they took 225 us of host time a block.
#include "common.h"

namespace tjh {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// Copies the keys and values of qkv [B, T, 3C] to positions [pos, pos + T)
// of the caches [B, H, L, hd], 16 bytes a lane; bound by latency at one
// token and by the 4 BTC floats moved at a prompt.
__global__ __launch_bounds__(256) void k_kv_append(const float* __restrict__ qkv,
                                                   float* __restrict__ kc, float* __restrict__ vc,
                                                   int64_t n4, int T, int C4, int hd4, int64_t L,
                                                   int64_t pos) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const int64_t row = i / C4;  // b * T + t
  const int c = (int)(i - row * C4), h = c / hd4, d = c - h * hd4;
  const int64_t b = row / T, t = row - b * T;
  const floatx4* s = reinterpret_cast<const floatx4*>(qkv) + row * 3 * C4 + c;
  const int64_t to = ((b * (C4 / hd4) + h) * L + pos + t) * hd4 + d;
  reinterpret_cast<floatx4*>(kc)[to] = s[C4];
  reinterpret_cast<floatx4*>(vc)[to] = s[2 * C4];
}

}  // namespace
}  // namespace tjh

using namespace tjh;

/* y = x1 + MLP(LN2(x1)), x1 = x + proj(attention(qkv(LN1(x)))) for x, y
 * [B, T, C], contiguous.  w: ln1 weight, bias, qkv weight, bias, proj weight,
 * bias, ln2 weight, bias, fc weight, bias, fc2 weight, bias (weights [out,
 * in]; norm and bias pointers may be NULL).  kc, vc: caches [B, heads, L, C /
 * heads] that get positions [pos, pos + T) (NULL: none, pos 0).  At pos 0
 * attention is causal over the T positions, else T is 1 and the query sees
 * all of [0, pos].  C / heads is a multiple of 4 and every pointer 16-byte
 * aligned.  For the Python host; not part of the library's declared
 * interface. */
extern "C" int tjh_block_infer(const float* x, float* y, const float* const* w, int64_t B,
                               int64_t T, int64_t C, int64_t heads, int64_t hidden, float eps1,
                               float eps2, float scale, float* kc, float* vc, int64_t L,
                               int64_t pos) {
  TJH_REQUIRE_INIT();
  TJH_ARG(x && y && w && (!kc == !vc), "tjh_block_infer: NULL operand");
  TJH_ARG(B > 0 && T > 0 && C > 0 && heads > 0 && hidden > 0 && C % heads == 0 &&
              (C / heads) % 4 == 0 && hidden % 4 == 0 && T < (1 << 30) && C < (1 << 30),
          "tjh_block_infer: bad sizes");
  TJH_ARG(pos >= 0 && (pos == 0 || T == 1) && (kc ? pos + T <= L : pos == 0),
          "tjh_block_infer: bad position");
  for (int i = 2; i < 12; i += i == 4 ? 4 : 2)
    TJH_ARG(w[i], "tjh_block_infer: NULL weight %d", i);
  TJH_ARG(aligned16(x) && aligned16(y) && aligned16(kc) && aligned16(vc),
          "tjh_block_infer: unaligned operand");
  const int64_t rows = B * T, hd = C / heads;
  // qkv is dead when the hidden layer is formed
  const int64_t wide = hidden > 3 * C ? hidden : 3 * C;
  const auto pad = [](int64_t n) { return cdiv(n, 64) * 64; };
  Scratch s((size_t)(2 * pad(rows * C) + pad(rows * wide) + 2 * pad(rows)) * sizeof(float));
  if (!s.ok()) return set_error(TJH_ERR_OOM, "tjh_block_infer: no scratch");
  float* h = s.as<float>();
  float* x1 = h + pad(rows * C);
  float* a = x1 + pad(rows * C);
  float* mean = a + pad(rows * wide);
  float* rstd = mean + pad(rows);
  const auto linear = [&](const float* in, int64_t K, int i, float* out, int64_t N,
                          const float* res, int act) {
    return tjh_gemm_split(0, 1, rows, N, K, 1.f, in, K, w[i], K, 0.f, out, N, w[i + 1],
                          w[i + 1] ? 1 : 0, res, res ? N : 0, act);
  };
  int rc = tjh_layer_norm_forward(x, w[0], w[1], h, mean, rstd, rows, C, eps1);
  if (rc == TJH_OK) rc = linear(h, C, 2, a, 3 * C, nullptr, 0);
  if (rc != TJH_OK) return rc;
  if (kc) {
    KernelScope ks("copy");
    const int64_t n4 = rows * C / 4;
    TJH_ARG(cdiv(n4, 256) < (int64_t(1) << 31), "tjh_block_infer: too many rows");
    tjh_launch(k_kv_append, dim3((unsigned)cdiv(n4, 256)), dim3(256), 0, stream(),
               (const float*)a, kc, vc, n4, (int)T, (int)(C / 4), (int)(hd / 4), L, pos);
    if ((rc = check_launch("kv_append")) != TJH_OK) return rc;
  }
  const int64_t qs[3] = {T * 3 * C, hd, 3 * C}, os[3] = {T * C, hd, C};
  const int64_t cs[3] = {heads * L * hd, L * hd, hd};
  rc = tjh_sdpa_forward(a, kc ? kc : a + C, vc ? vc : a + 2 * C, h, nullptr, B, heads, T, pos + T, hd,
                        qs, kc ? cs : qs, kc ? cs : qs, os, scale, pos == 0);
  if (rc == TJH_OK) rc = linear(h, C, 4, x1, C, x, 3);
  if (rc == TJH_OK) rc = tjh_layer_norm_forward(x1, w[6], w[7], h, mean, rstd, rows, C, eps2);
  if (rc == TJH_OK) rc = linear(h, C, 8, a, hidden, nullptr, 1);
  if (rc == TJH_OK) rc = linear(a, hidden, 10, y, C, x1, 3);
  return rc;
}
