// Attention of one query per head (a cached decoding step): softmax(q K^T
// scale) V with the lse, for the head dims and layouts of flash.hip, behind
// F.scaled_dot_product_attention (src/nn/functional.ts:866-890).
//
// Bound by reading K and V once (360 KB a head at 701 keys x 64, 17 MB over
// 48 heads: 3 us at 6 TB/s), on as many CUs as there are heads.  flash.hip's
// tiles would multiply 127 rows of padding per query and walk the keys in
// one chain of 32 at a time.  Here a workgroup of 16 waves has a head;
// each group of 16 lanes takes every 64th key, four at a time with their
// loads issued together, through an online softmax of its own, and the 64
// groups are merged once at the end in a fixed order.  701 keys x 64, 48
// heads: 12.8 us, bound by the loads that 48 CUs keep in flight (58 us in
// the flash kernel).
#include "common.h"
#include "wave.h"

#include <math.h>

namespace tjh {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int kThreads = 1024, kGroups = kThreads / 16, kUnroll = 4;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

struct OneArgs {
  const float *q, *k, *v;
  float *o, *lse;
  int64_t qb, qh, kb, kh, kt, vb, vh, vt, ob, oh;
  int64_t H, Tk;
  int D;
  float scale;
};

// NC: 64-column pieces of the head dim
template <int NC>
__global__ __launch_bounds__(kThreads) void k_attn_one(OneArgs a) {
  __shared__ float sm[kGroups], sl[kGroups];
  __shared__ float so[kGroups][NC * 64];
  const int64_t b = blockIdx.x / a.H, h = blockIdx.x % a.H;
  const int g = threadIdx.x >> 4, l = threadIdx.x & 15;
  const float* __restrict__ K = a.k + b * a.kb + h * a.kh;
  const float* __restrict__ V = a.v + b * a.vb + h * a.vh;
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  floatx4 q[NC], o[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int d = 64 * c + 4 * l;
    o[c] = zero;
    q[c] = zero;
    if (d < a.D)
      q[c] = *reinterpret_cast<const floatx4*>(a.q + b * a.qb + h * a.qh + d) * (a.scale * kLog2e);
  }
  float m = -INFINITY, sum = 0.f;
  for (int64_t t0 = g; t0 < a.Tk; t0 += kGroups * kUnroll) {
    floatx4 kv[kUnroll][NC], vv[kUnroll][NC];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      // keys past the end repeat the last one with a score of -infinity
      const int64_t t = t0 + u * kGroups < a.Tk ? t0 + u * kGroups : a.Tk - 1;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int d = 64 * c + 4 * l;
        kv[u][c] = d < a.D ? *reinterpret_cast<const floatx4*>(K + t * a.kt + d) : zero;
        vv[u][c] = d < a.D ? *reinterpret_cast<const floatx4*>(V + t * a.vt + d) : zero;
      }
    }
    float s[kUnroll], mn = m;
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      float x = 0.f;
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) x = __builtin_fmaf(q[c][e], kv[u][c][e], x);
      x = row16_sum(x);
      s[u] = t0 + u * kGroups < a.Tk ? x : -INFINITY;
      mn = fmaxf(mn, s[u]);
    }
    const float ms = mn == -INFINITY ? 0.f : mn;
    const float alpha = __builtin_amdgcn_exp2f(m - ms);
    m = mn;
    sum *= alpha;
#pragma unroll
    for (int c = 0; c < NC; ++c) o[c] *= alpha;
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const float p = __builtin_amdgcn_exp2f(s[u] - ms);
      sum += p;
      if (t0 + u * kGroups < a.Tk) {  // 0 x infinity of a repeated key stays out
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) o[c][e] = __builtin_fmaf(p, vv[u][c][e], o[c][e]);
      }
    }
  }
#pragma unroll
  for (int c = 0; c < NC; ++c)
    *reinterpret_cast<floatx4*>(&so[g][64 * c + 4 * l]) = o[c];
  if (l == 0) {
    sm[g] = m;
    sl[g] = sum;
  }
  __syncthreads();
  // column d of a group of D consecutive lanes; the first wave also has the lse
  const int d = threadIdx.x;
  if (d >= NC * 64) return;
  // groups without a key (m = -infinity, sum 0) add exact zeros
  float top = -INFINITY;
  for (int i = 0; i < kGroups; ++i) top = fmaxf(top, sm[i]);
  const float ts = top == -INFINITY ? 0.f : top;
  float den = 0.f, num = 0.f;
#pragma unroll 8
  for (int i = 0; i < kGroups; ++i) {
    const float f = __builtin_amdgcn_exp2f(sm[i] - ts);
    den = __builtin_fmaf(sl[i], f, den);
    num = __builtin_fmaf(so[i][d], f, num);
  }
  const float inv = den > 0.f ? 1.0f / den : 0.f;
  if (d < a.D) a.o[b * a.ob + h * a.oh + d] = num * inv;
  if (d == 0 && a.lse) a.lse[blockIdx.x] = (top + __log2f(den)) * kLn2;
}

}  // namespace

int attn_one_query(const float* q, const float* k, const float* v, float* o, float* lse, int64_t B,
                   int64_t H, int64_t Tk, int64_t D, const int64_t* qs, const int64_t* ks,
                   const int64_t* vs, const int64_t* os, float scale, int causal) {
  TJH_ARG(B * H < (int64_t(1) << 31), "sdpa: grid too large");
  OneArgs a{q,     k,     v,     o,     lse,   qs[0], qs[1], ks[0], ks[1],
            ks[2], vs[0], vs[1], vs[2], os[0], os[1], H,     causal ? 1 : Tk, (int)D, scale};
  KernelScope ks_("sdpa_fwd");
  const dim3 grid((unsigned)(B * H)), block(kThreads);
  if (D <= 64) tjh_launch(k_attn_one<1>, grid, block, 0, stream(), a);
  else tjh_launch(k_attn_one<2>, grid, block, 0, stream(), a);
  return check_launch("attn_one");
}

}  // namespace tjh
