// Choice of a token's experts from its logits: moe.hip (a kernel of its own) and rms_residual.hip
// (behind the residual step of a few rows).
#pragma once
#include "common.h"

namespace omnia {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float4v mfma16(short8 a, short8 b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Router for any score function: logits z[e] = x . router[e] (+ bias[e]) stay in fp32;
// weights are sigmoid(z) or softmax(z), renormalised over the chosen ones if asked.  The k
// largest choice scores are chosen: z, or with a correction score + correction (weights stay
// the plain scores); with groups, experts outside the `keep` groups of E / groups neighbours
// with the largest choice score are out of the choice.  Lower numbers win ties.
constexpr int kMaxExperts = 256;
constexpr float kRenormEps = 1e-20f;

struct Route {
  int* ids;    // [T, k]
  float* wts;  // [T, k]
  const float* corr;
  const float* bias;  // [E] added to the logits, or null
  int E, k, sigmoid, renorm, groups, keep;
};

// One token by LPT lanes (l of them), NPL experts a lane; its E logits lie in the LDS row
// zc, which ends as the choice scores.  Every expert counts the experts ahead of it: its
// rank is its slot.
template <int LPT, int NPL>
__device__ __forceinline__ void choose(float* zc, int l, int64_t t, const Route& a) {
  auto sync = [] {  // LDS of one wave
    __builtin_amdgcn_wave_barrier();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  float z[NPL], s[NPL], c[NPL], top = -INFINITY;
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    const int e = l + LPT * i;
    z[i] = e < a.E ? zc[e] + (a.bias ? a.bias[e] : 0.f) : -INFINITY;
    if (!(z[i] == z[i])) z[i] = -INFINITY;  // NaN rows (padding) still get distinct valid ids
    top = fmaxf(top, z[i]);
  }
  if (a.sigmoid) {
#pragma unroll
    for (int i = 0; i < NPL; ++i) s[i] = 1.f / (1.f + expf(-z[i]));
  } else {
#pragma unroll
    for (int o = LPT / 2; o > 0; o >>= 1) top = fmaxf(top, __shfl_xor(top, o, 64));
    if (!(top > -INFINITY)) top = 0.f;
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      s[i] = expf(z[i] - top);
      total += s[i];
    }
#pragma unroll
    for (int o = LPT / 2; o > 0; o >>= 1) total += __shfl_xor(total, o, 64);
    if (!(total > 0.f)) total = 1.f;
#pragma unroll
    for (int i = 0; i < NPL; ++i) s[i] /= total;
  }
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    const int e = l + LPT * i;
    c[i] = a.corr && e < a.E ? s[i] + a.corr[e] : z[i];
    if (e < a.E) zc[e] = c[i];
  }
  sync();
  if (a.groups > 1) {
    const int per = a.E / a.groups;
    int better[NPL], grp[NPL];
    float own[NPL];
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      grp[i] = min((l + LPT * i) / per, a.groups - 1);
      better[i] = 0;
      own[i] = -INFINITY;
      for (int j = 0; j < per; ++j) own[i] = fmaxf(own[i], zc[grp[i] * per + j]);
    }
    for (int g = 0; g < a.groups; ++g) {
      float m = -INFINITY;
      for (int j = 0; j < per; ++j) m = fmaxf(m, zc[g * per + j]);
#pragma unroll
      for (int i = 0; i < NPL; ++i) better[i] += m > own[i] || (m == own[i] && g < grp[i]);
    }
    sync();
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      if (better[i] >= a.keep) c[i] = -INFINITY;
      if (l + LPT * i < a.E) zc[l + LPT * i] = c[i];
    }
    sync();
  }
  int rank[NPL];
#pragma unroll
  for (int i = 0; i < NPL; ++i) rank[i] = 0;
  for (int e = 0; e < a.E; ++e) {
    const float v = zc[e];
#pragma unroll
    for (int i = 0; i < NPL; ++i) rank[i] += v > c[i] || (v == c[i] && e < l + LPT * i);
  }
  float sel = 0.f;
#pragma unroll
  for (int i = 0; i < NPL; ++i)
    if (l + LPT * i < a.E && rank[i] < a.k) sel += s[i];
#pragma unroll
  for (int o = LPT / 2; o > 0; o >>= 1) sel += __shfl_xor(sel, o, 64);
#pragma unroll
  for (int i = 0; i < NPL; ++i)
    if (l + LPT * i < a.E && rank[i] < a.k) {
      a.ids[t * a.k + rank[i]] = l + LPT * i;
      a.wts[t * a.k + rank[i]] = a.renorm ? s[i] / (sel + kRenormEps) : s[i];
    }
}

}  // namespace omnia
