// The sums of a block row's stretches put together, for the combining kernels of the fused attention (attn.hip, attn_f32.hip).
#ifndef SCORCH_AMD_ATTN_PARTS_HPP_
#define SCORCH_AMD_ATTN_PARTS_HPP_

#include "common.hpp"

namespace scorch {

typedef float PartsVec __attribute__((ext_vector_type(4)));

// `parts` stretches' (O, m, l) of a query, `base` the first one's and STRIDE floats apart, m at D and l behind it: acc and l the sums relative
// to the largest m, of the four features from `feature` on.  The first AT_ONCE stretches' sums are requested with their maxima, one
// round trip instead of two.
template <int D, int STRIDE, int AT_ONCE>
__device__ __forceinline__ void combine_parts_by(const float *__restrict__ base, int parts, int feature, PartsVec &acc, float &l) {
  // (past the last: the last again; a branch to each puts the waits between them)
  constexpr int kHeld = AT_ONCE > 0 ? AT_ONCE : 1, kBatch = 8;
  PartsVec first_o[kHeld];
  float first_m[kHeld], first_l[kHeld];
#pragma unroll
  for (int p = 0; p < AT_ONCE; ++p) {
    const float *part = base + (size_t)min(p, parts - 1) * STRIDE;
    first_o[p] = *reinterpret_cast<const PartsVec *>(part + feature);
    first_m[p] = part[D];
    first_l[p] = part[D + 1];
  }
  float m_star = -3.0e38f;
#pragma unroll 1
  for (int p = AT_ONCE; p < parts; p += kBatch) {
    float m[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) m[u] = base[(size_t)min(p + u, parts - 1) * STRIDE + D];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) m_star = fmaxf(m_star, m[u]);
  }
#pragma unroll
  for (int p = 0; p < AT_ONCE; ++p) m_star = fmaxf(m_star, first_m[p]);
  acc = PartsVec{0.f, 0.f, 0.f, 0.f};
  l = 0.0f;
  const auto add = [&](float m, float sum, const PartsVec &o) __attribute__((always_inline)) {
    const float weight = __builtin_amdgcn_exp2f(m - m_star);
    l += weight * sum;
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] += weight * o[r];
  };
#pragma unroll
  for (int p = 0; p < AT_ONCE; ++p)
    if (p < parts) add(first_m[p], first_l[p], first_o[p]);
#pragma unroll 1
  for (int p = AT_ONCE; p < parts; p += kBatch) {
    PartsVec o[kBatch];
    float m[kBatch], sum[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const float *part = base + (size_t)min(p + u, parts - 1) * STRIDE;
      o[u] = *reinterpret_cast<const PartsVec *>(part + feature);
      m[u] = part[D];
      sum[u] = part[D + 1];
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
      if (p + u < parts) add(m[u], sum[u], o[u]);
  }
}

// How many at once: reading the last again costs a row of few stretches more than it waits for, and a row of many asks for the rest in
// batches in any case.  Uniform over the workgroup: a row is its own.  Window of 64 and a global token, fp32, D = 64, 4,096 tokens, 4 heads,
// the global token's row in so many stretches, both launches, us, with maxima first and then the sums, loops that the compiler
// unrolls, and so: 2 65.9, 64.7; 4 40.9, 39.5; 6 34.2, 32.0; 8 28.2, 27.4; 16 28.4, 26.9; 32 25.6, 23.4; 64 35.8, 31.0.  (Eight at once
// whatever a row has: (2,048, 16), window of 256, rows of two 74.8 for 73.2; 64 stretches 37.6.  Loops that the compiler unrolls
// for the rest wait for every stretch: 16 29.2, 64 38.7.)
template <int D, int STRIDE>
__device__ __forceinline__ void combine_parts(const float *__restrict__ base, int parts, int feature, PartsVec &acc, float &l) {
  parts = uniform(parts);
  if (parts > 16 || parts <= 0) combine_parts_by<D, STRIDE, 0>(base, parts, feature, acc, l);
  else if (parts > 4) combine_parts_by<D, STRIDE, 8>(base, parts, feature, acc, l);
  else combine_parts_by<D, STRIDE, 4>(base, parts, feature, acc, l);
}

}  // namespace scorch

#endif  // SCORCH_AMD_ATTN_PARTS_HPP_
