// The splits of single-token attention into one, for whoever reads a (sequence, head)'s result: the kernel that writes it
// (attention_mfma.hip) and the product per head behind attention over a latent (latent.hip).
#pragma once
#include "common.h"

// Number d of a (sequence, head) whose n_splits partial outputs lie at src, [n_splits][D + 2] with maximum and sum behind each.  The splits'
// maxima and sums are a lane each, so that all of them are one trip to memory (a loop over the splits, once for the maximum and once for the
// sums, took 6.2 us for 8 splits of 32 heads, 4.7 this way with 16 splits of 32 heads).  A whole wave comes here with one src; mine: RB_WAVE
// pairs of LDS of its own, so that none waits for another.  sink: the head's, in units of the scores, or null.
// sum_only: the splits' outputs are added as they are (sigmoid weights), without maxima and denominators.
template <int D>
__device__ __forceinline__ float combined_split(const float* __restrict__ src, int n_splits, const float* __restrict__ sink, bool sum_only,
                                                float2* mine, int lane, int d) {
  constexpr int AHEAD = 8;
  constexpr float LOG2_E = 1.4426950408889634f;
  float mx = -INFINITY;
  if (!sum_only) {
    for (int s = lane; s < n_splits; s += RB_WAVE) mx = fmaxf(mx, src[(size_t)s * (D + 2) + D]);
    mx = wave_max(mx);
  }
  const float m_safe = (mx == -INFINITY) ? 0.f : mx;
  float a = 0.f, l = 0.f;
  for (int s0 = 0; s0 < n_splits; s0 += RB_WAVE) {
    const int here = n_splits - s0 < RB_WAVE ? n_splits - s0 : RB_WAVE;
    if (!sum_only && lane < here) {
      const float* of = src + (size_t)(s0 + lane) * (D + 2);
      mine[lane] = make_float2(exp2f(of[D] - m_safe), of[D + 1]);      // this wave's alone; a wave's LDS accesses complete in order
    }
    __builtin_amdgcn_wave_barrier();
    for (int s1 = 0; s1 < here; s1 += AHEAD) {
      float v[AHEAD];
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) v[u] = src[(size_t)(s0 + (s1 + u < here ? s1 + u : s1)) * (D + 2) + d];
#pragma unroll
      for (int u = 0; u < AHEAD; ++u)
        if (s1 + u < here) {                            // in the order of the splits
          if (sum_only) {
            a += v[u];
          } else {
            const float2 f = mine[s1 + u];
            a = fmaf(v[u], f.x, a);
            l = fmaf(f.y, f.x, l);
          }
        }
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (sum_only) return a;
  if (sink) l += exp2f(fmaf(*sink, LOG2_E, -m_safe));          // the sink: in the denominator only
  return l > 0.f ? a / l : 0.f;
}
