// A token's experts from its router logits.
#pragma once
#include "hy_common.h"

namespace k8sllm {

constexpr int kMaxE = 256;
constexpr int kMaxK = 16;

// A strict order of logits: NaN first (its weights then show it, as torch's topk does), larger ones, equal ones by number (-0 equals 0)
__device__ __forceinline__ bool goes_before(float a, int ia, float b, int ib) {
  const bool na = a != a, nb = b != b;
  if (na || nb) return na && nb ? ia < ib : na;
  return a > b || (a == b && ia < ib);
}

// One wave ranks a token's logits lg[E] (and lg[E], its gate's), a lane counting what goes before its expert, and writes the choice
__device__ __forceinline__ void router_choose(const float* lg, int* sel, int* ids, float* wts, float* gate, long t, int E, int K, int over_all) {
  const int lane = threadIdx.x & 63;
  for (int e = lane; e < E; e += 64) {
    int rank = 0;
    for (int i = 0; i < E; ++i) rank += goes_before(lg[i], i, lg[e], e);
    if (rank < K) sel[rank] = e;
  }
  __builtin_amdgcn_wave_barrier();  // a wave's LDS instructions execute in issue order
  if (lane < K) {
    float mx = -INFINITY, z = 0.f;
    for (int k = 0; k < K; ++k) mx = fmaxf(mx, lg[sel[k]]);
    if (over_all) {  // the denominator runs over every expert (the first chosen logit is the largest of all)
      for (int e = 0; e < E; ++e) z += expf(lg[e] - mx);
    } else {
      for (int k = 0; k < K; ++k) z += expf(lg[sel[k]] - mx);
    }
    ids[t * K + lane] = sel[lane];
    wts[t * K + lane] = expf(lg[sel[lane]] - mx) / z;
  }
  if (gate != nullptr && lane == 0) gate[t] = 1.f / (1.f + expf(-lg[E]));
}

}  // namespace k8sllm
