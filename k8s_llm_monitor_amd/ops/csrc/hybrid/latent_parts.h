// What latent attention's parts of a row's window leave for their merge (latent_attn.hip, latent_heads.hip).
#pragma once
#include "hy_common.h"

namespace k8sllm {

// part z, row t, head h at (z * rows + t) * heads + h: the unnormed output [R] and (largest base-2 logit, denominator); (-inf, 0): an
// empty part, whose output is not written
struct LatentParts {
  float* o;
  float2* ml;
};

}  // namespace k8sllm
