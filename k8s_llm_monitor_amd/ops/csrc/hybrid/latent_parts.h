// What latent attention's parts of a row's window leave for their merge (latent_attn.hip, latent_heads.hip).
#pragma once
#include "hy_common.h"

namespace k8sllm {

// n[t]: the parts of row t; of more than one, part z's unnormed output [R] and (largest base-2 logit, denominator) of head h are at
// (z * rows + t) * heads + h; what one part has is finished in ``out`` [rows][heads][R].  Rows of fewer than ``least`` tiles are one part.
struct LatentParts {
  float* o;
  float2* ml;
  int* n;
  int least;
};

}  // namespace k8sllm
