// GLU activations shared by the kernels that apply them.
#pragma once

#include "common.h"
#include "spiral_ggml.h"

namespace spiral {
namespace {

// act(a) * b for the ggml GLU variants (ids as in include/spiral_ggml.h):
// REGLU relu, GEGLU gelu (tanh form), SWIGLU silu, GEGLU_ERF gelu (erf form),
// GEGLU_QUICK x * sigmoid(1.702 x).
__device__ __forceinline__ float glu_act(int op, float a) {
  switch (op) {
    case SPIRAL_GLU_REGLU: return a > 0.0f ? a : 0.0f;
    case SPIRAL_GLU_GEGLU: {
      const float u = 0.7978845608028654f * a * (1.0f + 0.044715f * a * a);  // sqrt(2/pi) (a + 0.044715 a^3)
      return 0.5f * a * (1.0f + tanhf(u));
    }
    case SPIRAL_GLU_SWIGLU: return a / (1.0f + expf(-a));
    case SPIRAL_GLU_GEGLU_ERF: return 0.5f * a * (1.0f + erff(a * 0.7071067811865476f));
    default: return a / (1.0f + expf(-1.702f * a));  // SPIRAL_GLU_GEGLU_QUICK
  }
}

}  // namespace
}  // namespace spiral
