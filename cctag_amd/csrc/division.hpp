// Divisions of the sampling kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace cctagx {

// u / w and v / w, each correctly rounded, for w and quotients away from the
// ends of the float range: the reciprocal refined by one Newton step, a
// quotient and two remainder corrections (Markstein, IBM J. Res. Dev. 1990),
// which is the division's own sequence without its scaling of extreme
// operands, and with the reciprocal shared.
__device__ __forceinline__ void div2_rn(float u, float v, float w, float& x, float& y) {
  float r = __builtin_amdgcn_rcpf(w);
  r = __builtin_fmaf(__builtin_fmaf(-w, r, 1.f), r, r);
  float q = u * r;
  q = __builtin_fmaf(__builtin_fmaf(-w, q, u), r, q);
  x = __builtin_fmaf(__builtin_fmaf(-w, q, u), r, q);
  q = v * r;
  q = __builtin_fmaf(__builtin_fmaf(-w, q, v), r, q);
  y = __builtin_fmaf(__builtin_fmaf(-w, q, v), r, q);
}

}  // namespace cctagx
