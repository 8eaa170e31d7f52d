// SiLU of a gate in the matrix kernels' epilogues.
#pragma once

#include <hip/hip_runtime.h>

namespace esp {

// g / (1 + e^-g) (the form of Sources/CPUOps/SiLU.swift:5-8): the function that the single-row kernels have as 0.5 g (1 + tanh(0.5 g))
// (RealModelInferenceEngine.swift:6825-6827), in a third of the instructions and without that form's cancellation at negative gates.  e^-g is the hardware's 2^t at the
// rounded t = -g log2(e), times 1 + what the rounding left of it; the quotient is the hardware's reciprocal and one Newton step.  Relative error for gates down to -87: exponential
// 2^-23 + 2^-24, sum, quotient and product 2^-24 each; smaller gates come out below 2^-110 of themselves, where every consumer's fp16 numbers hold 0.
__device__ __forceinline__ float silu(float g) {
    const float c = g < -87.0f ? 87.0f : g > 87.0f ? -87.0f : -g;   // a NaN stays one
    const float log2e = 1.44269504f, t = __fmul_rn(c, log2e), left = __builtin_fmaf(c, 1.92596299e-8f, __builtin_fmaf(c, log2e, -t));
    float e = __builtin_amdgcn_exp2f(t);
    e = __builtin_fmaf(e, __fmul_rn(left, 0.693147181f), e);
    const float d = 1.0f + e, r = __builtin_amdgcn_rcpf(d);
    return __fmul_rn(g, __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r));
}

}  // namespace esp
