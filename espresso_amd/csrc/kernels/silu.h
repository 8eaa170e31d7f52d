// SiLU of a gate in the matrix kernels' epilogues.
#pragma once

#include <hip/hip_runtime.h>

namespace esp {

// g / (1 + e^-g) (the form of Sources/CPUOps/SiLU.swift:5-8): the function that the single-row kernels have as 0.5 g (1 + tanh(0.5 g))
// (RealModelInferenceEngine.swift:6825-6827), in half the instructions and without that form's cancellation at negative gates.  expf and a
// rounded division: within 2^-22 of itself, whatever the gate.
__device__ __forceinline__ float silu(float g) { return g / (1.0f + expf(-g)); }

}  // namespace esp
