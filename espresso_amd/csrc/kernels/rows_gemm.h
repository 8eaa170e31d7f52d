// Small products in one launch (kernels/rows_gemm.hip).
#pragma once

#include "../common.h"

namespace esp {

constexpr int kExactRows = 512;   // products that need not round packed weights (GemmParams::unrounded) are exact or not by their rows up to here, and as here beyond
bool rows_gemm_takes(const GemmParams &p);
// p.rows rows; y (+ residual), or swiglu_out for a matrix of (gate, up) row pairs.  The workspace is not used.
hipError_t launch_rows_gemm(const GemmParams &p, hipStream_t stream);
void rows_gemm_set_mode(int mode);   // 0 never, 1 where it is the faster form (default), 2 wherever it can (tests, measurements)
bool rows_gemm_by_size();

}  // namespace esp
