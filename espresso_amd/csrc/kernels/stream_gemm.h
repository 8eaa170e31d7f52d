// Small products of up to 32 activation rows, weights exact (kernels/stream_gemm.hip).
#pragma once

#include "../common.h"

namespace esp {

// Products that rows_gemm.hip or the exact form of block_gemm.hip would take otherwise.
bool stream_gemm_takes(const GemmParams &p);
// Complete in p.y (+ residual) or p.swiglu_out where *splits is 1; otherwise *splits planes of sums in p.workspace, the residual left to whoever adds them.
hipError_t launch_stream_gemm(const GemmParams &p, int *splits, hipStream_t stream);
void stream_gemm_set_mode(int mode);   // 0 never, 1 by size (default), 2 wherever it can

}  // namespace esp
