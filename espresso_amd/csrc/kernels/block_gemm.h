// Products of blocks of activation rows, fp16 operands (kernels/block_gemm.hip).
#pragma once

#include "../common.h"

namespace esp {

bool block_gemm_takes(const GemmParams &p);
// No caller adds shares of K: their sum is a launch of its own.
inline bool block_gemm_alone(const GemmParams &p) { return !p.deferred_splits && !p.swiglu_out; }
// Exact here rather than in the kernel of rows_gemm.hip?
bool block_gemm_keeps(const GemmParams &p);
bool block_gemm_exact(const GemmParams &p);   // of a product that runs here
// Do products of up to `rows` rows that need not round their weights (GemmParams::unrounded) keep them as they are?
bool block_gemm_exact(const DeviceMatrix &w, int rows);
// Complete in p.y (+ residual) or p.swiglu_out where *splits is 1; otherwise *splits planes of sums in p.workspace, residual and SiLU left to whoever adds them.
hipError_t launch_block_gemm(const GemmParams &p, int *splits, hipStream_t stream);
void block_gemm_set_form(int form);   // 0 by size (default), otherwise always: row tiles * 100 + wavefronts along the weights * 10 + shares of K (+ long tiles * 1000, 64 rows each behind them)
bool block_gemm_by_size();

}  // namespace esp
