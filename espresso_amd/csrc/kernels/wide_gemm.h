// Products of rows of activations with fp16 matrices (kernels/wide_gemm.hip).
#pragma once

#include "../common.h"
#include "wide_form.h"

namespace esp {

WideForm wide_gemm_form(const GemmParams &p);   // no tile: not an fp16 matrix
// Complete in p.y (+ residual) or p.swiglu_out where the form has one share of K; otherwise planes of sums in p.workspace.
hipError_t launch_wide_gemm(const GemmParams &p, const WideForm &form, hipStream_t stream);
void wide_gemm_set_form(int form);   // 0 by size (default), otherwise always, where its planes have room: rows of a tile * 10000 + weight rows * 10 + shares of K

}  // namespace esp
