// Steps of a batch of up to sixteen sequences with Q4_K matrices (kernels/batch_gemv.hip).
#pragma once

#include "../common.h"

namespace esp {

struct BatchGemvForm { int blocks = 0, shares = 0, waves = 0; float us = 0.0f; };   // row blocks of a workgroup (0: none), shares of K, wavefronts
// p.sixteen_rows: every epilogue but the arg-max; shares of K only with p.workspace and p.deferred_splits, which receives their number (planes [shares][batch][rows])
BatchGemvForm batch_gemv_form(const GemvParams &p);
hipError_t launch_batch_gemv(const GemvParams &p, const BatchGemvForm &f, hipStream_t stream);
void batch_gemv_set_form(int form);   // 0 by size (default), otherwise that one where it can be: row blocks of a workgroup * 10 + shares of K

}  // namespace esp
