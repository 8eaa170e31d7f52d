// Products of blocks of split rows with exact Q4_K weights (kernels/block_split.hip).
#pragma once

#include "../common.h"

namespace esp {

struct BlockSplitForm { int tm = 0, nw = 0, per = 0, splits = 0; float us = 0.0f; };   // tm 0: none
BlockSplitForm block_split_form(const GemmSplitParams &p);
// Complete in p.y (+ residual) or p.swiglu where f.splits is 1, planes of sums in p.workspace otherwise.
hipError_t launch_block_split(const GemmSplitParams &p, const BlockSplitForm &f, hipStream_t stream);
void block_split_set_form(int form);   // 0 by size (default), -1 never, otherwise always: row tiles * 100 + wavefronts along the weights * 10 + shares of K

}  // namespace esp
