// Products of many split rows with exact Q4_K weights (kernels/wide_split.hip).
#pragma once

#include "../common.h"

namespace esp {

struct WideSplitForm { int per = 0, splits = 0; float us = 0.0f; int long_tiles = 0; };   // super-blocks of a share of K (0: none), shares, expected time (0: asked for), tiles of 128 rows in front of tiles of 64 (0: all of 128)
WideSplitForm wide_split_form(const GemmSplitParams &p);
// Complete in p.y (+ residual) or p.swiglu where f.splits is 1, planes of sums in p.workspace otherwise.
hipError_t launch_wide_split(const GemmSplitParams &p, const WideSplitForm &f, hipStream_t stream);
void wide_split_set_shares(int shares);   // 0 by size (default), -1 never, otherwise always, with that many shares of K; 100 * tiles: two heights, so many of 128 rows

}  // namespace esp
