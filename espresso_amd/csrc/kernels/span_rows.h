// Rows of a tile of keys as 32-bit offsets from the tile's first row (kernels/span_attention.hip).
#pragma once

#include <stdint.h>

namespace esp {

constexpr int kSpanTile = 32;   // keys

// What a row's offset may be at most: the last key's, which lies `distance` rows behind the tile's first (none if the tile starts behind it).  A tile's own last row is the most that is asked for, so a longer
// distance is cut off before it is multiplied: as bytes it passes 32 bits in a cache of 4 GB a layer (32 key/value heads of 128 dims from 524288 positions on).
constexpr uint32_t last_row_offset(int distance, uint32_t row_bytes) {
    return (uint32_t)(distance < 0 ? 0 : distance < kSpanTile ? distance : kSpanTile - 1) * row_bytes;
}

}  // namespace esp
