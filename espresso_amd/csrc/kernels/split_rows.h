// What the kernels that write split rows (SplitRowsView) share.
#pragma once

#include "../common.h"

namespace esp {
namespace split_rows {

constexpr float kUnscale = 1.0f / 2048.0f, kScale = 2048.0f;
// The sum S of a sub-block (held by the first of each four lanes after the quad reduction) as the pair the GEMM's extra MFMA reads:
// sums[(row, super-block)][j] = fp16(S), [8 + j] = fp16((S - fp16(S)) * 2048).
__device__ __forceinline__ void store_subblock_sum(uint16_t *sums, size_t row, int cols, int group, float s) {
    s += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s), 0xB1, 0xF, 0xF, false));
    s += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s), 0x4E, 0xF, 0xF, false));
    if ((group & 3) == 0) {
        const int sub = group >> 2;   // sub-block of 32 columns
        uint16_t *p = sums + (row * (size_t)(cols / 256) + (sub >> 3)) * 16 + (sub & 7);
        const _Float16 h = (_Float16)s;
        p[0] = __builtin_bit_cast(uint16_t, h);
        p[8] = __builtin_bit_cast(uint16_t, (_Float16)__fmul_rn(__fsub_rn(s, (float)h), kScale));
    }
}

}  // namespace split_rows
}  // namespace esp
