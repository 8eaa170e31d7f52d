// What the block attention kernels share: the context of a row and head in the forms their consumers read, and the plain way to it.
#pragma once

#include "../common.h"
#include "decode_ops.h"

namespace esp {

// Four consecutive dims (from a multiple of four on) of a context row, fp16 or as split rows (SplitRowsView: the planes' order inside fours is 0, 2, 1,
// 3).  Returns what the planes hold of them, for the sub-block sums.
__device__ __forceinline__ float store_context4(const AttentionArgs &a, size_t at, const float (&v)[4]) {
    typedef _Float16 half4 __attribute__((ext_vector_type(4)));
    if (!a.ctx_hi) {
        *reinterpret_cast<half4 *>(a.ctx_f16 + at) = half4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
        return 0.0f;
    }
    half4 h, l;
    float s = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        h[e] = (_Float16)v[e];
        l[e] = (_Float16)__fmul_rn(__fsub_rn(v[e], (float)h[e]), 2048.0f);
        s += __builtin_fmaf((float)l[e], 1.0f / 2048.0f, (float)h[e]);
    }
    *reinterpret_cast<half4 *>(a.ctx_hi + at) = half4{h[0], h[2], h[1], h[3]};
    *reinterpret_cast<half4 *>(a.ctx_lo + at) = half4{l[0], l[2], l[1], l[3]};
    return s;
}
// the sum of sub-block `sub` (32 columns) of a row
__device__ __forceinline__ void store_context_sum(const AttentionArgs &a, size_t row, int cols, int sub, float s) {
    uint16_t *p = a.ctx_sums + (row * (size_t)(cols / 256) + (sub >> 3)) * 16 + (sub & 7);
    const _Float16 h = (_Float16)s;
    p[0] = __builtin_bit_cast(uint16_t, h);
    p[8] = __builtin_bit_cast(uint16_t, (_Float16)__fmul_rn(__fsub_rn(s, (float)h), 2048.0f));
}

// One row and query head by one wavefront, in fp32 and from the keys the row sees alone.  The matrix-core kernels come here with rows whose result is not
// finite: there a key that is masked still takes part, with weight 0, and 0 times an infinity would make NaN of rows that do not see it; and a part of a
// split operand may be zero, or overflow, where the operand does not.  Rare, so nothing here is fast.
template <int HD, bool KV_F16>
__device__ void plain_attention_row(const AttentionArgs &a, int row, int head) {
    const int lane = __lane_id(), kvh = head / (a.n_head / a.n_kv_head), kd = a.n_kv_head * HD;
    const size_t base = (size_t)a.seq[row] * a.cache_seq_stride + (size_t)kvh * HD;
    const float *q = a.q + (size_t)row * a.n_head * HD + (size_t)head * HD;
    const float scale = 1.0f / sqrtf((float)HD);
    // A query that is not finite has no score that is, so its context is NaN whatever the keys: no key at all, and 0 / 0.  Once a model's hidden state is NaN every row of
    // every layer comes here, and this loop would take a hundred times the block's own time.
    float check = 0.0f;
#pragma unroll
    for (int i = 0; i < HD / 64; i++) check = __builtin_fmaf(q[64 * i + lane], 0.0f, check);
    const int visible = __any(!(check == 0.0f)) ? 0 : a.pos[row] + 1;
    auto cached = [&](const void *cache, size_t at) {
        return KV_F16 ? (float)reinterpret_cast<const _Float16 *>(cache)[at] : reinterpret_cast<const float *>(cache)[at];
    };
    auto score = [&](int t) {
        float s = 0.0f;
#pragma unroll 1
        for (int d = 0; d < HD; d++) s = __builtin_fmaf(q[d], cached(a.k_cache, base + (size_t)t * kd + d), s);
        return __fmul_rn(s, scale);
    };
    float mx = -INFINITY, sum = 0.0f, acc[HD / 64];
#pragma unroll 1
    for (int t = lane; t < visible; t += 64) mx = fmaxf(mx, score(t));
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
#pragma unroll
    for (int i = 0; i < HD / 64; i++) acc[i] = 0.0f;
#pragma unroll 1
    for (int t0 = 0; t0 < visible; t0 += 64) {
        const float p = t0 + lane < visible ? expf(score(t0 + lane) - mx) : 0.0f;
        sum += p;
#pragma unroll 1
        for (int j = 0; j < 64 && t0 + j < visible; j++) {
            const float pj = __shfl(p, j);
#pragma unroll
            for (int i = 0; i < HD / 64; i++) acc[i] = __builtin_fmaf(pj, cached(a.v_cache, base + (size_t)(t0 + j) * kd + 64 * i + lane), acc[i]);
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off);
#pragma unroll
    for (int i = 0; i < HD / 64; i++) {
        const float mine = acc[i] / sum;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = __shfl(mine, (lane & ~3) + e);
        float s = 0.0f;
        if ((lane & 3) == 0) s = store_context4(a, (size_t)row * a.n_head * HD + (size_t)head * HD + 64 * i + lane, v);
        if (a.ctx_hi) {
#pragma unroll
            for (int off = 16; off >= 1; off >>= 1) s += __shfl_xor(s, off);
            if ((lane & 31) == 0) store_context_sum(a, row, a.n_head * HD, head * (HD / 32) + 2 * i + (lane >> 5), s);
        }
    }
}

}  // namespace esp
