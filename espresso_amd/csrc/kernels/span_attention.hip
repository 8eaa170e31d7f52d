// Causal attention of a prompt block on the matrix cores with 32-bit arithmetic, for any number of query heads per key/value head: the
// block form of models whose heads attention_prompt_kernel (decode_ops.hip) is not written for (three or eight query heads per key/value
// head, say), and of short blocks that must be as exact as the single-row steps.
//
// grid (query heads, tiles of 32 rows); a workgroup is KP wavefronts that share the 32 queries (in LDS) and deal the tiles of 32 keys
// among themselves (wavefront p takes tiles p, p + KP, ...).  A wavefront runs by itself from its first tile to its last, without a barrier; the
// KP states (maximum, sum, context) are merged pairwise through LDS at the end.  KP fills the chip where heads x row tiles do not
// (launch_span_attention).
//   * S^T = K Q^T and O^T += V^T P on 32 x 32 tiles: keys are the A rows, queries the B columns, so a lane's 16 accumulators are 16 keys of
//     one query, and its softmax weights are the B operand of the second product as they are.
//   * fp32 caches: v_mfma_f32_32x32x2_f32, fp32 fused multiply-adds throughout.  A lane's 16 bytes of a key row feed four products (the order of k
//     is free as long as both operands agree); values come straight from memory, 32 dims of one key per half wavefront.  Bound by those
//     products: 8192 cycles per tile of 128 dims.
//   * fp16 caches hold keys and values exactly, so only the fp32 operands are split, each into three fp16 parts that add up to its 24 bits: a query scaled
//     by a power of two that takes its largest value to 2^14..2^15, a softmax weight times 2^15 (parts end at 2^-25, so what they leave is below
//     2^-39 of the largest).  Three v_mfma_f32_32x32x16_f16 into one fp32 sum take 96 cycles where the fp32 form takes 512.
// A row whose result is not finite is done again from the keys it sees alone (plain_attention_row).
// 512 rows of 24 heads of 128 (8 key/value heads) behind 1024: 58 us with fp16 caches, 137 with fp32 ones; row by row 780 (fp16).  Pairs of fp16 parts
// (22 bits) in the place of the three took 53 and 98, but were less exact than the row by row kernel.
// Query heads of a key/value head are x, x + kv_heads, ...: with eight key/value heads they share one L2.
#include "../common.h"
#include "attention_rows.h"
#include "span_attention.h"

namespace esp {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// v = p[0] + p[1] + p[2] in element e, for |v| up to 2^15
__device__ __forceinline__ void split3(float v, half8 (&p)[3], int e) {
    p[0][e] = (_Float16)v;
    const float rest = __fsub_rn(v, (float)p[0][e]);
    p[1][e] = (_Float16)rest;
    p[2][e] = (_Float16)__fsub_rn(rest, (float)p[1][e]);
}

// e^x for x <= 0: the hardware's 2^t at the rounded t = x log2(e), times 1 + what the rounding left of it.  Within 2^-22 of e^x for results above 2^-126 (smaller ones are
// 0, and count for nothing beside the largest weight's 1); e^-inf = 0, e^NaN = NaN.  Half of expf's instructions, of which a tile has sixteen a lane.
__device__ __forceinline__ float exp_weight(float x) {
    const float c = x < -128.0f ? -128.0f : x;
    const float log2e = 1.44269504f, t = __fmul_rn(c, log2e), left = __builtin_fmaf(c, 1.92596299e-8f, __builtin_fmaf(c, log2e, -t));
    const float e = __builtin_amdgcn_exp2f(t);
    return __builtin_fmaf(e, __fmul_rn(left, 0.693147181f), e);
}

// Two wavefronts per SIMD where the registers (without copies to accumulator registers) and the LDS of one wavefront allow it: a tile of an fp16 cache is more vector work
// than matrix work, and one wavefront's hides under the other's.
constexpr int span_waves_per_simd(int hd, bool kv_f16, int kp) { return hd == 64 || (kv_f16 && kp > 1) ? 2 : 1; }

template <int HD, bool KV_F16, int KP>
__global__ __launch_bounds__(KP * 64, span_waves_per_simd(HD, KV_F16, KP)) void span_attention_kernel(AttentionArgs a, int rows) {
    constexpr int KS = HD / 16, MT = HD / 32, LDV = 32 + 8, VP = HD / 16;   // VP: 8-dim pieces of an fp16 value tile per lane
    constexpr int LDQ = KV_F16 ? HD + 8 : HD + 4;                           // elements between the queries' rows
    constexpr int kQueryBytes = KV_F16 ? 3 * 32 * LDQ * 2 : 32 * LDQ * 4;
    constexpr int kWave = KV_F16 ? HD * LDV * 2 : 0;                        // a value tile per wavefront
    constexpr int kMergeBytes = KP > 1 ? (KP / 2) * MT * 16 * 64 * 4 : 16;
    __shared__ __attribute__((aligned(16))) unsigned char query_mem[kQueryBytes];
    __shared__ __attribute__((aligned(16))) unsigned char smem[KP * kWave > kMergeBytes ? KP * kWave : kMergeBytes];
    __shared__ int not_finite;
    __shared__ float state[KP][2][64];
    const int lane = threadIdx.x & 63, phase = threadIdx.x >> 6, half = lane >> 5, col = lane & 31;
    const int group = a.n_head / a.n_kv_head, kvh = blockIdx.x % a.n_kv_head, head = kvh * group + blockIdx.x / a.n_kv_head;
    const int y = (int)(gridDim.y - 1 - blockIdx.y);                           // the row tiles with the most keys start first
    asm volatile("" ::"s"(a.tiles), "s"(a.pos), "s"(a.seq), "s"(a.q), "s"(a.k_cache), "s"(a.v_cache));   // fetched together, ahead of the branch
    const int2 tile = a.tiles ? a.tiles[y] : int2{32 * y, rows - 1 - 32 * y};
    const int m0 = tile.x, last_row = tile.y < 31 ? tile.y : 31;
    const int pos0 = a.pos[m0], t_max = pos0 + last_row, kd = a.n_kv_head * HD;
    const size_t base = (size_t)a.seq[m0] * a.cache_seq_stride + (size_t)kvh * HD;
    float scale = 1.0f / sqrtf((float)HD);   // fp16 caches: of the scaled queries
    const int qpos = pos0 + col;

    // Keys beyond t_max are clamped to it: in bounds, and masked.  A lane's keys: row `col` of the tile, dims 16 ks + 8 half .. (fp16), 8 j + 4 half .. (fp32)
    constexpr int NK = KV_F16 ? KS : HD / 8;
    float4 kr[NK];
    auto load_keys = [&](int t0) {
        const size_t kt = base + (size_t)(t0 + col < t_max ? t0 + col : t_max) * kd;
#pragma unroll
        for (int j = 0; j < NK; j++)
            kr[j] = KV_F16 ? *reinterpret_cast<const float4 *>(reinterpret_cast<const uint16_t *>(a.k_cache) + kt + 16 * j + 8 * half)
                           : *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(a.k_cache) + kt + 8 * j + 4 * half);
    };
    // an fp16 value tile on its way to LDS: key = lane % 32, dims 8 (lane / 32 + 2 i) ..: the transposed two-byte writes spread over the banks
    uint4 vr[KV_F16 ? VP : 1];
    auto load_values = [&](int t0) {
        const size_t kt = base + (size_t)(t0 + col < t_max ? t0 + col : t_max) * kd;
#pragma unroll
        for (int i = 0; i < (KV_F16 ? VP : 0); i++) vr[i] = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(a.v_cache) + kt + 8 * (half + 2 * i));
    };
    // The first tile's keys: ahead of the queries from fp32 caches (512 rows behind 1024: 152 -> 137 us), behind them from fp16 ones, whose queries take longer to lay out
    // and then come first (93 rows of 64 dims behind 700: 15.3 us against 16.3).
    if (!KV_F16 && 32 * phase <= t_max) load_keys(32 * phase);

    // query `col` (rows beyond the block repeat its last row, never stored)
    const float *query = a.q + (size_t)(m0 + (col <= last_row ? col : last_row)) * a.n_head * HD + (size_t)head * HD;
    _Float16 *q16 = reinterpret_cast<_Float16 *>(query_mem);                   // [3][32][LDQ]
    float *q32 = reinterpret_cast<float *>(query_mem);                         // [32][LDQ]
    {
        float4 x[KS][2];   // dims 16 ks + 8 half ..
        int q_exp = 0;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int w = 0; w < 2; w++) x[ks][w] = *reinterpret_cast<const float4 *>(query + 16 * ks + 8 * half + 4 * w);
        if constexpr (KV_F16) {
            float most = 0.0f;
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
#pragma unroll
                for (int w = 0; w < 2; w++) most = fmaxf(fmaxf(most, fmaxf(fabsf(x[ks][w].x), fabsf(x[ks][w].y))), fmaxf(fabsf(x[ks][w].z), fabsf(x[ks][w].w)));
            most = fmaxf(most, __shfl_xor(most, 32));
            // where the power of two would not be a float (scores are 0 or beyond every type there), some other will do
            q_exp = 15 - __builtin_amdgcn_frexp_expf(most);
            q_exp = q_exp < -100 ? -100 : q_exp > 100 ? 100 : q_exp;
            scale = __builtin_amdgcn_ldexpf(scale, -q_exp);
        }
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            if (ks % KP != phase) continue;   // the wavefronts share the work; each has read the row for its exponent
            if constexpr (KV_F16) {
                const float v[8] = {x[ks][0].x, x[ks][0].y, x[ks][0].z, x[ks][0].w, x[ks][1].x, x[ks][1].y, x[ks][1].z, x[ks][1].w};
                half8 p[3];
#pragma unroll
                for (int e = 0; e < 8; e++) split3(__builtin_amdgcn_ldexpf(v[e], q_exp), p, e);
#pragma unroll
                for (int i = 0; i < 3; i++) *reinterpret_cast<half8 *>(q16 + (i * 32 + col) * LDQ + 16 * ks + 8 * half) = p[i];
            } else {
#pragma unroll
                for (int w = 0; w < 2; w++) *reinterpret_cast<float4 *>(q32 + col * LDQ + 16 * ks + 8 * half + 4 * w) = x[ks][w];
            }
        }
    }
    __syncthreads();

    // fp32 values of dims 32 mt .. for the product's 16 steps: step r takes key 8 (r / 4) + 4 half + r % 4, the key of accumulator r
    auto load_value_dims = [&](int t0, int mt, float (&v)[16]) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int t = t0 + 8 * (r >> 2) + 4 * half + (r & 3);
            v[r] = reinterpret_cast<const float *>(a.v_cache)[base + (size_t)(t < t_max ? t : t_max) * kd + 32 * mt + col];
        }
    };

    floatx16 o[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[mt][r] = 0.0f;
    float mx = -INFINITY, l = 0.0f;
    _Float16 *vt = reinterpret_cast<_Float16 *>(smem + phase * kWave);

    if (KV_F16 && 32 * phase <= t_max) { load_keys(32 * phase); load_values(32 * phase); }
    for (int t0 = 32 * phase; t0 <= t_max; t0 += 32 * KP) {
        float vd[KV_F16 ? 1 : 2][16];
        if constexpr (!KV_F16) load_value_dims(t0, 0, vd[0]);
        floatx16 s0;
#pragma unroll
        for (int r = 0; r < 16; r++) s0[r] = 0.0f;
        if constexpr (KV_F16) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const half8 k = __builtin_bit_cast(half8, kr[ks]);
                const _Float16 *qp = q16 + col * LDQ + 16 * ks + 8 * half;
#pragma unroll
                for (int p = 2; p >= 0; p--) s0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(k, *reinterpret_cast<const half8 *>(qp + p * 32 * LDQ), s0, 0, 0, 0);
                if (KP == 8 && ks % 2 == 1) __builtin_amdgcn_sched_barrier(0);   // two wavefronts per SIMD: query parts of two steps at a time
            }
            // values of this tile into LDS, transposed; nobody else reads this stretch, and a wavefront's LDS operations keep their order
#pragma unroll
            for (int i = 0; i < VP; i++) {
                const half8 v = __builtin_bit_cast(half8, vr[i]);
#pragma unroll
                for (int e = 0; e < 8; e++) vt[(8 * (half + 2 * i) + e) * LDV + col] = v[e];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            load_keys(t0 + 32 * KP);   // clamped beyond the last tile
            load_values(t0 + 32 * KP);
        } else {
#pragma unroll
            for (int j = 0; j < HD / 8; j++) {
                const float4 q = *reinterpret_cast<const float4 *>(q32 + col * LDQ + 8 * j + 4 * half);
                s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[j].x, q.x, s0, 0, 0, 0);
                s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[j].y, q.y, s0, 0, 0, 0);
                s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[j].z, q.z, s0, 0, 0, 0);
                s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[j].w, q.w, s0, 0, 0, 0);
            }
            load_keys(t0 + 32 * KP);
        }
        // accumulator r: key t0 + 8 (r / 4) + 4 half + r % 4 against query `col`
        float tile_max = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            s0[r] = t0 + 8 * (r >> 2) + 4 * half + (r & 3) <= qpos ? __fmul_rn(s0[r], scale) : -INFINITY;
            tile_max = fmaxf(tile_max, s0[r]);
        }
        tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32));
        // a wavefront may see only masked keys of a query for a while: its state stays (-inf, 0, 0), exponents taken against 0
        const float m_new = fmaxf(mx, tile_max), m_ref = m_new == -INFINITY ? 0.0f : m_new;
        const float alpha = exp_weight(mx - m_ref);      // exp(-inf) = 0 on the first tile
        float psum = 0.0f, pr[16];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            pr[r] = exp_weight(s0[r] - m_ref);           // masked keys: exp(-inf) = 0
            psum += pr[r];
        }
        l = __builtin_fmaf(l, alpha, psum);
        mx = m_new;
        if (!KV_F16 || __any(alpha != 1.0f)) {   // the maximum has moved (beside fp32 products it makes no difference)
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[mt][r] *= alpha;
        }
        if constexpr (KV_F16) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                half8 p[3];
#pragma unroll
                for (int i = 0; i < 8; i++) split3(__fmul_rn(pr[8 * j + i], 32768.0f), p, i);
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    // k slot (lane / 32, i) is key 16 j + 8 (i / 4) + 4 (lane / 32) + i % 4, the key of accumulator 8 j + i
                    const _Float16 *vrow = vt + (32 * mt + col) * LDV + 16 * j + 4 * half;
                    const half4 lo = *reinterpret_cast<const half4 *>(vrow), hi = *reinterpret_cast<const half4 *>(vrow + 8);
                    const half8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
                    for (int i = 2; i >= 0; i--) o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, p[i], o[mt], 0, 0, 0);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        } else {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                if (mt + 1 < MT) load_value_dims(t0, mt + 1, vd[(mt + 1) & 1]);
#pragma unroll
                for (int r = 0; r < 16; r++) o[mt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vd[mt & 1][r], pr[r], o[mt], 0, 0, 0);
            }
        }
    }
    l += __shfl_xor(l, 32);
    // the upper half of the wavefronts hands its states to the lower half, until wavefront 0 holds the sum of all
    float *merge = reinterpret_cast<float *>(smem);
#pragma unroll
    for (int s = KP / 2; s >= 1; s >>= 1) {
        __syncthreads();
        if (phase >= s && phase < 2 * s) {
            state[phase][0][lane] = mx;
            state[phase][1][lane] = l;
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int r = 0; r < 16; r++) merge[(((phase - s) * MT + mt) * 16 + r) * 64 + lane] = o[mt][r];
        }
        __syncthreads();
        if (phase < s) {
            const float m1 = state[phase + s][0][lane], l1 = state[phase + s][1][lane];
            const float m_all = fmaxf(mx, m1), m_ref = m_all == -INFINITY ? 0.0f : m_all;
            const float f0 = exp_weight(mx - m_ref), f1 = exp_weight(m1 - m_ref);
            l = __builtin_fmaf(l, f0, __fmul_rn(l1, f1));
            mx = m_all;
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[mt][r] = __builtin_fmaf(o[mt][r], f0, __fmul_rn(merge[((phase * MT + mt) * 16 + r) * 64 + lane], f1));
        }
    }
    if (phase == 0) {
        float check = 0.0f;
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int r = 0; r < 16; r++) check = __builtin_fmaf(o[mt][r], 0.0f, check);
        const bool odd = __any(!(check == 0.0f && l < INFINITY));   // NaN wherever an infinity or a NaN went in
        if (lane == 0) not_finite = odd;
        if (!odd) {
            const float inv = 1.0f / (KV_F16 ? __fmul_rn(l, 32768.0f) : l);   // key 0 is visible to every query: l > 0
            const size_t row = (size_t)(m0 + (col <= last_row ? col : last_row));
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                float s = 0.0f;
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) {
                    const float v[4] = {__fmul_rn(o[mt][4 * q4], inv), __fmul_rn(o[mt][4 * q4 + 1], inv), __fmul_rn(o[mt][4 * q4 + 2], inv), __fmul_rn(o[mt][4 * q4 + 3], inv)};
                    if (col <= last_row) s += store_context4(a, row * a.n_head * HD + (size_t)head * HD + 32 * mt + 8 * q4 + 4 * half, v);
                }
                if (a.ctx_hi) {
                    s += __shfl_xor(s, 32);
                    if (half == 0 && col <= last_row) store_context_sum(a, row, a.n_head * HD, head * (HD / 32) + mt, s);
                }
            }
        }
    }
    __syncthreads();
    if (not_finite)
        for (int i = phase; i <= last_row; i += KP) plain_attention_row<HD, KV_F16>(a, m0 + i, head);
}

template <int HD, bool KV_F16>
void launch_shape(const AttentionArgs &a, int rows, int sets, hipStream_t s) {
    const dim3 grid(a.n_head, a.tiles ? a.tile_count : (rows + 31) / 32);
    if (sets == 1) hipLaunchKernelGGL((span_attention_kernel<HD, KV_F16, 1>), grid, dim3(64), 0, s, a, rows);
    else if (sets == 2) hipLaunchKernelGGL((span_attention_kernel<HD, KV_F16, 2>), grid, dim3(128), 0, s, a, rows);
    else if (sets == 4) hipLaunchKernelGGL((span_attention_kernel<HD, KV_F16, 4>), grid, dim3(256), 0, s, a, rows);
    else hipLaunchKernelGGL((span_attention_kernel<HD, KV_F16, 8>), grid, dim3(512), 0, s, a, rows);
}

}  // namespace

bool span_attention_supported(int n_head, int n_kv_head, int head_dim) {
    return n_kv_head > 0 && n_head % n_kv_head == 0 && (head_dim == 64 || head_dim == 128);
}

hipError_t launch_span_attention(const AttentionArgs &a, int rows, int keys, bool kv_f16, hipStream_t s) {
    if (rows <= 0 || (a.tiles && a.tile_count <= 0) || !span_attention_supported(a.n_head, a.n_kv_head, a.head_dim)) return hipErrorInvalidValue;
    if (a.ctx_hi ? !a.ctx_lo || !a.ctx_sums || (a.n_head * a.head_dim) % 256 != 0 : !a.ctx_f16) return hipErrorInvalidValue;
    // Wavefronts per workgroup, fp32 caches: as many as it takes to give every SIMD one (256 compute units x 4), each with a tile of keys at least.
    // fp16 caches: four, whose value tiles leave room for a second workgroup on the compute unit; two where a few tiles of keys are over before four have met (128 dims: below ten), and for 128 dims
    // where three workgroups of two fill the chip; eight where a workgroup of 64 dims has the compute unit to itself and keys for all of them.  One wavefront / two / four / eight, us: 1777 rows of 24 heads
    // of 128 136 / 109 / 112 / 152, 800 of them 63 / 39 / 36 / 53, 160 16.5 / 12.4 / 13.2 / 14.9, 31 rows behind 500 42 / 23 / 19 / 21.5;  512 rows of 32 heads of 64 behind 1024 71 / 53 / 35 / 42, 93 of
    // them behind 1500 69 / 38 / 24.3 / 22.6, 1200 60 / 46 / 42 / 64.  (One set a SIMD, the rule before, was up to 1.5 times as slow: 1777 rows of 12 heads of 64 54 us, four sets 37.)
    const int tiles = (keys + 31) / 32, groups = a.n_head * (a.tiles ? a.tile_count : (rows + 31) / 32);
    int sets = 1;
    if (!kv_f16) {
        while (sets < 8 && groups * sets < 1024 && sets * 2 <= tiles) sets *= 2;
    } else if (a.head_dim == 128) {
        sets = tiles < 2 ? 1 : tiles < 10 || groups > 3 * (device_compute_units() > 0 ? device_compute_units() : 256) ? 2 : 4;
    } else {
        sets = tiles < 2 ? 1 : tiles < 3 ? 2 : tiles >= 24 && groups <= (device_compute_units() > 0 ? device_compute_units() : 256) ? 8 : 4;
    }
    if (a.head_dim == 128) {
        if (kv_f16) launch_shape<128, true>(a, rows, sets, s);
        else launch_shape<128, false>(a, rows, sets, s);
    } else {
        if (kv_f16) launch_shape<64, true>(a, rows, sets, s);
        else launch_shape<64, false>(a, rows, sets, s);
    }
    return hipGetLastError();
}

}  // namespace esp
