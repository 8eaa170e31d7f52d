// Causal attention of a prompt block on the matrix cores with 32-bit arithmetic, for any number of query heads per key/value head: every block of models with fp16 caches, and with 32-bit caches the
// blocks of head groups that attention_prompt_kernel (decode_ops.hip) is not written for and short blocks that must be as exact as the single-row steps.
//
// grid (query heads, tiles of 32 rows); a workgroup is KP wavefronts that share the 32 queries (in LDS) and deal the tiles of 32 keys
// among themselves (wavefront p takes tiles p, p + KP, ...).  A wavefront runs by itself from its first tile to its last, without a barrier; the
// KP states (maximum, sum, context) meet in LDS at the end, where each wavefront finishes a share of the dims.  KP fills the chip where heads x row tiles do not
// (launch_span_attention).
//   * S^T = K Q^T and O^T += V^T P on 32 x 32 tiles: keys are the A rows, queries the B columns, so a lane's 16 accumulators are 16 keys of
//     one query, and its softmax weights are the B operand of the second product as they are.
//   * fp32 caches: v_mfma_f32_32x32x2_f32, fp32 fused multiply-adds throughout.  A lane's 16 bytes of a key row feed four products (the order of k
//     is free as long as both operands agree); values come straight from memory, 32 dims of one key per half wavefront.  Bound by those
//     products: 8192 cycles per tile of 128 dims.
//   * fp16 caches hold keys and values exactly, so only the fp32 operands are split, each into three fp16 parts that add up to its 24 bits: a query scaled
//     by a power of two that takes its largest value to 2^14..2^15, a softmax weight times 2^15 (parts end at 2^-24, so what they leave is below
//     2^-38 of the largest).  Three v_mfma_f32_32x32x16_f16 take 96 cycles where the fp32 form takes 512.  Values go through LDS as rows, whose transposed reads
//     (ds_read_b64_tr_b16) are the A operand.
//     Every product rounds its sum, so the smaller parts of a score and of a tile's context are added up before the first ones, and a tile's context goes into the row's in one addition.  Root mean square
//     error against 64 bits relative to the context, scores of 1 / 4 / 16 / 60, parts in turn into one sum for all tiles -> this: 300 rows of 8 heads (2 key/value heads) of 128 behind 200
//     2.4 / 5.3 / 9.1 / 17.2e-7 -> 1.8 / 3.9 / 6.5 / 12.4e-7, 93 rows of 12 heads (4) of 64 behind 1500 2.3 / 4.9 / 8.3 / 16.5e-7 -> 1.7 / 3.6 / 6.3 / 12.1e-7.  Pairs of parts with rounded differences instead
//     of exponents of differences, this kernel's forerunner: 2.3 / 5.3 / 9.3 / 17.4e-7 and 2.1 / 4.6 / 7.8 / 15.3e-7.  A correction term of the exponential changes less than 2 % of it.
// A row whose result is not finite is done again from the keys it sees alone (plain_attention_row).
// What bounds it (fp16 caches, 128 dims, a tile): 48 products, 0.78 us of a SIMD at the 2 GHz that the chip holds with all of them at work, beside 200 vector instructions: 1.5 us with two wavefronts a
// SIMD; and a workgroup's way in and out.  Transposed two-byte writes of values, exponentials with a correction term, parts by rounding conversions, every wavefront reading every
// query for its exponent and states handed on pairwise took: 512 rows of 24 heads (8 key/value heads) 21.6 -> 15.4 us, 93 rows of 32 heads of 64 behind 700 15.0 -> 9.4.  Against
// attention_prompt_kernel with fp16 operands (and with pairs of them, inside a model), 32 heads, 8 key/value heads: 128 dims, 64 / 512 rows 10.4 / 20.8 (38) -> 6.9 / 16.7, 512 behind
// 3000 95 -> 92 with two parts; 64 dims, 128 rows 8.0 -> 5.4; slower alone for few heads that share nothing and few rows (33 rows of 12 heads of 64 4.0 -> 4.7): that kernel has 32-bit caches alone.
// 512 rows of 24 heads of 128 behind 1024 from fp32 caches: 136 us.
// Query heads of a key/value head are x, x + kv_heads, ...: with eight key/value heads they share one L2.
#include "../common.h"
#include "attention_rows.h"
#include "span_attention.h"
#include "span_rows.h"
#include <atomic>
#include <type_traits>

namespace esp {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2 __attribute__((ext_vector_type(2)));
typedef short short4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// Two numbers of up to 2^15 as fp16 parts, elements e, e + 1 of p: three, each cut off towards 0, add up to their 24 bits; two rounded ones leave 2^-23 of a number.
template <int PARTS>
__device__ __forceinline__ void split(float v0, float v1, half8 (&p)[PARTS], int e) {
    float minus = -1.0f;
    asm("" : "+v"(minus));   // v - part as one v_fma_mix: a conversion and a subtraction otherwise
#pragma unroll
    for (int i = 0; i < PARTS; i++) {
        const half2 part = PARTS == 3 ? __builtin_bit_cast(half2, __builtin_amdgcn_cvt_pkrtz(v0, v1)) : half2{(_Float16)v0, (_Float16)v1};
        p[i][e] = part[0];
        p[i][e + 1] = part[1];
        if (i == PARTS - 1) break;
        v0 = __builtin_fmaf((float)part[0], minus, v0);
        v1 = __builtin_fmaf((float)part[1], minus, v1);
    }
}

__device__ __forceinline__ half4 read_transposed(const _Float16 *p) {
    return __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4 *)p));
}

// the larger of what the two halves of a wavefront hold
__device__ __forceinline__ float max_of_halves(float v) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, v);
    const auto p = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
    const uint32_t lower = p[0], upper = p[1];
    return fmaxf(__builtin_bit_cast(float, lower), __builtin_bit_cast(float, upper));
}

// the largest of 16 or 32 neighbouring lanes
template <int LANES>
__device__ __forceinline__ float row_max(float v) {
    static_assert(LANES == 16 || LANES == 32, "rows of the wavefront");
    auto from = [](float x, auto control) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(control)::value, 0xF, 0xF, false)); };
    v = fmaxf(v, from(v, std::integral_constant<int, 0xB1>{}));    // quad_perm [1,0,3,2]
    v = fmaxf(v, from(v, std::integral_constant<int, 0x4E>{}));    // quad_perm [2,3,0,1]
    v = fmaxf(v, from(v, std::integral_constant<int, 0x141>{}));   // row_half_mirror
    v = fmaxf(v, from(v, std::integral_constant<int, 0x128>{}));   // row_ror:8
    if constexpr (LANES == 32) {
        const uint32_t bits = __builtin_bit_cast(uint32_t, v);
        const auto p = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
        const uint32_t even = p[0], odd = p[1];
        v = fmaxf(__builtin_bit_cast(float, even), __builtin_bit_cast(float, odd));
    }
    return v;
}

// e^x for x <= 0: the hardware's 2^t at the rounded t = x log2(e), times 1 + what the rounding left of it.  Within 2^-22 of e^x for results above 2^-126 (smaller ones are
// 0, and count for nothing beside the largest weight's 1); e^-inf = 0, e^NaN = NaN.  Half of expf's instructions, of which a tile has sixteen a lane.
__device__ __forceinline__ float exp_weight(float x) {
    const float c = x < -128.0f ? -128.0f : x;
    const float log2e = 1.44269504f, t = __fmul_rn(c, log2e), left = __builtin_fmaf(c, 1.92596299e-8f, __builtin_fmaf(c, log2e, -t));
    const float e = __builtin_amdgcn_exp2f(t);
    return __builtin_fmaf(e, __fmul_rn(left, 0.693147181f), e);
}

// The lane, found again where it is used: three registers more through the loop over the keys are a spill.
__device__ __forceinline__ int lane_again() {
    uint32_t zero = 0;
    asm volatile("" : "+v"(zero));
    return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero));
}

// Two wavefronts per SIMD where the registers (without copies to accumulator registers) and the LDS of one wavefront allow it: a tile of an fp16 cache is more vector work
// than matrix work, and one wavefront's hides under the other's.
constexpr int span_waves_per_simd(int hd, bool kv_f16, int kp) { return hd == 64 || (kv_f16 && kp > 1) ? 2 : 1; }

// PARTS: of the 32-bit operands that meet fp16 caches
template <int HD, bool KV_F16, int KP, int PARTS = 3>
__global__ __launch_bounds__(KP * 64, span_waves_per_simd(HD, KV_F16, KP)) void span_attention_kernel(AttentionArgs a, int rows) {
    constexpr int KS = HD / 16, MT = HD / 32, LDV = HD + 16, VP = HD / 16;   // VP: 8-dim pieces of an fp16 value tile per lane; LDV: four keys' dims fall on all banks
    constexpr int LDQ = KV_F16 ? HD + 8 : HD + 4;                           // elements between the queries' rows
    constexpr int kQueryBytes = KV_F16 ? PARTS * 32 * LDQ * 2 : 32 * LDQ * 4;
    constexpr int kWave = KV_F16 ? 32 * LDV * 2 : 0;                        // a value tile per wavefront
    constexpr int OWN = MT * 16 / KP, kMergeBytes = KP > 1 ? KP * KP * OWN * 64 * 4 : 16;   // accumulators that a wavefront finishes
    __shared__ __attribute__((aligned(16))) unsigned char smem[kQueryBytes + KP * kWave > kMergeBytes ? kQueryBytes + KP * kWave : kMergeBytes];
    unsigned char *const query_mem = smem;
    __shared__ int not_finite;
    __shared__ float state[KP][2][64], row_scale[32];
    const int phase = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int lane = threadIdx.x & 63, half = lane >> 5, col = lane & 31;
    const int group = a.n_head / a.n_kv_head, kvh = blockIdx.x % a.n_kv_head, head = kvh * group + blockIdx.x / a.n_kv_head;
    const int y = (int)(gridDim.y - 1 - blockIdx.y);                           // the row tiles with the most keys start first
    asm volatile("" ::"s"(a.tiles), "s"(a.pos), "s"(a.seq), "s"(a.q), "s"(a.k_cache), "s"(a.v_cache));   // fetched together, ahead of the branch
    const int2 tile = a.tiles ? a.tiles[y] : int2{32 * y, rows - 1 - 32 * y};
    const int m0 = tile.x, last_row = tile.y < 31 ? tile.y : 31;
    const int pos0 = __builtin_amdgcn_readfirstlane(a.pos[m0]), t_max = pos0 + last_row, kd = a.n_kv_head * HD;
    const size_t base = (size_t)__builtin_amdgcn_readfirstlane(a.seq[m0]) * a.cache_seq_stride + (size_t)kvh * HD;
    const int qpos = pos0 + col;

    // Keys beyond t_max are clamped to it: in bounds, and masked.
    // fp32 keys: row `col` of the tile, dims 8 j + 4 half ..
    float4 kr32[KV_F16 ? 1 : HD / 8];
    auto load_keys32 = [&](int t0) {
        const size_t kt = base + (size_t)(t0 + col < t_max ? t0 + col : t_max) * kd;
#pragma unroll
        for (int j = 0; j < HD / 8; j++) kr32[j] = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(a.k_cache) + kt + 8 * j + 4 * half);
    };
    // fp16 keys: row `col`, dims 16 ks + 8 half ..; values on their way to LDS, whole rows by neighbouring lanes.  The tile's first row is uniform, so a lane adds 32-bit offsets alone.
    constexpr int VL = HD / 8, VR = 64 / VL;   // lanes of a row, rows of a load
    uintx4 kr[KV_F16 ? KS : 1], vr[KV_F16 ? VP : 1];
    const uint32_t row_bytes = (uint32_t)kd * 2, k_row = (uint32_t)col * row_bytes, v_row = (uint32_t)(lane / VL) * row_bytes;
    auto first_row = [&](const void *cache, int t0) { return reinterpret_cast<const uint8_t *>(cache) + (base + (size_t)(t0 < t_max ? t0 : t_max) * kd) * 2; };
    auto last_offset = [&](int t0) { return last_row_offset(t_max - t0, row_bytes); };
    auto load_keys = [&](int t0) __attribute__((always_inline)) {
        const uint8_t *from = first_row(a.k_cache, t0);
        const uint32_t most = last_offset(t0), at = (k_row < most ? k_row : most) + 16 * half;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) kr[ks] = *reinterpret_cast<const uintx4 *>(from + at + 32 * ks);
    };
    auto load_values = [&](int t0) __attribute__((always_inline)) {
        const uint8_t *from = first_row(a.v_cache, t0);
        const uint32_t most = last_offset(t0);
#pragma unroll
        for (int i = 0; i < VP; i++) {
            const uint32_t row = v_row + i * VR * row_bytes;
            vr[i] = *reinterpret_cast<const uintx4 *>(from + ((row < most ? row : most) + 16 * (lane % VL)));
        }
    };
    // The first tile of fp32 keys ahead of the queries (512 rows behind 1024: 152 -> 137 us).
    if (!KV_F16 && 32 * phase <= t_max) load_keys32(32 * phase);

    // the queries (rows beyond the block repeat its last row, never stored)
    const size_t q_pitch = (size_t)a.n_head * HD;
    const float *queries = a.q + (size_t)m0 * q_pitch + (size_t)head * HD;
    _Float16 *q16 = reinterpret_cast<_Float16 *>(query_mem);                   // [PARTS][32][LDQ]
    float *q32 = reinterpret_cast<float *>(query_mem);                         // [32][LDQ]
    if constexpr (KV_F16) {   // whole rows by neighbouring lanes, 32 / KP of them a wavefront
        constexpr int QL = HD / 4, QR = 64 / QL, PASSES = 32 / KP / QR;   // lanes of a row, rows of a load
        float4 x[PASSES];
#pragma unroll
        for (int i = 0; i < PASSES; i++) {
            const int r = phase * (32 / KP) + i * QR + lane / QL;
            x[i] = *reinterpret_cast<const float4 *>(queries + (size_t)(r <= last_row ? r : last_row) * q_pitch + 4 * (lane % QL));
        }
        if (32 * phase <= t_max) { load_keys(32 * phase); load_values(32 * phase); }
#pragma unroll
        for (int i = 0; i < PASSES; i++) {
            const int r = phase * (32 / KP) + i * QR + lane / QL;
            const float most = row_max<QL>(fmaxf(fmaxf(fabsf(x[i].x), fabsf(x[i].y)), fmaxf(fabsf(x[i].z), fabsf(x[i].w))));
            // never below -113; where the power of two would not be a float (queries of 2^-86 and less: their scores are 0), some other will do
            const int wanted = 15 - __builtin_amdgcn_frexp_expf(most), q_exp = wanted > 100 ? 100 : wanted;
            half8 p[PARTS];
            split(__builtin_amdgcn_ldexpf(x[i].x, q_exp), __builtin_amdgcn_ldexpf(x[i].y, q_exp), p, 0);
            split(__builtin_amdgcn_ldexpf(x[i].z, q_exp), __builtin_amdgcn_ldexpf(x[i].w, q_exp), p, 2);
#pragma unroll
            for (int k = 0; k < PARTS; k++) *reinterpret_cast<half4 *>(q16 + (k * 32 + r) * LDQ + 4 * (lane % QL)) = half4{p[k][0], p[k][1], p[k][2], p[k][3]};
            if (lane % QL == 0) row_scale[r] = __builtin_amdgcn_ldexpf(__fmul_rn(1.0f / sqrtf((float)HD), 1.44269504f), -q_exp);
        }
    } else {
        // the wavefronts share the dims, 16 in turn; all of a wavefront's loads are on their way before the first store waits (33 rows of 24 heads of 128 dims, two wavefronts: 12.1 us, 11.9 so)
        const float *query = queries + (size_t)(col <= last_row ? col : last_row) * q_pitch;
        constexpr int QS = (KS + KP - 1) / KP;
        float4 x[QS][2];
#pragma unroll
        for (int i = 0; i < QS; i++)
#pragma unroll
            for (int w = 0; w < 2; w++) x[i][w] = *reinterpret_cast<const float4 *>(query + 16 * (KS % KP == 0 || phase < KS ? i * KP + phase : 0) + 8 * half + 4 * w);
        if (KS % KP == 0 || phase < KS)
#pragma unroll
            for (int i = 0; i < QS; i++)
#pragma unroll
                for (int w = 0; w < 2; w++) *reinterpret_cast<float4 *>(q32 + col * LDQ + 16 * (i * KP + phase) + 8 * half + 4 * w) = x[i][w];
    }
    if (threadIdx.x == 0) not_finite = 0;
    __syncthreads();
    // fp16 caches: of the scaled query, in powers of two
    const float scale = KV_F16 ? row_scale[col] : 1.0f / sqrtf((float)HD);
    auto weight_of = [&](float above) { return KV_F16 ? __builtin_amdgcn_exp2f(__fmul_rn(above, scale)) : exp_weight(above); };

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
    _Float16 *vt = reinterpret_cast<_Float16 *>(smem + kQueryBytes + phase * kWave);

    if constexpr (KV_F16) {
        for (int t0 = 32 * phase; t0 <= t_max; t0 += 32 * KP) {
            floatx16 s;
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = 0.0f;
            // The smaller parts of all queries first: their sums are small, and so is what rounds them.  Parts are read three products ahead.
            half8 qf[4];
            constexpr int SMALLER = KS * (PARTS - 1), ALL = KS * PARTS;
            auto dims_of = [](int i) { return i < SMALLER ? i / (PARTS - 1) : i - SMALLER; };   // product i: of sixteen dims, with this part of the queries
            auto read_part = [&](int i) __attribute__((always_inline)) {
                const int part = i < SMALLER ? PARTS - 1 - i % (PARTS - 1) : 0;
                qf[i & 3] = *reinterpret_cast<const half8 *>(q16 + (part * 32 + col) * LDQ + 16 * dims_of(i) + 8 * half);
            };
#pragma unroll
            for (int i = 0; i < 3; i++) read_part(i);
#pragma unroll
            for (int i = 0; i < ALL; i++) {
                if (i + 3 < ALL) read_part(i + 3);
                s = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, kr[dims_of(i)]), qf[i & 3], s, 0, 0, 0);
                if (i % 3 == 2) __builtin_amdgcn_sched_barrier(0);
            }
            // values of this tile into LDS; nobody else reads this stretch, and a wavefront's LDS operations keep their order
#pragma unroll
            for (int i = 0; i < VP; i++) *reinterpret_cast<uintx4 *>(vt + (i * VR + lane / VL) * LDV + 8 * (lane % VL)) = vr[i];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            load_keys(t0 + 32 * KP);   // clamped beyond the last tile
            load_values(t0 + 32 * KP);
            // Accumulator r: key t0 + 8 (r / 4) + 4 half + r % 4 against query `col`.  Scores stay as they are summed: a weight is 2^((s - m) c) with c = scale log2(e), a subtraction, a product and
            // the hardware's 2^t.
            if (t0 + 31 > pos0) {
                const int first = t0 + 4 * (lane_again() >> 5);
#pragma unroll
                for (int r = 0; r < 16; r++) s[r] = first + 8 * (r >> 2) + (r & 3) <= qpos ? s[r] : -INFINITY;
            }
            float tile_max = s[0];
#pragma unroll
            for (int r = 1; r < 16; r++) tile_max = fmaxf(tile_max, s[r]);
            // a wavefront may see only masked keys of a query for a while: its state stays (-inf, 0, 0), exponents taken against 0
            const float m_new = fmaxf(mx, max_of_halves(tile_max)), m_ref = m_new == -INFINITY ? 0.0f : m_new;
            const float alpha = weight_of(mx - m_ref);       // 2^-inf = 0 on the first tile
            mx = m_new;
            // A operand of the second product, k slot (lane / 32, i): key 16 j + 8 (i / 4) + 4 (lane / 32) + i % 4 of dim 32 mt + col, the key of accumulator 8 j + i
            // (ds_read_tr: of sixteen lanes, lane 4 k + c names four dims of key k; lane i receives dim i of all four keys)
            auto read_value = [&](int j, int mt) __attribute__((always_inline)) {
                const _Float16 *vrow = vt + (16 * j + 4 * half + ((lane & 15) >> 2)) * LDV + 32 * mt + (lane & 16) + 4 * (lane & 3);
                const half4 lo = read_transposed(vrow), hi = read_transposed(vrow + 8 * LDV);
                return half8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            };
            half8 v[2][MT], p[2][PARTS];
            float psum = 0.0f;
#pragma unroll
            for (int mt = 0; mt < MT; mt++) v[0][mt] = read_value(0, mt);
            auto weights = [&](int j) __attribute__((always_inline)) {
                float w[8];
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    w[i] = weight_of(s[8 * j + i] - m_ref);   // masked keys: 2^-inf = 0
                    psum += w[i];
                }
#pragma unroll
                for (int i = 0; i < 8; i += 2) split(__fmul_rn(w[i], 32768.0f), __fmul_rn(w[i + 1], 32768.0f), p[j], i);
            };
            weights(0);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) v[1][mt] = read_value(1, mt);
            weights(1);
            l = __builtin_fmaf(l, alpha, psum);
            // A tile's context by itself, the smaller parts of the weights first; then one addition, which takes the maximum's move along
#pragma unroll
            for (int mt = 0; mt < MT; mt += 2) {
                floatx16 t[2];
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int r = 0; r < 16; r++) t[u][r] = 0.0f;
#pragma unroll
                for (int i = PARTS - 1; i >= 0; i--)
#pragma unroll
                    for (int j = 0; j < 2; j++)
#pragma unroll
                        for (int u = 0; u < 2; u++) t[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[j][mt + u], p[j][i], t[u], 0, 0, 0);
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int r = 0; r < 16; r++) o[mt + u][r] = __builtin_fmaf(o[mt + u][r], alpha, t[u][r]);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    } else {
        for (int t0 = 32 * phase; t0 <= t_max; t0 += 32 * KP) {
            float vd[2][16];
            load_value_dims(t0, 0, vd[0]);
            floatx16 s0;
#pragma unroll
            for (int r = 0; r < 16; r++) s0[r] = 0.0f;
#pragma unroll
            for (int j = 0; j < HD / 8; j++) {
                const float4 q = *reinterpret_cast<const float4 *>(q32 + col * LDQ + 8 * j + 4 * half);
                s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr32[j].x, q.x, s0, 0, 0, 0);
                s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr32[j].y, q.y, s0, 0, 0, 0);
                s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr32[j].z, q.z, s0, 0, 0, 0);
                s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr32[j].w, q.w, s0, 0, 0, 0);
            }
            load_keys32(t0 + 32 * KP);
            // accumulator r: key t0 + 8 (r / 4) + 4 half + r % 4 against query `col`
            float tile_max = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                s0[r] = t0 + 8 * (r >> 2) + 4 * half + (r & 3) <= qpos ? __fmul_rn(s0[r], scale) : -INFINITY;
                tile_max = fmaxf(tile_max, s0[r]);
            }
            tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32));
            const float m_new = fmaxf(mx, tile_max), m_ref = m_new == -INFINITY ? 0.0f : m_new;
            const float alpha = weight_of(mx - m_ref);      // exp(-inf) = 0 on the first tile
            float psum = 0.0f, pr[16];
#pragma unroll
            for (int r = 0; r < 16; r++) {
                pr[r] = weight_of(s0[r] - m_ref);            // masked keys: exp(-inf) = 0
                psum += pr[r];
            }
            l = __builtin_fmaf(l, alpha, psum);
            mx = m_new;
#pragma unroll
            for (int mt = 0; mt < MT; mt++)   // whether the maximum has moved or not: beside fp32 products it makes no difference
#pragma unroll
                for (int r = 0; r < 16; r++) o[mt][r] *= alpha;
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                if (mt + 1 < MT) load_value_dims(t0, mt + 1, vd[(mt + 1) & 1]);
#pragma unroll
                for (int r = 0; r < 16; r++) o[mt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vd[mt & 1][r], pr[r], o[mt], 0, 0, 0);
            }
        }
    }
    if constexpr (KV_F16) { lane = lane_again(); half = lane >> 5; col = lane & 31; }
    // The wavefronts' states meet: each leaves its accumulators in LDS and finishes OWN of everybody's, with factors that take every state to the largest maximum, sums in pairs.
    l += __shfl_xor(l, 32);
    float mine[OWN];
    if constexpr (KP > 1) {
        state[phase][0][lane] = mx;
        state[phase][1][lane] = l;
        __syncthreads();   // and everybody is done with queries and values
        float m_all = mx;
#pragma unroll
        for (int w = 0; w < KP; w++) m_all = fmaxf(m_all, state[w][0][lane]);
        const float m_ref = m_all == -INFINITY ? 0.0f : m_all;
        float f[KP], part[KP];
#pragma unroll
        for (int w = 0; w < KP; w++) { f[w] = weight_of(state[w][0][lane] - m_ref); part[w] = state[w][1][lane]; }
        auto total = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int w = 0; w < KP; w += 2) part[w] = __builtin_fmaf(part[w + 1], f[w + 1], __fmul_rn(part[w], f[w]));
#pragma unroll
            for (int d = 2; d < KP; d *= 2)
#pragma unroll
                for (int w = 0; w < KP; w += 2 * d) part[w] += part[w + d];
            return part[0];
        };
        l = total();
        float *merge = reinterpret_cast<float *>(smem);   // [from][to][OWN][64], a wavefront's own share too: kept apart it was a branch for each accumulator, and a wait for each load (33 rows of
                                                            // 24 heads of 128 7.9 us, 6.4 so; from fp32 caches, two wavefronts, 11.9 and 9.8)
#pragma unroll
        for (int w = 0; w < KP; w++)
#pragma unroll
            for (int r = 0; r < OWN; r++) merge[((phase * KP + w) * OWN + r) * 64 + lane] = o[(w * OWN + r) >> 4][(w * OWN + r) & 15];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < OWN; r++) {
#pragma unroll
            for (int w = 0; w < KP; w++) part[w] = merge[((w * KP + phase) * OWN + r) * 64 + lane];
            mine[r] = total();
        }
    } else {
#pragma unroll
        for (int r = 0; r < OWN; r++) mine[r] = o[r >> 4][r & 15];
    }
    float check = 0.0f;
#pragma unroll
    for (int r = 0; r < OWN; r++) check = __builtin_fmaf(mine[r], 0.0f, check);
    bool finite = !__any(!(check == 0.0f && l < INFINITY));   // NaN wherever an infinity or a NaN went in
    if constexpr (KP > 1) {
        if (!finite && lane == 0) not_finite = 1;
        __syncthreads();
        finite = !not_finite;
    }
    if (finite) {
        const float inv = 1.0f / (KV_F16 ? __fmul_rn(l, 32768.0f) : l);   // key 0 is visible to every query: l > 0
        const size_t row = (size_t)(m0 + (col <= last_row ? col : last_row));
        float sums[OWN < 16 ? 1 : OWN / 16];   // of 32 dims each, or of this wavefront's share of them
#pragma unroll
        for (int r = 0; r < OWN; r += 4) {
            const int at = phase * OWN + r;   // accumulator: dims 32 (at / 16) + 8 (at / 4 % 4) + 4 half ..
            const float v[4] = {__fmul_rn(mine[r], inv), __fmul_rn(mine[r + 1], inv), __fmul_rn(mine[r + 2], inv), __fmul_rn(mine[r + 3], inv)};
            float s = 0.0f;
            if (col <= last_row) s = store_context4(a, row * q_pitch + (size_t)head * HD + 32 * (at >> 4) + 8 * ((at >> 2) & 3) + 4 * half, v);
            sums[r >> 4] = r % 16 == 0 ? s : sums[r >> 4] + s;
        }
        if (a.ctx_hi) {
            constexpr int SHARERS = OWN < 16 ? 16 / OWN : 1;   // wavefronts that share 32 dims
            float *parts = reinterpret_cast<float *>(smem);  // [SHARERS][32 queries] of every 32 dims; the merge is behind everybody
            if constexpr (SHARERS > 1) {
                const float s = sums[0] + __shfl_xor(sums[0], 32);
                if (half == 0) parts[phase * 32 + col] = s;
                __syncthreads();
            }
#pragma unroll
            for (int i = 0; i < (OWN < 16 ? 1 : OWN / 16); i++) {
                float s = 0.0f;
                if constexpr (SHARERS > 1) {
#pragma unroll
                    for (int w = 0; w < SHARERS; w++) s += parts[(phase / SHARERS * SHARERS + w) * 32 + col];
                } else s = sums[i] + __shfl_xor(sums[i], 32);
                if (phase % SHARERS == 0 && half == 0 && col <= last_row) store_context_sum(a, row, a.n_head * HD, head * (HD / 32) + (phase * OWN >> 4) + i, s);
            }
        }
        return;
    }
    for (int i = phase; i <= last_row; i += KP) plain_attention_row<HD, KV_F16>(a, m0 + i, head);
}

template <int HD, bool KV_F16>
void launch_shape(const AttentionArgs &a, int rows, int sets, bool pairs, hipStream_t s) {
    const dim3 grid(a.n_head, a.tiles ? a.tile_count : (rows + 31) / 32);
    auto go = [&](auto waves) {
        constexpr int KP = decltype(waves)::value;
        hipLaunchKernelGGL((span_attention_kernel<HD, KV_F16, KP>), grid, dim3(64 * KP), 0, s, a, rows);
    };
    if constexpr (HD == 128 && KV_F16)
        if (pairs) {
            hipLaunchKernelGGL((span_attention_kernel<HD, KV_F16, 4, 2>), grid, dim3(256), 0, s, a, rows);
            return;
        }
    if constexpr (!KV_F16) {
        if (sets == 1) return go(std::integral_constant<int, 1>{});
        if (sets == 2) return go(std::integral_constant<int, 2>{});
    }
    if (sets == 4) go(std::integral_constant<int, 4>{});
    else go(std::integral_constant<int, 8>{});
}

std::atomic<int> g_key_sets{0};

}  // namespace

void attention_prompt_set_key_sets(int sets) { g_key_sets.store(sets == 1 || sets == 2 ? sets : 0); }

bool span_attention_supported(int n_head, int n_kv_head, int head_dim) {
    return n_kv_head > 0 && n_head % n_kv_head == 0 && (head_dim == 64 || head_dim == 128);
}

hipError_t launch_span_attention(const AttentionArgs &a, int rows, int keys, bool kv_f16, hipStream_t s, bool pairs_do) {
    if (rows <= 0 || (a.tiles && a.tile_count <= 0) || !span_attention_supported(a.n_head, a.n_kv_head, a.head_dim)) return hipErrorInvalidValue;
    if (a.ctx_hi ? !a.ctx_lo || !a.ctx_sums || (a.n_head * a.head_dim) % 256 != 0 : !a.ctx_f16) return hipErrorInvalidValue;
    // Wavefronts per workgroup, fp32 caches: as many as it takes to give every SIMD one (256 compute units x 4), each with a tile of keys at least.
    // fp16 caches: four, whose value tiles leave room for a second workgroup on the compute unit, or eight where a workgroup has the compute unit to itself and keys for all of them.  Four / eight, us:
    // 512 rows of 24 heads of 128 15.3 / 18.6, 64 rows 6.8 / 7.0, 93 rows behind 500 / 800 / 1000 14.9 / 13.3, 17.9 / 15.7, 20.8 / 17.8, 31 rows behind 300 / 500 / 4000 (32 heads) 10.9 / 10.5, 14.3 / 12.9, 52 / 45;
    // heads of 64: 512 rows of 32 heads 9.7 / 13.0, 128 rows 5.3 / 5.6, 93 rows behind 300 / 500 / 700 / 1500 8.0 / 7.7, 9.0 / 8.2, 10.7 / 9.4, 16.4 / 13.3, 512 rows behind 1024 23.9 / 26.6.  Under 24 tiles of keys the sums of four stay, as they were when eight were no faster there.
    // One or two where there are no more tiles of keys than that: the same bits, and slower, since the queries are split by all wavefronts (16 rows 4.5 -> 4.9, of 24 heads of 128 6.1 -> 7.8; 64 rows 6.8 -> 7.1).
    const int tiles = (keys + 31) / 32, groups = a.n_head * (a.tiles ? a.tile_count : (rows + 31) / 32), cus = device_compute_units() > 0 ? device_compute_units() : 256;
    int sets = 1;
    if (!kv_f16) {
        while (sets < 8 && groups * sets < 1024 && sets * 2 <= tiles) sets *= 2;
    } else {
        const int forced = g_key_sets.load();
        sets = forced ? 4 * forced : tiles >= 24 && groups <= cus ? 8 : 4;
    }
    // Long walks over the keys are bound by the products (48 of a tile of 128 dims with three parts, 32 with two), and a context that is rounded to fp16 shows neither.  512 rows of 32 heads (8 key/value heads)
    // behind 1500 / 2000 / 3000 / 6000 / 15000, fp16 operands / three parts / two, us: 58 / 56 / 54, 71 / 73 / 67, 95 / 100 / 92, 168 / 180 / 164, 382 / 402 / 367.  Up to 2048 keys three parts are no slower
    // than fp16 operands were; nor are they where the workgroups are eight wavefronts (93 rows behind 3000 77 / 37) or heads are 64 dims (512 behind 8000 220 / 127).
    const bool pairs = pairs_do && kv_f16 && a.head_dim == 128 && !a.ctx_hi && sets == 4 && keys > 2048;
    if (a.head_dim == 128) {
        if (kv_f16) launch_shape<128, true>(a, rows, sets, pairs, s);
        else launch_shape<128, false>(a, rows, sets, false, s);
    } else {
        if (kv_f16) launch_shape<64, true>(a, rows, sets, false, s);
        else launch_shape<64, false>(a, rows, sets, false, s);
    }
    return hipGetLastError();
}

}  // namespace esp
