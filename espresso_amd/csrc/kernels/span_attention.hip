// Causal attention of a prompt block on the matrix cores for any number of query heads per key/value head, with 32-bit queries, caches
// and softmax weights kept to 22 bits: the block form of models whose heads attention_prompt_kernel (decode_ops.hip) is not written
// for (three or eight query heads per key/value head, say).  Those took the general single-query kernel, in which every row reads its
// whole prefix by itself; per layer, 512 rows of 24 heads of 128 up to position 1535: 782 -> 37 us; 93 rows of 32 heads of 64 behind
// 700 tokens: 123 -> 13.4 us.
//
// grid (query heads, tiles of 32 rows); a workgroup is KP wavefronts that share the 32 queries and deal the tiles of 32 keys among
// themselves (wavefront p takes tiles p, p + KP, ...).  A wavefront runs by itself from its first tile to its last: its value tile is its
// own stretch of LDS, so there is no barrier in the loop; the KP states (maximum, sum, context) are merged pairwise through the same LDS
// at the end.  KP fills the chip where heads x row tiles do not (launch_span_attention).  What bounds it: the chain of a tile (scores,
// maximum, exponentials, transposed values) with one or two wavefronts per SIMD; keys and values come from the L2 a tile ahead.
//   * S^T = K Q^T with v_mfma_f32_32x32x16_f16: keys are the A rows, queries the B columns, so a lane's 16 accumulators are 16 keys of
//     one query.  Queries go in as hi + lo / 2048 (two products), fp32 keys as well (three: hi hi, lo hi, hi lo).
//   * O^T += V^T P: a lane's softmax weights are its B fragment as they are.  They go in times 2^15 as a pair hi + lo at one scale (a
//     weight is at most 1, so nothing overflows and what the pair leaves is below 2^-40), which needs one accumulator; fp32 values as hi + lo.
// Query heads of a key/value head are x, x + kv_heads, ...: with eight key/value heads they share one L2.
#include "../common.h"
#include "span_attention.h"

namespace esp {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr float kMostHalf = 65504.0f;

// v = hi + lo / 2048 (fp16 each); what fp16 cannot hold is cut to its largest value
__device__ __forceinline__ void split8(const float4 &x0, const float4 &x1, half8 &hi, half8 &lo) {
    const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float c = __builtin_amdgcn_fmed3f(v[e], -kMostHalf, kMostHalf);
        hi[e] = (_Float16)c;
        lo[e] = (_Float16)__fmul_rn(__fsub_rn(c, (float)hi[e]), 2048.0f);
    }
}
// the same without a scale on the second part: v = hi + lo to 22 bits or 2^-25, whichever is coarser
__device__ __forceinline__ void split8_plain(const float4 &x0, const float4 &x1, half8 &hi, half8 &lo) {
    const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
    for (int e = 0; e < 8; e++) {
        hi[e] = (_Float16)v[e];
        lo[e] = (_Float16)__fsub_rn(v[e], (float)hi[e]);
    }
}

template <int HD, bool KV_F16, int KP>
__global__ __launch_bounds__(KP * 64) void span_attention_kernel(AttentionArgs a, int rows) {
    constexpr int KS = HD / 16, MT = HD / 32, LDV = 32 + 8, PLANES = KV_F16 ? 1 : 2, VP = HD / 16;   // VP: 8-dim pieces of a value tile per lane
    constexpr int kTile = PLANES * HD * LDV;                                   // fp16 per wavefront
    constexpr int kValueBytes = KP * kTile * 2, kMergeBytes = (KP / 2) * MT * 16 * 64 * 4;
    __shared__ __attribute__((aligned(16))) unsigned char smem[kValueBytes > kMergeBytes ? kValueBytes : kMergeBytes];
    __shared__ float state[KP][2][64];
    const int lane = threadIdx.x & 63, phase = threadIdx.x >> 6, half = lane >> 5, col = lane & 31;
    const int group = a.n_head / a.n_kv_head, kvh = blockIdx.x % a.n_kv_head, head = kvh * group + blockIdx.x / a.n_kv_head;
    const int m0 = (int)(gridDim.y - 1 - blockIdx.y) * 32;                     // the row tiles with the most keys start first
    const int last_row = rows - 1 - m0 < 31 ? rows - 1 - m0 : 31;
    const int pos0 = a.pos[m0], t_max = pos0 + last_row, kd = a.n_kv_head * HD;
    const size_t base = (size_t)a.seq[m0] * a.cache_seq_stride + (size_t)kvh * HD;
    const float scale = 1.0f / sqrtf((float)HD);
    _Float16 *vt = reinterpret_cast<_Float16 *>(smem) + phase * kTile;

    // queries: column = query `col` (rows beyond the block repeat its last row, never stored), dims 16 ks + 8 half ..
    half8 qh[KS], ql[KS];
    {
        const float *qp = a.q + (size_t)(m0 + (col <= last_row ? col : last_row)) * a.n_head * HD + (size_t)head * HD + 8 * half;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) split8(*reinterpret_cast<const float4 *>(qp + 16 * ks), *reinterpret_cast<const float4 *>(qp + 16 * ks + 4), qh[ks], ql[ks]);
    }
    // A tile on its way: fp16 caches 8 values per 128-bit load, fp32 caches two loads.  Keys beyond t_max are clamped to it: in bounds, and masked.
    constexpr int W = KV_F16 ? 1 : 2;
    float4 kr[KS * W], vr[VP * W];
    auto load = [&](int t0) {
        const size_t kt = base + (size_t)(t0 + col < t_max ? t0 + col : t_max) * kd + 8 * half;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int w = 0; w < W; w++)
                kr[ks * W + w] = KV_F16 ? *reinterpret_cast<const float4 *>(reinterpret_cast<const uint16_t *>(a.k_cache) + kt + 16 * ks)
                                        : *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(a.k_cache) + kt + 16 * ks + 4 * w);
        // a value tile's piece: key = lane % 32, dims 8 (lane / 32 + 2 i) ..: the transposed two-byte writes spread over the banks
#pragma unroll
        for (int i = 0; i < VP; i++)
#pragma unroll
            for (int w = 0; w < W; w++) {
                const size_t o = kt - 8 * half + 8 * (half + 2 * i);
                vr[i * W + w] = KV_F16 ? *reinterpret_cast<const float4 *>(reinterpret_cast<const uint16_t *>(a.v_cache) + o)
                                       : *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(a.v_cache) + o + 4 * w);
            }
    };

    floatx16 o[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[mt][r] = 0.0f;
    float mx = -INFINITY, l = 0.0f;
    const int qpos = pos0 + col;
    if (32 * phase <= t_max) load(32 * phase);
    for (int t0 = 32 * phase; t0 <= t_max; t0 += 32 * KP) {
        floatx16 sc, sl;
#pragma unroll
        for (int r = 0; r < 16; r++) sc[r] = sl[r] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            half8 kh, kl;
            if constexpr (KV_F16) kh = __builtin_bit_cast(half8, kr[ks]);
            else split8(kr[2 * ks], kr[2 * ks + 1], kh, kl);
            sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, qh[ks], sc, 0, 0, 0);
            sl = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, ql[ks], sl, 0, 0, 0);
            if constexpr (!KV_F16) sl = __builtin_amdgcn_mfma_f32_32x32x16_f16(kl, qh[ks], sl, 0, 0, 0);
        }
        // values of this tile into LDS, transposed; nobody else reads this stretch, and a wavefront's LDS operations keep their order
#pragma unroll
        for (int i = 0; i < VP; i++) {
            half8 vh, vl;
            if constexpr (KV_F16) vh = __builtin_bit_cast(half8, vr[i]);
            else split8_plain(vr[2 * i], vr[2 * i + 1], vh, vl);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                vt[(8 * (half + 2 * i) + e) * LDV + col] = vh[e];
                if constexpr (!KV_F16) vt[HD * LDV + (8 * (half + 2 * i) + e) * LDV + col] = vl[e];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        load(t0 + 32 * KP);   // clamped beyond the last tile
        // accumulator r: key t0 + 8 (r / 4) + 4 half + r % 4 against query `col`
        float tile_max = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int key = t0 + 8 * (r >> 2) + 4 * half + (r & 3);
            const float s = __builtin_fmaf(sl[r], 1.0f / 2048.0f, sc[r]);
            sc[r] = key <= qpos ? __fmul_rn(s, scale) : -INFINITY;
            tile_max = fmaxf(tile_max, sc[r]);
        }
        tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32));
        // a wavefront may see only masked keys of a query for a while: its state stays (-inf, 0, 0), exponents taken against 0
        const float m_new = fmaxf(mx, tile_max), m_ref = m_new == -INFINITY ? 0.0f : m_new;
        const float alpha = __expf(mx - m_ref);      // exp(-inf) = 0 on the first tile
        float psum = 0.0f;
        half8 ph[2], pl[2];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const float pr = __expf(sc[r] - m_ref);  // masked keys: exp(-inf) = 0
            psum += pr;
            const float big = __fmul_rn(pr, 32768.0f);
            ph[r >> 3][r & 7] = (_Float16)big;
            pl[r >> 3][r & 7] = (_Float16)__fsub_rn(big, (float)ph[r >> 3][r & 7]);
        }
        l = __builtin_fmaf(l, alpha, psum);
        mx = m_new;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
#pragma unroll
            for (int r = 0; r < 16; r++) o[mt][r] *= alpha;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                // k slot (lane / 32, i) is key 16 j + 8 (i / 4) + 4 (lane / 32) + i % 4, the key of accumulator 8 j + i
                const _Float16 *vrow = vt + (32 * mt + col) * LDV + 16 * j + 4 * half;
                const half4 lo = *reinterpret_cast<const half4 *>(vrow), hi = *reinterpret_cast<const half4 *>(vrow + 8);
                const half8 vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, ph[j], o[mt], 0, 0, 0);
                o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pl[j], o[mt], 0, 0, 0);
                if constexpr (!KV_F16) {
                    const half4 lo2 = *reinterpret_cast<const half4 *>(vrow + HD * LDV), hi2 = *reinterpret_cast<const half4 *>(vrow + HD * LDV + 8);
                    const half8 vf2 = {lo2[0], lo2[1], lo2[2], lo2[3], hi2[0], hi2[1], hi2[2], hi2[3]};
                    o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf2, ph[j], o[mt], 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
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
            const float f0 = __expf(mx - m_ref), f1 = __expf(m1 - m_ref);
            l = __builtin_fmaf(l, f0, __fmul_rn(l1, f1));
            mx = m_all;
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[mt][r] = __builtin_fmaf(o[mt][r], f0, __fmul_rn(merge[((phase * MT + mt) * 16 + r) * 64 + lane], f1));
        }
    }
    if (phase == 0 && col <= last_row) {
        const float inv = 1.0f / __fmul_rn(l, 32768.0f);   // key 0 is visible to every query: l > 0
        uint16_t *out = a.ctx_f16 + (size_t)(m0 + col) * a.n_head * HD + (size_t)head * HD;
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int q4 = 0; q4 < 4; q4++)
                *reinterpret_cast<half4 *>(out + 32 * mt + 8 * q4 + 4 * half) = half4{(_Float16)__fmul_rn(o[mt][4 * q4], inv), (_Float16)__fmul_rn(o[mt][4 * q4 + 1], inv),
                                                                                       (_Float16)__fmul_rn(o[mt][4 * q4 + 2], inv), (_Float16)__fmul_rn(o[mt][4 * q4 + 3], inv)};
    }
}

template <int HD, bool KV_F16>
void launch_shape(const AttentionArgs &a, int rows, int sets, hipStream_t s) {
    const dim3 grid(a.n_head, (rows + 31) / 32);
    if (sets == 1) hipLaunchKernelGGL((span_attention_kernel<HD, KV_F16, 1>), grid, dim3(64), 0, s, a, rows);
    else if (sets == 2) hipLaunchKernelGGL((span_attention_kernel<HD, KV_F16, 2>), grid, dim3(128), 0, s, a, rows);
    else if (sets == 4 || (!KV_F16 && HD == 128)) hipLaunchKernelGGL((span_attention_kernel<HD, KV_F16, 4>), grid, dim3(256), 0, s, a, rows);
    else hipLaunchKernelGGL((span_attention_kernel<HD, KV_F16, (!KV_F16 && HD == 128) ? 4 : 8>), grid, dim3(512), 0, s, a, rows);
}

}  // namespace

bool span_attention_supported(int n_head, int n_kv_head, int head_dim) {
    return n_kv_head > 0 && n_head % n_kv_head == 0 && (head_dim == 64 || head_dim == 128);
}

hipError_t launch_span_attention(const AttentionArgs &a, int rows, int keys, bool kv_f16, hipStream_t s) {
    if (rows <= 0 || !a.ctx_f16 || !span_attention_supported(a.n_head, a.n_kv_head, a.head_dim)) return hipErrorInvalidValue;
    // Wavefronts per workgroup: as many as it takes to give every SIMD one (256 compute units x 4), each with a tile of keys at least.
    // A 512-row block of 24 heads gets four (36.9 us), its 241-row rest eight (36.3), 93 rows of 32 heads eight (13.4).
    const int tiles = (keys + 31) / 32, groups = a.n_head * ((rows + 31) / 32);
    int sets = 1;
    while (sets < 8 && groups * sets < 1024 && sets * 2 <= tiles) sets *= 2;
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
