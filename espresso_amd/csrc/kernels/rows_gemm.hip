// y[m][n] = sum_k x[m][k] * W[n][k] for small products (rows_gemm_takes: few activation rows, or many of a small matrix), W in Q4_K, Q4_0,
// Q8_0 or fp16: fp16 activations, weights exact, fp32 sums.
//
// The tile kernel of gemm.hip wants 128 rows of each operand, and its narrow form splits K over workgroups and leaves fp32 planes for
// another launch to add.  A small product is the weights' way from memory plus fixed costs, so here everything stays in one launch: a
// workgroup owns 32 weight rows and up to 32 activation rows, and its wavefronts split K between them (contiguous ranges, so that a 128-byte
// line of a row is used up by one wavefront).  The wavefronts share nothing on the way: weights go from memory into the B operand's registers
// (v_mfma_f32_32x32x16_f16: a lane holds eight k of its own weight row), activations through a stretch of LDS that is the wavefront's
// own, which puts whole 128-byte pieces of rows into the A operand's order; there is no barrier until the wavefronts' sums meet at the end, in wavefront order.
// What bounds it: the trip to memory and the weights' bandwidth; kAhead steps of 64 k are in flight per wavefront.
//   * Integers go to the matrix cores, scales are applied to the sums: Q8_0's bytes and Q4_0's q - 8 per block of 32 (two products),
//     Q4_K's sc q <= 945 per super-block, its minimum as a second chain over the same activations whose B operand is the sub-block's m.
//     No weight is rounded (the tile kernel rounds each one to fp16).
//   * Lane (n = lane % 32, h = lane / 32) loads sixteen bytes of row n at a time.  Which k those are is matched by the activations' addresses:
//     Q8_0, Q4_K: 32 p + 16 h + 8 i; fp16 and (after the two halves of a wavefront exchanged half of two blocks) Q4_0: 32 p + 16 i + 8 h.
#include "../common.h"
#include "block_gemm.h"
#include "wide_gemm.h"
#include "rows_gemm.h"
#include "silu.h"
#include <cstdlib>
#include <type_traits>

namespace esp {
namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32;

constexpr int kStep = 64;      // k per step
constexpr int kWaves = 8;
constexpr int kAhead = 4;      // steps in flight (a whole super-block of Q4_K)

struct RowsArgs {
    const uint8_t *qs;
    const uint16_t *scales;
    size_t row_bytes;
    int N, K, M;
    const uint16_t *x;
    float *y;
    const float *residual;
    uint16_t *act;
};

__device__ __forceinline__ h2 as_h2(u32 v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ u32 as_u32(h2 v) { return __builtin_bit_cast(u32, v); }
__device__ __forceinline__ half8 as_half8(const uint4 &v) { return __builtin_bit_cast(half8, v); }
__device__ __forceinline__ float half_bits_to_float(u32 bits16) { return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16); }
__device__ __forceinline__ h2 splat(float v) { const _Float16 h = (_Float16)v; return h2{h, h}; }
__device__ __forceinline__ u32 dword_of(const uint4 &v, int k) { return k == 0 ? v.x : k == 1 ? v.y : k == 2 ? v.z : v.w; }

// a lane's packed weights of one step of its row
template <int FMT> struct Packed { uint4 q; };                               // Q4_K
template <> struct Packed<FMT_Q4_0> { uint4 q; u32 d; };                     // block p = h of the step's two; both blocks' scales
template <> struct Packed<FMT_Q8_0> { uint4 q[2]; u32 d; };
template <> struct Packed<FMT_F16> { uint4 q[4]; };

// Eight weights of two dwords of nibbles, natural order: nibbles at bits 0..3 read 1024 + q under 0x6400, at bits 4..7 64 + q under 0x5400.
// mul * (offset + q) + add, exact for the integers used here.
__device__ __forceinline__ half8 nibbles(u32 w0, u32 w1, bool high, h2 mul, h2 add) {
    const u32 mask = high ? 0x00F000F0u : 0x000F000Fu, magic = high ? 0x54005400u : 0x64006400u;
    const u32 a = __builtin_amdgcn_perm(w0, w0, 0x03010200u), b = __builtin_amdgcn_perm(w1, w1, 0x03010200u);   // bytes 0 2 1 3: pairs come out adjacent
    return as_half8(make_uint4(as_u32(__builtin_elementwise_fma(as_h2((a & mask) | magic), mul, add)), as_u32(__builtin_elementwise_fma(as_h2(((a >> 8) & mask) | magic), mul, add)),
                               as_u32(__builtin_elementwise_fma(as_h2((b & mask) | magic), mul, add)), as_u32(__builtin_elementwise_fma(as_h2(((b >> 8) & mask) | magic), mul, add))));
}
// eight signed bytes as fp16 integers
__device__ __forceinline__ half8 bytes8(u32 w0, u32 w1) {
    const h2 off = {(_Float16)-1152.0f, (_Float16)-1152.0f};   // 1024 + 128
    const u32 a = w0 ^ 0x80808080u, b = w1 ^ 0x80808080u;
    return as_half8(make_uint4(as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, a, 0x04010400u)) + off), as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, a, 0x04030402u)) + off),
                               as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, b, 0x04010400u)) + off), as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, b, 0x04030402u)) + off)));
}

__device__ __forceinline__ u32 scale_byte(const uint4 &hdr, int idx) {
    const u32 word = idx < 4 ? hdr.y : idx < 8 ? hdr.z : hdr.w;
    return (word >> ((idx & 3) * 8)) & 0xFFu;
}
// ggml's get_scale_min_k4
__device__ __forceinline__ void q4k_scale_min(const uint4 &hdr, int j, u32 &sc, u32 &m) {
    if (j < 4) {
        sc = scale_byte(hdr, j) & 63u;
        m = scale_byte(hdr, j + 4) & 63u;
    } else {
        sc = (scale_byte(hdr, j + 4) & 0xFu) | ((scale_byte(hdr, j - 4) >> 6) << 4);
        m = (scale_byte(hdr, j + 4) >> 4) | ((scale_byte(hdr, j) >> 6) << 4);
    }
}

// NL groups of eight activation rows (1, 2 or 4)
constexpr int kXRow = 72;      // fp16 between staged activation rows: 16-byte reads of 32 rows spread over the banks
constexpr size_t rows_lds_bytes(int nl) {
    const size_t x = (size_t)kWaves * nl * 8 * kXRow * 2, sums = (size_t)kWaves * 16 * 64 * 4;
    return x > sums ? x : sums;
}
static_assert(rows_lds_bytes(4) <= 64 * 1024, "the default limit of dynamic LDS");
template <int FMT, int NL>
__global__ __launch_bounds__(kWaves * 64) void rows_gemm_kernel(RowsArgs a) {
    constexpr bool kBlocks = FMT == FMT_Q4_0 || FMT == FMT_Q8_0, kSuper = FMT == FMT_Q4_K;
    extern __shared__ float red[];             // first [wavefront][8 NL rows][kXRow] fp16, then [wavefront][16][64] sums
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5, col = lane & 31;
    const int n = blockIdx.x * 32 + col, row = n < a.N ? n : a.N - 1;   // clamped, never stored
    const int m0 = blockIdx.y * 32;
    // this wavefront's steps; whole super-blocks of Q4_K
    constexpr int kUnit = kSuper ? 4 : 1;
    const int units = a.K / (kStep * kUnit), per = (units + kWaves - 1) / kWaves;
    const int s_begin = (wave * per < units ? wave * per : units) * kUnit, s_end = ((wave + 1) * per < units ? (wave + 1) * per : units) * kUnit;

    const uint8_t *wrow = a.qs + (size_t)row * a.row_bytes;
    const uint16_t *srow = kBlocks ? a.scales + (size_t)row * (a.K / 32) : nullptr;
    // Activations of a step: eight lanes per row take its 128 bytes, eight rows per load; they go through the wavefront's own stretch of
    // LDS into fragment order.  Rows beyond M repeat the last one; rows of a tile beyond 8 NL repeat those before (sums never stored).
    const uint16_t *xrow[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int m = m0 + 8 * i + (lane >> 3);
        xrow[i] = a.x + (size_t)(m < a.M ? m : a.M - 1) * a.K + 8 * (lane & 7);
    }
    _Float16 *xs = reinterpret_cast<_Float16 *>(red) + (size_t)wave * NL * 8 * kXRow;
    _Float16 *xs_write = xs + (lane >> 3) * kXRow + 8 * (lane & 7);
    const _Float16 *xs_read = xs + (NL >= 4 ? col : col & (8 * NL - 1)) * kXRow + (FMT == FMT_Q8_0 || FMT == FMT_Q4_K ? 16 : 8) * h;
    auto load_w = [&](int s) {
        Packed<FMT> p;
        if constexpr (FMT == FMT_Q4_K) p.q = *reinterpret_cast<const uint4 *>(wrow + (size_t)(s >> 2) * 144 + 16 + (s & 3) * 32 + 16 * h);
        else if constexpr (FMT == FMT_Q4_0) {
            p.q = *reinterpret_cast<const uint4 *>(wrow + (size_t)s * 32 + 16 * h);
            p.d = *reinterpret_cast<const u32 *>(srow + 2 * s);
        } else if constexpr (FMT == FMT_Q8_0) {
#pragma unroll
            for (int b = 0; b < 2; b++) p.q[b] = *reinterpret_cast<const uint4 *>(wrow + (size_t)s * 64 + 32 * b + 16 * h);
            p.d = *reinterpret_cast<const u32 *>(srow + 2 * s);
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) p.q[j] = *reinterpret_cast<const uint4 *>(wrow + (size_t)s * 128 + 32 * j + 16 * h);
        }
        return p;
    };
    struct XStep { uint4 v[NL]; };
    auto load_x = [&](int s) {
        XStep x;
#pragma unroll
        for (int i = 0; i < NL; i++) x.v[i] = *reinterpret_cast<const uint4 *>(xrow[i] + (size_t)s * kStep);
        return x;
    };
    // fragment j: eight k at 32 (j / 2) + 8 (j % 2) or 16 j (see above)
    auto frag = [&](int j) {
        return *reinterpret_cast<const half8 *>(xs_read + (FMT == FMT_Q8_0 || FMT == FMT_Q4_K ? 32 * (j >> 1) + 8 * (j & 1) : 16 * j));
    };
    auto load_hdr = [&](int s) { return *reinterpret_cast<const uint4 *>(wrow + (size_t)(s >> 2) * 144); };

    const floatx16 zero16 = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    floatx16 tot = zero16, acc, accm;

    Packed<FMT> w[kAhead];
    XStep x[kAhead];
    uint4 hdr = {0, 0, 0, 0}, hdr_next = {0, 0, 0, 0};
    if (s_begin < s_end) {
        const int last = s_end - 1;
        auto at = [&](int s) { return s < last ? s : last; };   // steps past the end repeat the last one: in bounds, never used
        if constexpr (kSuper) { hdr = load_hdr(s_begin); hdr_next = load_hdr(at(s_begin + 4)); }
#pragma unroll
        for (int d = 0; d < kAhead; d++) { w[d] = load_w(at(s_begin + d)); x[d] = load_x(at(s_begin + d)); }
        auto step = [&](auto slot_c, int c, int s) {   // c: the step's place in its super-block
            constexpr int S = decltype(slot_c)::value;
            // a wavefront's LDS operations keep their order: the reads of the step before are done when these writes land
#pragma unroll
            for (int i = 0; i < NL; i++) *reinterpret_cast<uint4 *>(xs_write + 8 * i * kXRow) = x[S].v[i];
            x[S] = load_x(at(s + kAhead));
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if constexpr (FMT == FMT_F16) {
#pragma unroll
                for (int j = 0; j < 4; j++) tot = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag(j), as_half8(w[S].q[j]), tot, 0, 0, 0);
            } else if constexpr (FMT == FMT_Q8_0) {
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    const half8 f0 = bytes8(w[S].q[b].x, w[S].q[b].y), f1 = bytes8(w[S].q[b].z, w[S].q[b].w);
                    const float d = half_bits_to_float(b ? w[S].d >> 16 : w[S].d & 0xFFFFu);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag(2 * b), f0, zero16, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag(2 * b + 1), f1, acc, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 16; r++) tot[r] = __builtin_fmaf(d, acc[r], tot[r]);
                }
            } else if constexpr (FMT == FMT_Q4_0) {
                // lanes 0..31 hold block 0 of the step, lanes 32..63 block 1: after the exchange every lane holds bytes 8 h .. 8 h + 7 of both
                const auto e0 = __builtin_amdgcn_permlane32_swap(w[S].q.x, w[S].q.z, false, false);
                const auto e1 = __builtin_amdgcn_permlane32_swap(w[S].q.y, w[S].q.w, false, false);
                const h2 one = {(_Float16)1.0f, (_Float16)1.0f}, lo_off = {(_Float16)-1032.0f, (_Float16)-1032.0f}, hi_off = {(_Float16)-72.0f, (_Float16)-72.0f};
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    const half8 f0 = nibbles(e0[b], e1[b], false, one, lo_off), f1 = nibbles(e0[b], e1[b], true, one, hi_off);
                    const float d = half_bits_to_float(b ? w[S].d >> 16 : w[S].d & 0xFFFFu);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag(2 * b), f0, zero16, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag(2 * b + 1), f1, acc, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 16; r++) tot[r] = __builtin_fmaf(d, acc[r], tot[r]);
                }
            } else {
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    u32 sc, mn;
                    q4k_scale_min(hdr, 2 * c + p, sc, mn);
                    const _Float16 s1 = (_Float16)(unsigned short)sc, m1 = (_Float16)(unsigned short)mn;
                    const h2 mul = {s1, s1}, add = mul * (p ? h2{(_Float16)-64.0f, (_Float16)-64.0f} : h2{(_Float16)-1024.0f, (_Float16)-1024.0f});
                    const u32 mm = as_u32(h2{m1, m1});
                    const half8 f0 = nibbles(w[S].q.x, w[S].q.y, p, mul, add), f1 = nibbles(w[S].q.z, w[S].q.w, p, mul, add), fm = as_half8(make_uint4(mm, mm, mm, mm));
                    const half8 x0 = frag(2 * p), x1 = frag(2 * p + 1);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(x0, f0, (c == 0 && p == 0) ? zero16 : acc, 0, 0, 0);
                    accm = __builtin_amdgcn_mfma_f32_32x32x16_f16(x0, fm, (c == 0 && p == 0) ? zero16 : accm, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(x1, f1, acc, 0, 0, 0);
                    accm = __builtin_amdgcn_mfma_f32_32x32x16_f16(x1, fm, accm, 0, 0, 0);
                }
                if (c == 3) {
                    const float d = half_bits_to_float(hdr.x & 0xFFFFu), dmin = half_bits_to_float(hdr.x >> 16);
#pragma unroll
                    for (int r = 0; r < 16; r++) tot[r] = __builtin_fmaf(-dmin, accm[r], __builtin_fmaf(d, acc[r], tot[r]));
                    hdr = hdr_next;
                    hdr_next = load_hdr(at(s + 5));
                }
            }
            w[S] = load_w(at(s + kAhead));
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        };
        int s = s_begin;
        for (; s + 4 <= s_end; s += 4) {   // no branch around a load: the compiler then knows how many are in flight
            step(std::integral_constant<int, 0>{}, 0, s);
            step(std::integral_constant<int, 1>{}, 1, s + 1);
            step(std::integral_constant<int, 2>{}, 2, s + 2);
            step(std::integral_constant<int, 3>{}, 3, s + 3);
        }
        if constexpr (!kSuper) {
            if (s < s_end) step(std::integral_constant<int, 0>{}, 0, s);
            if (s + 1 < s_end) step(std::integral_constant<int, 1>{}, 1, s + 1);
            if (s + 2 < s_end) step(std::integral_constant<int, 2>{}, 2, s + 2);
        }
    }

    // ---- the wavefronts' sums meet in LDS; wavefront w finishes accumulators w * kShare .. of every lane ----
    constexpr int kShare = 16 / kWaves;
    static_assert(kShare % 2 == 0, "whole pairs of accumulators per wavefront");
    __syncthreads();   // everybody is done with the activations
#pragma unroll
    for (int r = 0; r < 16; r++) red[((size_t)wave * 16 + r) * 64 + lane] = tot[r];
    // accumulator r: activation row 8 (r / 4) + 4 h + r % 4
    float res[kShare];
#pragma unroll
    for (int k = 0; k < kShare; k++) {
        const int r = wave * kShare + k, m = m0 + 8 * (r >> 2) + 4 * h + (r & 3);
        res[k] = a.residual && n < a.N && m < a.M ? a.residual[(size_t)m * a.N + n] : 0.0f;
    }
    __syncthreads();
    float sum[kShare];
#pragma unroll
    for (int k = 0; k < kShare; k++) {
        const int r = wave * kShare + k;
        float v = red[(size_t)r * 64 + lane];
#pragma unroll
        for (int wv = 1; wv < kWaves; wv++) v += red[((size_t)wv * 16 + r) * 64 + lane];
        sum[k] = v;
    }
    if (a.act) {   // weight rows are (gate, up) pairs, neighbouring lanes: the even lane finishes the even accumulators, the odd lane the odd ones
#pragma unroll
        for (int k = 0; k < kShare; k += 2) {
            const float p0 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, sum[k]), 0xB1, 0xF, 0xF, false));       // quad_perm [1,0,3,2]
            const float p1 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, sum[k + 1]), 0xB1, 0xF, 0xF, false));
            const bool odd = lane & 1;
            const float g = odd ? p1 : sum[k], up = odd ? sum[k + 1] : p0;
            const int r = wave * kShare + k + (odd ? 1 : 0), m = m0 + 8 * (r >> 2) + 4 * h + (r & 3);
            if (m < a.M && (n | 1) < a.N) {
                a.act[(size_t)m * (a.N / 2) + n / 2] = __builtin_bit_cast(uint16_t, (_Float16)__fmul_rn(silu(g), up));
            }
        }
        return;
    }
#pragma unroll
    for (int k = 0; k < kShare; k++) {
        const int r = wave * kShare + k, m = m0 + 8 * (r >> 2) + 4 * h + (r & 3);
        if (m < a.M && n < a.N) a.y[(size_t)m * a.N + n] = a.residual ? res[k] + sum[k] : sum[k];
    }
}

template <int FMT, int NL>
hipError_t launch(const RowsArgs &a, hipStream_t s) {
    hipLaunchKernelGGL((rows_gemm_kernel<FMT, NL>), dim3((a.N + 31) / 32, (a.M + 8 * NL - 1) / (8 * NL)), dim3(kWaves * 64), rows_lds_bytes(NL), s, a);
    return hipGetLastError();
}

template <int FMT>
hipError_t launch_format(const RowsArgs &a, hipStream_t s) {
    if (a.M <= 8) return launch<FMT, 1>(a, s);
    if (a.M <= 16) return launch<FMT, 2>(a, s);
    return launch<FMT, 4>(a, s);   // more rows: one workgroup more per 32 of them
}

}  // namespace

static int g_rows_gemm_mode = -1;
static int rows_gemm_mode() {
    if (g_rows_gemm_mode < 0) { const char *e = getenv("ESPRESSO_HIP_ROWS_GEMM"); g_rows_gemm_mode = e ? atoi(e) : 1; }
    return g_rows_gemm_mode;
}
void rows_gemm_set_mode(int mode) { g_rows_gemm_mode = mode < 0 ? 1 : mode; }
bool rows_gemm_by_size() { return rows_gemm_mode() == 1; }

bool rows_gemm_takes(const GemmParams &p) {
    const DeviceMatrix &w = p.w;
    const int mode = rows_gemm_mode();
    if (mode == 0 || (mode == 1 && !p.unrounded) || (p.swiglu_out && (w.rows % 2 != 0 || p.residual)) || p.rows < 1 || w.cols % kStep != 0 || w.qs_row_bytes % 16 != 0) return false;
    if (w.format == FMT_Q4_K) { if (w.cols % 256 != 0) return false; }
    else if (w.format != FMT_Q4_0 && w.format != FMT_Q8_0 && w.format != FMT_F16) return false;
    if (mode == 2) return true;
    // Where a launch is a few steps deep and its workgroups are resident at once (us, tile or narrow kernel with its reduction -> this one):
    //   576 x 576, 16 / 93 / 256 rows: q8_0 6.9 / 11.2 / 11.4 -> 5.6 / 5.6 / 5.9, f16 6.6 / 10.8 / 11.1 -> 5.3 / 5.3 / 5.5
    //   2304 x 768, 16 / 93 / 256 rows: q4_k 7.6 / 14.6 / 15.0 -> 4.6 / 5.6 / 10.9;  512 rows 15.6 -> 17.7
    //   2048 x 2048, 16 / 93 / 256 rows: q8_0 10.6 / 16.2 / 19.2 -> 9.6 / 11.0 / 19.7, q4_k 9.3 / 16.2 / 19.2 -> 6.9 / 8.4 / 15.2
    //   4096 x 768, 93 / 256 / 512 rows: q8_0 14.8 / 15.3 / 16.0 -> 8.4 / 15.8 / 29.4
    //   3072 x 3072, 16 / 33 rows: q4_0 10.7 / 12.5 -> 9.2 / 9.5;  2048 x 5632, 16 / 93 rows: q8_0 14.0 / 21.6 -> 18.4 / 18.9 (a wavefront's eleven
    //   steps one after the other);  32000 x 768, 32 rows: q8_0 15.4 -> 17.9
    // Over 3 to 512 rows of seventeen shapes (576 to 8192 rows, 256 to 3072 columns) and the four formats, what the rule takes is 0.3 to 1.0 times the tile kernel's
    // time; at three rows of the 2048-column Q4_0 and 512 x 256 matrices, five to seven microseconds each way, up to 1.1 times.
    // Up to 32 rows that no next kernel finishes: deeper launches too, while all workgroups are resident at once (8192 x 3072, 8 / 32 rows, with shares of K and their sum -> here: q4_0
    // 10.5 / 11.9 -> 9.2 / 11.1, q8_0 12.4 / 14.1 -> 11.6 / 13.9, q4_k 16 rows 12.6 -> 9.3).
    // Beyond kExactRows the rule is what it is there: a prompt's rows keep the weights that they keep in a block of that length, however long theirs is (30 layers of 576 columns, 1000 / 1777
    // tokens, rounded -> kept: Q8_0 2660 / 4040 -> 2750 / 4380 us, Q4_0 2220 / 3010 -> 2320 / 3290).
    const int steps = w.cols / kStep, rows = w.format != FMT_F16 && p.rows > kExactRows ? kExactRows : p.rows;
    const long groups = (long)((w.rows + 31) / 32) * ((rows + 31) / 32);
    if (w.format == FMT_F16) {
        // rounds of one workgroup per compute unit against the kernel of wide_gemm.hip (us, here / there: 3072 x 576, 64 / 96 rows 5.1 / 6.3, 8.3 / 6.4;  576 x 1536, 16 / 200 / 400 rows
        // 6.0 / 5.4, 6.7 / 6.6, 6.8 / 7.6;  1152 x 576, 200 / 320 rows 5.3 / 6.1, 8.5 / 6.2;  2048 columns: there at any number of rows)
        const int cus = device_compute_units() > 0 ? device_compute_units() : 256;
        return w.cols <= 1536 && 1.7f + (float)((groups + cus - 1) / cus) * (2.6f + 0.19f * (float)steps) < wide_gemm_form(p).us;
    }
    const bool deep = groups * steps > 8192 && (rows > 32 || !block_gemm_alone(p) || groups > (device_compute_units() > 0 ? device_compute_units() : 256));
    return w.cols <= 3072 && !deep && !block_gemm_keeps(p);
}

hipError_t launch_rows_gemm(const GemmParams &p, hipStream_t stream) {
    const DeviceMatrix &w = p.w;
    RowsArgs a{w.qs, w.scales, w.qs_row_bytes, w.rows, w.cols, p.rows, p.x, p.y, p.residual, p.swiglu_out};
    switch (w.format) {
    case FMT_Q4_K: return launch_format<FMT_Q4_K>(a, stream);
    case FMT_Q4_0: return launch_format<FMT_Q4_0>(a, stream);
    case FMT_Q8_0: return launch_format<FMT_Q8_0>(a, stream);
    case FMT_F16: return launch_format<FMT_F16>(a, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace esp
