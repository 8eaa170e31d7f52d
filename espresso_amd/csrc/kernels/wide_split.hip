// y[m][n] = sum_k x[m][k] * W[n][k] for blocks of split rows (SplitRowsView) and Q4_K weights, exact as in gemm_split.hip: integers sc q on the matrix cores, the hi plane against them and the
// lo plane against them / 2048 into one set of sums, d and the minimums' product once per super-block.
//
// The walk is that of wide_tile.h, eight wavefronts, two buffers of 64 k, one barrier a step, with three operands in LDS: both planes of 128 rows, and the integers of 256 weight rows, which two threads
// a row unpack on their way there.  A wavefront of 64 x 64 reads six fragments for eight products, where block_split.hip, whose weights skip LDS, reads one for each.  Fragments are not read a whole
// slice of sixteen k ahead (that spills: 128 sums and totals) but half of one: the lo plane's while the hi plane's are multiplied, the next slice's hi plane and integers while the lo plane's are.
// What bounds it: power.  With all compute units at work a step takes 2.0 us, 1.4 with few, 1.7 with all and activations of zero.  What helped: lanes' offsets of 32 bits at uniform bases (load_at; 512 rows of
// 28672 x 4096 295 -> 275 us), two steps of a row's nibbles in one visit to its line.
// Against the kernels these products had (gemm_q4k_split_regb_kernel behind a SiLU, block_split.hip otherwise), us with their planes added:
//   28672 x 4096 behind a SiLU, 256 / 512 / 960 / 2048 rows 157 / 318 / 611 / 1099 -> 124 / 276 / 556 / 1029;  16384 x 2048, 512 / 2048 rows 82 / 368 -> 71 / 327;
//   4096 x 14336, 512 / 960 / 2048 rows 140 / 282 / 636 -> 122 / 232 / 472;  4096 x 4096, 2048 rows 171 -> 134;  6144 x 4096, 512 rows 70 -> 68.
// Kept out: tiles of 64 x 128 and 128 x 128, and 64 x 256 alone (0.7 to 1.0 times as fast as what those sizes have).
#include "../common.h"
#include "silu.h"
#include "split_rows.h"
#include "wide_split.h"
#include "wide_tile.h"
#include <atomic>
#include <type_traits>

namespace esp {
namespace {

using namespace wide;
using split_rows::kScale;
using split_rows::kUnscale;
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32;

struct WideSplitArgs {
    const uint8_t *qs;
    size_t row_bytes;
    int N, K, M;
    const uint16_t *xh, *xl, *xs;
    float *y;
    const float *residual;
    float *partial;
    uint16_t *sw_hi, *sw_lo, *sw_sums;
    int per, splits, n_tiles, m_tiles;   // per: super-blocks of a share
    int long_tiles;                      // two heights: the first of the m_tiles have 128 rows, the others 64
};

__device__ __forceinline__ h2 as_h2(u32 v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ u32 as_u32(h2 v) { return __builtin_bit_cast(u32, v); }
__device__ __forceinline__ float half_bits_to_float(u32 bits16) { return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16); }

// A pair of sub-blocks of Q4_K rows a step on its way to LDS as integers sc q, in the planes' order inside fours (0, 2, 1, 3).
template <int ROWS>
struct Packed {
    static constexpr int kParts = kThreads / ROWS, kWords = 8 / kParts;   // threads of a row, dwords of its 32 bytes that each has
    static_assert(kParts == 2, "sixteen bytes a thread");
    typedef u32 words __attribute__((ext_vector_type(kWords)));
    const uint8_t *base;                 // of the share's first super-block
    u32 row, offset;                     // bytes from base on: the row, and this thread's part of its nibbles
    words raw[2];                        // of a step of even number and the one behind it
    u32 scales, more, next_scales, next_more;   // the header's dwords 1 and 3, of this super-block and the next
    int at_lds, last;                    // last: step
    // eight neighbouring lanes have eight rows, whose LDS rows begin on different banks
    __device__ __forceinline__ Packed(const uint8_t *qs, size_t row_bytes, int row0, int count, int first, int steps) : base(qs + (size_t)row0 * row_bytes + (size_t)first * 144), last(steps - 1) {
        const int part = (threadIdx.x >> 3) & (kParts - 1), r = (threadIdx.x & 7) | (threadIdx.x / (8 * kParts) * 8);
        row = (u32)(row0 + r < count ? r : count - 1 - row0) * (u32)row_bytes;
        offset = row + 16 + part * kWords * 4;
        at_lds = r * kPitch + part * kWords * 4;
    }
    __device__ __forceinline__ void load(int s) {   // steps s (even) and s + 1: 64 bytes of a row, so that a line is fetched twice and not four times
        const int c = s < last ? s : last - 1;
        const uint8_t *from = base + (size_t)(c >> 2) * 144 + (c & 3) * 32;
        raw[0] = load_at<words>(from, offset);
        raw[1] = load_at<words>(from + 32, offset);
    }
    __device__ __forceinline__ void load_header(int s) {   // of step s's super-block
        const int c = s < last ? s : last;
        const uintx4 h = load_at<uintx4>(base + (size_t)(c >> 2) * 144, row);
        next_scales = h.y; next_more = h.w;
    }
    __device__ __forceinline__ void take_header() { scales = next_scales; more = next_more; }
    // the low nibbles (HIGH 0: sub-block 2 PAIR) or the high ones of the super-block's pair PAIR
    template <int PAIR, int HIGH>
    __device__ __forceinline__ void unpack(uint16_t *lds, u32 mask, u32 magic) {
        constexpr int j = 2 * PAIR + HIGH;
        u32 sc;
        if constexpr (j < 4) sc = (scales >> (8 * j)) & 63u;
        else sc = ((more >> (8 * (j - 4))) & 0xFu) | ((scales >> (8 * (j - 4) + 2)) & 0x30u);
        const _Float16 s1 = (_Float16)(unsigned short)sc;
        const h2 mul = {s1, s1}, add = mul * (HIGH ? h2{(_Float16)-64.0f, (_Float16)-64.0f} : h2{(_Float16)-1024.0f, (_Float16)-1024.0f});
#pragma unroll
        for (int g = 0; g < kWords / 2; g++) {
            uintx4 o;
#pragma unroll
            for (int i = 0; i < 4; i++) o[i] = as_u32(__builtin_elementwise_fma(as_h2(((i & 1 ? raw[PAIR & 1][2 * g + (i >> 1)] >> 8 : raw[PAIR & 1][2 * g + (i >> 1)]) & mask) | magic), mul, add));
            *reinterpret_cast<uintx4 *>(lds + at_lds + 32 * HIGH + 8 * g) = o;
        }
    }
};

constexpr int kWM = 2, kWN = 4, TN = 2, BN = 32 * kWN * TN, kLd = BN / 2 + 8;   // wavefronts, products of each, weight rows of a tile; units between the rows of the epilogue's planes
constexpr int rows_of(int tm) { return 32 * kWM * tm; }
constexpr int buffer_of(int tm) { return (2 * rows_of(tm) + BN) * kPitch; }
constexpr int kLong = rows_of(2), kShort = rows_of(1);
constexpr size_t kLdsBytes = (size_t)2 * buffer_of(2) * 2;
static_assert(kLdsBytes <= 160 * 1024 && (size_t)2 * kLong * kLd * 2 <= kLdsBytes, "LDS of a compute unit");

template <int TM>
__device__ __forceinline__ void wide_split_tile(const WideSplitArgs &a, const int m0, const int n_tile, const int split, uint16_t *lds) {
    constexpr int BM = rows_of(TM), kBuffer = buffer_of(TM);
    const int n0 = n_tile * BN, sbs = a.K / 256, first = split * a.per, blocks = sbs - first < a.per ? sbs - first : a.per, steps = 4 * blocks;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave / kWN, wn = wave % kWN, h = lane >> 5, col = lane & 31;
    Plain<BM, 1> hi(a.xh, (size_t)a.K, m0, a.M, (size_t)first * 256, steps), lo(a.xl, (size_t)a.K, m0, a.M, (size_t)first * 256, steps);
    Packed<BN> w(a.qs, a.row_bytes, n0, a.N, first, steps);

    // what the fold reads: headers of the wavefront's weight rows, the rows' sums over sub-blocks (8 x hi, 8 x lo)
    u32 ho[TN], so[TM];
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int n = n0 + (wn * TN + j) * 32 + col;
        ho[j] = (u32)((n < a.N ? n : a.N - 1) - n0) * (u32)a.row_bytes;
    }
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int m = m0 + (wm * TM + i) * 32 + col;
        so[i] = (u32)((m < a.M ? m : a.M - 1) - m0) * (u32)(sbs * 32) + 16 * h;
    }
    const uint8_t *sums = reinterpret_cast<const uint8_t *>(a.xs + ((size_t)m0 * sbs + first) * 16), *heads = a.qs + (size_t)n0 * a.row_bytes + (size_t)first * 144;

    floatx16 tot[TM][TN], acc[TM][TN];
    const floatx16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) { tot[i][j] = zero16; acc[i][j] = zero16; }
    // constants of the nibble trick, hidden from the optimiser so that (w & mask) | magic stays one v_and_or_b32
    u32 mask_lo = 0x000F000Fu, mask_hi = 0x00F000F0u, magic_lo = 0x64006400u, magic_hi = 0x54005400u;
    asm volatile("" : "+s"(mask_lo), "+s"(mask_hi));
    asm volatile("" : "+v"(magic_lo), "+v"(magic_hi));

    const int fx = (wm * TM * 32 + col) * kPitch + 8 * h, fw = (2 * BM + wn * TN * 32 + col) * kPitch + 8 * h;
    uintx4 hf[TM], lf[TM], wf[TN], wl[TN];
    auto read_top = [&](int buf, int ks) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < TN; j++) wf[j] = *reinterpret_cast<const uintx4 *>(lds + buf * kBuffer + fw + j * 32 * kPitch + ks * 16);
#pragma unroll
        for (int i = 0; i < TM; i++) hf[i] = *reinterpret_cast<const uintx4 *>(lds + buf * kBuffer + fx + i * 32 * kPitch + ks * 16);
    };
    auto read_rest = [&](int buf, int ks) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; i++) lf[i] = *reinterpret_cast<const uintx4 *>(lds + buf * kBuffer + fx + (BM + i * 32) * kPitch + ks * 16);
    };
    auto order = [&] __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < TM * TN; n++) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);     // a product
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // an LDS read
            __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);     // a share of the unpacking
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);   // an LDS write
            __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);    // a load
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    typedef std::integral_constant<int, 0> C0;
    typedef std::integral_constant<int, 1> C1;
    typedef std::integral_constant<int, 2> C2;
    typedef std::integral_constant<int, 3> C3;
    // a third of step `next - 1`, the PAIR-th of its super-block, to LDS, and of step `next` on its way
    auto stage = [&](auto part, auto pair, int buf, int next) __attribute__((always_inline)) {
        constexpr int PART = decltype(part)::value, PAIR = decltype(pair)::value;
        uint16_t *to = lds + buf * kBuffer;
        if constexpr (PART == 0) {
            hi.template stage<0, 0>(to, next); hi.template stage<1, 0>(to, next); hi.template stage<2, 0>(to, next);
        } else if constexpr (PART == 1) {
            if constexpr (PAIR == 0) w.take_header();
            w.template unpack<PAIR, 0>(to + 2 * BM * kPitch, mask_lo, magic_lo);
            lo.template stage<0, 0>(to + BM * kPitch, next); lo.template stage<1, 0>(to + BM * kPitch, next); lo.template stage<2, 0>(to + BM * kPitch, next);
        } else {
            w.template unpack<PAIR, 1>(to + 2 * BM * kPitch, mask_hi, magic_hi);
            if constexpr (PAIR & 1) w.load(next);
            if constexpr (PAIR == 1) w.load_header(next + 2);   // (step next - 1 is 1 mod 4: the next super-block's)
        }
    };
    hi.load(0, 0);
    lo.load(0, 0);
    w.load(0);
    w.load_header(0);
    stage(C0{}, C0{}, 0, 1);
    stage(C1{}, C0{}, 0, 1);
    stage(C2{}, C0{}, 0, 1);
    __syncthreads();
    read_top(0, 0);
    uintx4 head[TN], fs[TM];
    const h2 unscale = {(_Float16)kUnscale, (_Float16)kUnscale};
    auto step = [&](auto turn, int s) __attribute__((always_inline)) {
        constexpr int P = decltype(turn)::value, B = P & 1;
        constexpr std::integral_constant<int, (P + 1) & 3> pair{};   // of the next step
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            // the hi plane's products, while the lo plane's fragments come in
            read_rest(B, ks);
            if (ks == 0) stage(C0{}, pair, B ^ 1, s + 2);
            else if (ks == 1) stage(C1{}, pair, B ^ 1, s + 2);
            else if (ks == 2) stage(C2{}, pair, B ^ 1, s + 2);
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) wl[j][e] = as_u32(as_h2(wf[j][e]) * unscale);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = multiply<false>(hf[i], wf[j], P == 0 && ks == 0 ? zero16 : acc[i][j]);
            order();
            // the lo plane's, while the others of the next slice do
            if (ks == 3) __syncthreads();   // everybody has read this buffer, and written the other one
            if (ks < 3) read_top(B, ks + 1);
            else read_top(B ^ 1, 0);
            if (P == 3 && ks == 2) {
                const size_t block = (size_t)(s >> 2);
#pragma unroll
                for (int j = 0; j < TN; j++) head[j] = load_at<uintx4>(heads + block * 144, ho[j]);
#pragma unroll
                for (int i = 0; i < TM; i++) fs[i] = load_at<uintx4>(sums + block * 32, so[i]);
            }
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = multiply<false>(lf[i], wl[j], acc[i][j]);
            order();
        }
        if constexpr (P == 3) {   // the super-block's fold: d times its sums less dmin sum_j m_j S_j, one product against (m_0..m_7) and (m_0..m_7) / 2048
            const _Float16 f = (_Float16)(h ? kUnscale : 1.0f);
            const h2 off = {(_Float16)1024.0f, (_Float16)1024.0f}, k = {f, f};
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const u32 low = head[j].z & 0x3F3F3F3Fu, high = ((head[j].w >> 4) & 0x0F0F0F0Fu) | ((head[j].z >> 2) & 0x30303030u);
                uintx4 mq;
                mq.x = as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, low, 0x04010400u)) - off) * k);
                mq.y = as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, low, 0x04030402u)) - off) * k);
                mq.z = as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, high, 0x04010400u)) - off) * k);
                mq.w = as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, high, 0x04030402u)) - off) * k);
                const float d = half_bits_to_float(head[j].x & 0xFFFFu), dmin = half_bits_to_float(head[j].x >> 16);
#pragma unroll
                for (int i = 0; i < TM; i++) {   // (the minimums' product in the registers of the sums it follows: there are no others)
#pragma unroll
                    for (int r = 0; r < 16; r++) tot[i][j][r] = __builtin_fmaf(d, acc[i][j][r], tot[i][j][r]);
                    acc[i][j] = multiply<false>(fs[i], mq, zero16);
                }
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) tot[i][j][r] = __builtin_fmaf(-dmin, acc[i][j][r], tot[i][j][r]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int s = 0; s < steps; s += 4) {
        step(C0{}, s);
        step(C1{}, s + 1);
        step(C2{}, s + 2);
        step(C3{}, s + 3);
    }

    // a lane's sum r of tile (i, j): row m0 + 32 (wm TM + i) + 8 (r / 4) + 4 h + r % 4, weight row n0 + 32 (wn TN + j) + col
    if (a.sw_hi) {   // weight rows as (gate, up) pairs are neighbouring lanes: the even lane finishes rows 2 k of both, the odd lane rows 2 k + 1; the units leave through LDS
        constexpr int RP = BN / 16;   // sixteen-byte pieces of a row of units
        uint16_t *top = lds, *rest = lds + BM * kLd;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int u = ((wn * TN + j) * 32 + col) >> 1, slot = u & 3, at_u = (u & ~3) + (slot == 1 ? 2 : slot == 2 ? 1 : slot);   // the planes' order inside fours: 0, 2, 1, 3
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const float even = tot[i][j][2 * k], uneven = tot[i][j][2 * k + 1];
                    const float p0 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, even), 0xB1, 0xF, 0xF, false));   // quad_perm [1,0,3,2]
                    const float p1 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, uneven), 0xB1, 0xF, 0xF, false));
                    const float act = __fmul_rn(silu(lane & 1 ? p1 : even), lane & 1 ? uneven : p0);
                    const int r = 2 * k + (lane & 1), o = ((wm * TM + i) * 32 + 8 * (r >> 2) + 4 * h + (r & 3)) * kLd + at_u;
                    const _Float16 t = (_Float16)act;
                    top[o] = __builtin_bit_cast(uint16_t, t);
                    rest[o] = __builtin_bit_cast(uint16_t, (_Float16)__fmul_rn(__fsub_rn(act, (float)t), kScale));
                }
            }
        __syncthreads();
        const int units = a.N / 2, unit0 = n_tile * (BN / 2);
        for (int p = threadIdx.x; p < BM * RP; p += kThreads) {   // units is a multiple of 32: the four lanes of a sub-block are in or out together
            const int r = p / RP, c8 = (p % RP) * 8, m = m0 + r;
            if (m >= a.M || unit0 + c8 >= units) continue;
            const uintx4 hv = *reinterpret_cast<const uintx4 *>(top + r * kLd + c8), lv = *reinterpret_cast<const uintx4 *>(rest + r * kLd + c8);
            const size_t o = (size_t)m * units + unit0 + c8;
            *reinterpret_cast<uintx4 *>(a.sw_hi + o) = hv;
            *reinterpret_cast<uintx4 *>(a.sw_lo + o) = lv;
            float sum = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const h2 hp = as_h2(hv[e]), lp = as_h2(lv[e]);
                sum += __builtin_fmaf((float)lp.x, kUnscale, (float)hp.x) + __builtin_fmaf((float)lp.y, kUnscale, (float)hp.y);
            }
            split_rows::store_subblock_sum(a.sw_sums, (size_t)m, units, (unit0 + c8) >> 3, sum);
        }
        return;
    }
    float *out = a.splits > 1 ? a.partial + (size_t)split * a.M * a.N : a.y;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int n = n0 + (wn * TN + j) * 32 + col, mb = m0 + (wm * TM + i) * 32 + 4 * h;
            auto row = [&](int r) { return mb + 8 * (r >> 2) + (r & 3); };
            if (a.splits == 1 && a.residual) {   // requested together: y may be the residual's own memory, and a load behind each store is a trip to memory each
                float before[16];
#pragma unroll
                for (int r = 0; r < 16; r++) before[r] = a.residual[(size_t)(row(r) < a.M ? row(r) : a.M - 1) * a.N + (n < a.N ? n : a.N - 1)];
#pragma unroll
                for (int r = 0; r < 16; r++) tot[i][j][r] += before[r];
            }
#pragma unroll
            for (int r = 0; r < 16; r++) if (row(r) < a.M && n < a.N) out[(size_t)row(r) * a.N + n] = tot[i][j][r];
        }
}

// TWO: two heights of tiles in one launch, the long ones first (no shares of K).
template <bool TWO>
__global__ __launch_bounds__(kThreads) void wide_split_kernel(WideSplitArgs a) {
    extern __shared__ uint4 smem[];
    uint16_t *lds = reinterpret_cast<uint16_t *>(smem);
    if constexpr (!TWO) {
        const auto [m_tile, n_tile, split] = place_of(a.m_tiles, a.n_tiles, blockIdx.x, gridDim.x);
        wide_split_tile<2>(a, m_tile * kLong, n_tile, split, lds);
    } else {
        const int longs = a.long_tiles * a.n_tiles;
        if ((int)blockIdx.x < longs) {
            const auto [m_tile, n_tile, split] = place_of(a.long_tiles, a.n_tiles, blockIdx.x, longs);
            wide_split_tile<2>(a, m_tile * kLong, n_tile, 0, lds);
        } else {
            const auto [m_tile, n_tile, split] = place_of(a.m_tiles - a.long_tiles, a.n_tiles, blockIdx.x - longs, gridDim.x - longs);
            wide_split_tile<1>(a, a.long_tiles * kLong + m_tile * kShort, n_tile, 0, lds);
        }
    }
}

std::atomic<int> g_wide_split_shares{0};

}  // namespace

void wide_split_set_shares(int shares) { g_wide_split_shares.store(shares < -1 ? 0 : shares); }

// Expected time: a start; rounds of one workgroup per compute unit, whose super-blocks take 4.5 us with few units at work and 7.4 with all (power); filling and emptying a tile; what it stores; planes that
// the next kernel reads once more.  Fitted to 600 launches with weights that no cache holds (thirteen shapes of 1536 to 28672 weight rows and 768 to 14336 columns, 128 to 2048 rows): off by
// 3 % at the median, 9 at the ninetieth percentile.
WideSplitForm wide_split_form(const GemmSplitParams &p) {
    const bool swiglu = p.swiglu.hi != nullptr;
    const int forced = g_wide_split_shares.load(), N = p.w.rows, M = p.rows, blocks = p.w.cols / 256, cus = device_compute_units() > 0 ? device_compute_units() : 256;
    WideSplitForm best;
    if (forced < 0 || (forced == 0 && M <= 64) || (swiglu && ((N / 2) % 32 != 0 || !p.swiglu.sums))) return best;
    const int kShares[] = {1, 2, 3, 4, 6, 8};
    for (int want : kShares) {
        if (forced > 0 && want != (swiglu || forced >= 100 ? 1 : forced)) continue;
        const int per = (blocks + want - 1) / want, splits = (blocks + per - 1) / per;
        if ((splits != want && forced == 0) || (splits > 1 && (swiglu || !p.workspace || (size_t)splits * M * N > p.workspace_floats))) continue;
        const long wgs = (long)((N + BN - 1) / BN) * ((M + kLong - 1) / kLong) * splits, rounds = (wgs + cus - 1) / cus;
        float us = 1.3f + (float)per * (4.46f * (float)rounds + 2.93f * (float)wgs / (float)cus) + 5.5f * (float)rounds + 0.22f * (float)splits * (float)M * (float)N * (swiglu ? 2e-6f : 4e-6f);
        if (splits > 1) us += 1.75f + 0.35f * (float)splits;
        if (!best.per || us < best.us) best = WideSplitForm{per, splits, us};
    }
    // Where the last round of tiles would be nearly empty, or the last tile: tiles of 64 rows at the end, which each compute unit takes as it comes free (0.65 of a tile's time, half of its power).  What the
    // rule takes was the best of 159 launches' forms every time, 1.00 to 1.18 times as fast as tiles of one height; behind a SiLU, us: 28672 x 4096, 300 / 600 / 800 / 1777 rows 230 / 360 / 488 / 900 ->
    // 194 / 334 / 421 / 871;  11264 x 2048, 800 / 1000 rows 121 / 125 -> 104 / 111;  16384 x 2048, 400 / 600 / 1777 rows 72 / 122 / 271 -> 68 / 107 / 258.  512 rows: tiles of one height, like 1000 and 1400 of
    // the widest.
    if (forced == 0 && best.per) {
        const int n_tiles = (N + BN - 1) / BN;
        float least = 0.98f * best.us;
        for (int longs = 1; longs * kLong < M; longs++) {
            const int shorts = n_tiles * ((M - longs * kLong + kShort - 1) / kShort), full = n_tiles * longs / cus, ahead = n_tiles * longs % cus;
            float early = (float)full, late = (float)(full + (ahead ? 1 : 0));
            for (int left = shorts; left > 0;) {
                const bool at_early = early <= late || !ahead;
                left -= at_early ? cus - ahead : ahead;
                (at_early ? early : late) += 0.65f;
            }
            const float rounds = early > late ? early : late;
            const float us = 1.3f + (float)blocks * (4.46f * rounds + 2.93f * ((float)(n_tiles * longs) + 0.5f * (float)shorts) / (float)cus) + 5.5f * rounds + 0.22f * (float)M * (float)N * (swiglu ? 2e-6f : 4e-6f);
            if (us < least) { least = us; best = WideSplitForm{blocks, 1, us, longs}; }
        }
    }
    if (forced > 0) best.us = 0.0f;
    if (forced >= 100 && forced / 100 * kLong < M) best.long_tiles = forced / 100;
    return best;
}

hipError_t launch_wide_split(const GemmSplitParams &p, const WideSplitForm &f, hipStream_t stream) {
    const WideSplitArgs a{p.w.qs, p.w.qs_row_bytes, p.w.rows, p.w.cols, p.rows, p.x.hi, p.x.lo, p.x.sums, p.y, p.residual, p.workspace, p.swiglu.hi, p.swiglu.lo, p.swiglu.sums,
                          f.per, f.splits, (p.w.rows + BN - 1) / BN, f.long_tiles ? f.long_tiles + (p.rows - f.long_tiles * kLong + kShort - 1) / kShort : (p.rows + kLong - 1) / kLong, f.long_tiles};
    auto go = [&](auto kernel, std::atomic<uint64_t> &raised) {
        const hipError_t err = raise_lds_limit(reinterpret_cast<const void *>(kernel), kLdsBytes, raised);
        if (err != hipSuccess) return err;
        hipLaunchKernelGGL(kernel, dim3(a.n_tiles * a.m_tiles * a.splits), dim3(kThreads), kLdsBytes, stream, a);
        return hipGetLastError();
    };
    static std::atomic<uint64_t> raised_one{0}, raised_two{0};
    return f.long_tiles ? go(wide_split_kernel<true>, raised_two) : go(wide_split_kernel<false>, raised_one);
}

}  // namespace esp
