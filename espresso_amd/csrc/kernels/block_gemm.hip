// y[m][n] = sum_k x[m][k] * W[n][k] for blocks of activation rows, W in Q4_K, Q4_0 or Q8_0: fp16 operands (every dequantised weight is rounded to fp16
// once), fp32 sums.
//
// A workgroup is eight wavefronts, two on every SIMD, so that one unpacks weights while the other multiplies.  NW of them lie side by side along 32 NW weight rows and
// 8 / NW groups share K; each wavefront owns 32 weight rows and all 32 TM activation rows of the workgroup's tile.
//   * The weights never enter LDS: a lane unpacks eight k of its own row into the B operand of v_mfma_f32_32x32x16_f16, which then serves TM products.
//   * Four lanes cover 64 bytes of a row (sixteen rows a load), and v_permlane16_swap brings each lane the two pieces of its own row: a quarter to a half of the cache
//     accesses of lanes that read their own rows.  Those lanes are sixteen apart, so the cache still looks every sixteen bytes up by themselves; Q8_0, which has two such loads for each of the others',
//     takes neighbouring lanes and turns the rows in LDS, one fragment ahead of their use.  us, exchanged -> turned: 2048 x 5632, 33 / 93 / 512 rows 11.7 / 13.6 / 27.8 -> 10.8 / 12.4 / 26.2;
//     2560 x 2048 exact, 33 / 64 / 93 rows 9.5 / 10.3 / 10.2 -> 8.8 / 9.3 / 8.4;  11264 x 2048, 64 / 320 / 512 rows 16.8 / 33.8 / 42.1 -> 15.1 / 30.3 / 40.4, 1777 rows the same.  The others
//     lose 2 to 10 % by the longer way (3072 x 2048 Q4_0, 64 rows 7.7 -> 9.6; 3072 x 8192 Q4_K, 33 rows 13.3 -> 15.4).
//   * Loads are spread over the step, one step of 128 k ahead: more in flight only blocks the wavefronts that issue them (two steps ahead, requested in one go:
//     11264 x 2048 Q8_0, 512 rows 38.8 us, 16 rows 11.9 against 37.8 and 11.6; 3072 x 8192 Q4_0, 512 rows 35.9 against 33.9).
//   * Activations go through LDS, two buffers and one barrier a step, fragment g + 1 read while g is multiplied (left to the compiler: 3 to 5 % slower).
//   * Q4_K's n s - dm is one v_fma_mix a weight (a nibble alone in sixteen bits is the fp16 number n 2^-24), rounded once as before; v_cvt_f32_ubyte, an fp32
//     multiply-add and a conversion take almost twice the instructions.
// What bounds it: at 512 rows no unit alone (16384 x 3072 Q4_K, 63 us in a prompt's trace: matrix cores 20 us of their own, 10 000 vector instructions a SIMD 17, 52 MB read 10, no LDS
// bank conflicts; a copy without loads and unpacking took 37); at 100 rows and less the weights' way from memory and the steps' latencies.  Against the kernel of 128 x 128 tiles
// whose weights go through LDS (gemm.hip), both in turn, us:
//   16384 x 3072 Q4_0, 512 / 192 / 96 rows 69 / 48 / 33 -> 55 / 30 / 23;  3072 x 8192 Q4_0 45 / 32 / 20 -> 33 / 20 / 14;  11264 x 2048 Q8_0 44 / 36 / 27 -> 38 / 24 / 17;
//   11264 x 2048 Q4_K 44 / 37 / 29 -> 35 / 20 / 15.
#include "../common.h"
#include "block_gemm.h"
#include "block_tile.h"
#include "silu.h"
#include <type_traits>

namespace esp {
namespace {

using namespace block_tile;
typedef u32 uintx4 __attribute__((ext_vector_type(4)));

struct BlockArgs {
    const uint8_t *qs;
    const uint16_t *scales;
    size_t row_bytes;
    int N, K, M;
    const uint16_t *x;
    float *y;
    const float *residual;
    float *partial;
    uint16_t *swiglu_out;
    int per, splits, n_tiles, m_tiles;   // per: steps of one group of wavefronts
    int long_tiles;                      // mixed heights: the first of the m_tiles have the kernel's height, the others the shorter one
};

__device__ __forceinline__ h2 splat_bits(u32 bits16) { return as_h2(__builtin_amdgcn_perm(bits16, bits16, 0x01000100u)); }
__device__ __forceinline__ uint4 swap_middle(const uint4 &v) {
    return make_uint4(__builtin_amdgcn_perm(v.y, v.x, 0x05040100u), __builtin_amdgcn_perm(v.y, v.x, 0x07060302u), __builtin_amdgcn_perm(v.w, v.z, 0x05040100u),
                      __builtin_amdgcn_perm(v.w, v.z, 0x07060302u));
}
constexpr int pairs_of(int fmt) { return fmt == FMT_Q8_0 ? 2 : 1; }   // 64-byte stretches of a row in a step

// Weights through LDS on their way to the lanes of their rows
constexpr bool turned(int fmt, int tm, int nw) { return fmt == FMT_Q8_0 && !(tm == 3 && nw == 2); }   // (that form has one buffer for its activations as it is, and was 2 to 5 % slower)
constexpr int kTurn = 80;                          // bytes between the rows there
constexpr size_t turn_bytes(int fmt, int tm, int nw) { return turned(fmt, tm, nw) ? (size_t)kWaves * 32 * kTurn : 0; }
template <int FMT, int TM, int NW>
constexpr int block_buffers() { return 2 * (kWaves / NW) * 32 * TM * kRow * 2 + turn_bytes(FMT, TM, NW) <= 160 * 1024 ? 2 : 1; }
template <int FMT, int TM, int NW>
constexpr size_t block_lds_bytes() {
    const size_t x = (size_t)block_buffers<FMT, TM, NW>() * (kWaves / NW) * 32 * TM * kRow * 2 + turn_bytes(FMT, TM, NW), sums = kWaves / NW > 1 ? (size_t)kWaves * TM * 16 * 64 * 4 : 0;
    return x > sums ? x : sums;
}

// EXACT (Q8_0, Q4_0; one row tile): integers go to the matrix cores, a block's scale to its sums.  Every product then contracts one block, each half of a wavefront holding half of it.
template <int FMT, int TM, int NW, bool EXACT>
__device__ __forceinline__ void block_product(const BlockArgs &a, const int m0, const int n_tile, const int split, uint4 *smem) {
    static_assert(!EXACT || FMT == FMT_Q8_0 || FMT == FMT_Q4_0, "formats of one scale per block");
    constexpr int KW = kWaves / NW, MT = 32 * TM, GT = 64 * NW, BUFS = block_buffers<FMT, TM, NW>();
    constexpr int XP = MT * (kStep / 8) / GT;       // sixteen-byte pieces of the activations per thread and step
    static_assert(MT * (kStep / 8) % GT == 0 && XP >= 1, "whole pieces");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, col = lane & 31;
    const int wn = wave % NW, wk = wave / NW, gtid = wn * 64 + lane;
    const int n0 = (n_tile * NW + wn) * 32, n = n0 + col;
    const int row0 = n0 < a.N ? n0 : a.N - 1;
    auto row_of = [&](int r) { return row0 + r < a.N ? r : a.N - 1 - row0; };   // rows from row0 on, clamped: those beyond are never stored
    // every group of wavefronts passes the same barriers and has steps of its own
    const int all = a.K / kStep, s0 = (split * KW + wk) * a.per, own = all - s0 < a.per ? (all > s0 ? all - s0 : 0) : a.per;
    auto at = [&](int s) { return s0 + s < all ? s0 + s : all - 1; };          // steps past the end repeat the last: in bounds, never used

    _Float16 *xt = reinterpret_cast<_Float16 *>(smem) + wk * BUFS * MT * kRow;   // [BUFS][MT][kRow]
    uint4 xv[XP];
    u32 xo[XP];                                // elements from row m0 on
#pragma unroll
    for (int i = 0; i < XP; i++) {
        const int piece = gtid + i * GT, r = piece >> 4, part = piece & 15;
        xo[i] = (u32)(m0 + r < a.M ? r : a.M - 1 - m0) * (u32)a.K + part * 8;
    }
    const uint16_t *xbase = a.x + (size_t)m0 * a.K;
    auto load_x = [&](int s) __attribute__((always_inline)) {
        const uint16_t *p = xbase + (size_t)at(s) * kStep;
#pragma unroll
        for (int i = 0; i < XP; i++) xv[i] = *reinterpret_cast<const uint4 *>(p + xo[i]);
    };
    auto store_x = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < XP; i++) {
            const int piece = gtid + i * GT, r = piece >> 4, part = piece & 15;
            *reinterpret_cast<uint4 *>(xt + buf * MT * kRow + r * kRow + part * 8) = FMT == FMT_Q4_0 ? swap_middle(xv[i]) : xv[i];
        }
    };
    // Weights.  Turned: four neighbouring lanes load 64 bytes of a row, and a stretch of LDS of the wavefront's own brings each lane two pieces of row lane % 32.  Otherwise lanes sixteen apart, for
    // exchange_rows.  Pieces 2 h and 2 h + 1; exact: h and 2 + h.
    constexpr bool TURN = turned(FMT, TM, NW);
    const int piece = TURN ? lane & 3 : EXACT ? 2 * ((lane >> 4) & 1) + h : lane >> 4, wrow = TURN ? lane >> 2 : lane & 15;
    const uint8_t *wbase = a.qs + (size_t)row0 * a.row_bytes;
    const u32 wlo = (u32)row_of(wrow) * (u32)a.row_bytes + piece * 16, whi = (u32)row_of(16 + wrow) * (u32)a.row_bytes + piece * 16;
    uint8_t *turn = reinterpret_cast<uint8_t *>(smem) + (size_t)BUFS * KW * MT * kRow * 2 + wave * 32 * kTurn, *turn_in = turn + wrow * kTurn + piece * 16;
    const uint8_t *turn_out = turn + col * kTurn + (EXACT ? h : 2 * h) * 16;
    const uint16_t *sbase = a.scales + (size_t)row0 * (a.K / 32);
    const u32 so = (u32)row_of(col) * (u32)(a.K / 32) + (FMT == FMT_Q4_0 && !EXACT ? 2 * h : 0), ho = (u32)row_of(col) * (u32)a.row_bytes;
    constexpr int PAIRS = pairs_of(FMT);
    uintx4 raw[PAIRS][2], next_q[2];            // the next step's stretches as they were loaded; turned: the next stretch, of the lane's own row
    uint4 q[2];                                 // the stretch in use
    auto load_pair = [&](int s, int j) __attribute__((always_inline)) {
        const uint8_t *from = wbase + (FMT == FMT_Q4_K ? (size_t)(at(s) >> 1) * 144 + 16 + (at(s) & 1) * 64 : (size_t)at(s) * (64 * PAIRS)) + 64 * j;
        raw[j][0] = *reinterpret_cast<const uintx4 *>(from + wlo);
        raw[j][1] = *reinterpret_cast<const uintx4 *>(from + whi);
    };
    // turned: stretch j of the step in raw becomes the next one, step `then` goes on its way
    auto turn_pair = [&](auto j_c, int then) __attribute__((always_inline)) {
        constexpr int j = decltype(j_c)::value;
        *reinterpret_cast<uintx4 *>(turn_in) = raw[j][0];
        *reinterpret_cast<uintx4 *>(turn_in + 16 * kTurn) = raw[j][1];
        load_pair(then, j);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // a wavefront's LDS operations keep their order
        __builtin_amdgcn_wave_barrier();
        next_q[0] = *reinterpret_cast<const uintx4 *>(turn_out);
        next_q[1] = *reinterpret_cast<const uintx4 *>(turn_out + (EXACT ? 32 : 16));
    };
    auto use_pair = [&](int j) __attribute__((always_inline)) {
        if constexpr (TURN) {
            q[0] = __builtin_bit_cast(uint4, next_q[0]);
            q[1] = __builtin_bit_cast(uint4, next_q[1]);
            return;
        }
        const uint4 loaded[2] = {__builtin_bit_cast(uint4, raw[j][0]), __builtin_bit_cast(uint4, raw[j][1])};
        exchange_rows(loaded, q);
        if constexpr (EXACT && FMT == FMT_Q4_0) {   // each half of a wavefront holds a block; it needs bytes 8 h .. of both
#pragma unroll
            for (int p = 0; p < 2; p++) {
                const auto e0 = __builtin_amdgcn_permlane32_swap(q[p].x, q[p].z, false, false);
                const auto e1 = __builtin_amdgcn_permlane32_swap(q[p].y, q[p].w, false, false);
                q[p] = make_uint4(e0[0], e1[0], e0[1], e1[1]);
            }
        }
    };
    auto load_scales = [&](int s) __attribute__((always_inline)) {   // Q4_0: blocks 2 h, 2 h + 1; Q8_0 and exact: all four
        uint2 d = {0, 0};
        if constexpr (EXACT) d = *reinterpret_cast<const uint2 *>(sbase + 4 * at(s) + so);
        else if constexpr (FMT == FMT_Q4_0) d.x = *reinterpret_cast<const u32 *>(sbase + 4 * at(s) + so);
        else if constexpr (FMT == FMT_Q8_0) d = *reinterpret_cast<const uint2 *>(sbase + 4 * at(s) + so);
        return d;
    };
    auto load_hdr = [&](int s) __attribute__((always_inline)) { return *reinterpret_cast<const uint4 *>(wbase + (size_t)(at(s) >> 1) * 144 + ho); };
    // where fragment g (0..7) of a step begins among its 128 k
    auto koff = [&](int g) {
        if constexpr (EXACT) return 32 * (g >> 1) + (FMT == FMT_Q4_0 ? 16 * (g & 1) + 8 * h : 16 * h + 8 * (g & 1));
        else return FMT == FMT_Q4_0 ? 64 * h + 8 * g : FMT == FMT_Q4_K ? 64 * h + 32 * (g & 1) + 8 * (g >> 1) : 64 * (g >> 2) + 32 * h + 8 * (g & 3);
    };

    floatx16 acc[TM];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = 0.0f;

    uint4 hdr[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};   // of this super-block and the next, by turns
    uint2 scale[2];                                // of this step and the next, by turns
    load_x(0);
#pragma unroll
    for (int j = 0; j < PAIRS; j++) load_pair(0, j);
    if constexpr (FMT == FMT_Q4_K) { hdr[0] = load_hdr(0); hdr[1] = load_hdr(2); }
    scale[0] = load_scales(0);
    store_x(0);
    load_x(1);
    scale[1] = load_scales(1);
    if constexpr (TURN) turn_pair(std::integral_constant<int, 0>{}, 1);
    __syncthreads();

    // eight weights of the lane's row as fp16
    auto decode = [&](const uint4 &head, const uint2 &scales, auto odd, int g) __attribute__((always_inline)) {
        if constexpr (EXACT) {   // fragment g % 2 of block g / 2: q - 8 or q
            const uint4 &v = q[FMT == FMT_Q4_0 ? g >> 2 : (g >> 1) & 1];
            const bool upper = FMT == FMT_Q4_0 ? g & 2 : g & 1;
            const u32 w[2] = {upper ? v.z : v.x, upper ? v.w : v.y};
            u32 o[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if constexpr (FMT == FMT_Q4_0) {
                    const u32 mask = g & 1 ? 0x00F000F0u : 0x000F000Fu, magic = g & 1 ? 0x54005400u : 0x64006400u;
                    const h2 off = g & 1 ? h2{(_Float16)72.0f, (_Float16)72.0f} : h2{(_Float16)1032.0f, (_Float16)1032.0f};
                    o[j] = as_u32(as_h2(((j & 1 ? w[j >> 1] >> 8 : w[j >> 1]) & mask) | magic) - off);
                } else {
                    const h2 off = {(_Float16)1152.0f, (_Float16)1152.0f};   // 1024 + 128
                    o[j] = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, w[j >> 1] ^ 0x80808080u, j & 1 ? 0x04030402u : 0x04010400u)) - off);
                }
            }
            return as_half8(make_uint4(o[0], o[1], o[2], o[3]));
        } else if constexpr (FMT == FMT_Q4_K) {
            // Sub-block 4 odd + 2 h + g % 2.  A nibble alone in sixteen bits is the fp16 number n 2^-24 (or 16 n 2^-24): n s - dm with product and
            // subtraction in fp32 and one rounding to fp16, as one v_fma_mix a weight.
            const float d = half_bits_to_float(head.x & 0xFFFFu), dmin = half_bits_to_float(head.x >> 16);
            const int sh = 16 * h + 8 * (g & 1);
            u32 sc, m;
            if constexpr (decltype(odd)::value == 0) { sc = (head.y >> sh) & 63u; m = (head.z >> sh) & 63u; }
            else {
                sc = ((head.w >> sh) & 0xFu) | (((head.y >> sh) & 0xC0u) >> 2);
                m = ((head.w >> (sh + 4)) & 0xFu) | (((head.z >> sh) & 0xC0u) >> 2);
            }
            const float s = d * (float)sc * (g & 1 ? 1048576.0f : 16777216.0f), dm = dmin * (float)m;
            const uint4 &v = q[g >> 2];
            const u32 w[2] = {g & 2 ? v.z : v.x, g & 2 ? v.w : v.y};
            const u32 mask = g & 1 ? 0x00F000F0u : 0x000F000Fu;
            u32 o[4];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const h2 even = as_h2(w[j] & mask), uneven = as_h2((w[j] >> 8) & mask);
                o[2 * j] = as_u32(h2{(_Float16)__builtin_fmaf((float)even.x, s, -dm), (_Float16)__builtin_fmaf((float)uneven.x, s, -dm)});
                o[2 * j + 1] = as_u32(h2{(_Float16)__builtin_fmaf((float)even.y, s, -dm), (_Float16)__builtin_fmaf((float)uneven.y, s, -dm)});
            }
            return as_half8(make_uint4(o[0], o[1], o[2], o[3]));
        } else if constexpr (FMT == FMT_Q4_0) {
            // (n - 8) * d from n under an fp16 exponent; elements of every four come out as 0, 2, 1, 3, like the activations'
            const h2 sc = splat_bits(g >> 2 ? scales.x >> 16 : scales.x & 0xFFFFu);
            const uint4 &v = q[g >> 2];
            const u32 w[2] = {g & 1 ? v.z : v.x, g & 1 ? v.w : v.y};
            const u32 mask = g & 2 ? 0x00F000F0u : 0x000F000Fu, magic = g & 2 ? 0x54005400u : 0x64006400u;
            const h2 off = g & 2 ? h2{(_Float16)72.0f, (_Float16)72.0f} : h2{(_Float16)1032.0f, (_Float16)1032.0f};
            u32 o[4];
#pragma unroll
            for (int j = 0; j < 4; j++) o[j] = as_u32((as_h2(((j & 1 ? w[j >> 1] >> 8 : w[j >> 1]) & mask) | magic) - off) * sc);
            return as_half8(make_uint4(o[0], o[1], o[2], o[3]));
        } else {
            const u32 pair = g >> 2 ? scales.y : scales.x;
            const h2 sc = splat_bits(h ? pair >> 16 : pair & 0xFFFFu), off = {(_Float16)1152.0f, (_Float16)1152.0f};   // 1024 + 128
            const uint4 &v = q[(g >> 1) & 1];
            const u32 w[2] = {(g & 1 ? v.z : v.x) ^ 0x80808080u, (g & 1 ? v.w : v.y) ^ 0x80808080u};
            u32 o[4];
#pragma unroll
            for (int j = 0; j < 4; j++) o[j] = as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, w[j >> 1], j & 1 ? 0x04030402u : 0x04010400u)) - off) * sc);
            return as_half8(make_uint4(o[0], o[1], o[2], o[3]));
        }
    };
    constexpr int VALU = 16;   // of a fragment, to be spread over its products
    auto step = [&](auto slot_c, int s) __attribute__((always_inline)) {   // slot: s % 4: the buffers by turns, half of a super-block, super-blocks by turns
        constexpr int S = decltype(slot_c)::value & 1, H = decltype(slot_c)::value >> 1;
        constexpr std::integral_constant<int, S> odd{};
        constexpr int B = BUFS == 2 ? S : 0;
        const _Float16 *xb = xt + B * MT * kRow + col * kRow;
        half8 xf[2][TM], wf[2];
        auto fragments = [&](int g) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < TM; i++) xf[g & 1][i] = *reinterpret_cast<const half8 *>(xb + 32 * i * kRow + koff(g));
            if (g % (8 / PAIRS) == 0) {   // a stretch is taken into use, the next step's goes on its way
                use_pair(g / (8 / PAIRS));
                if constexpr (!TURN) load_pair(s + 1, g / (8 / PAIRS));
            }
            if constexpr (TURN) if (PAIRS == 2 && g == 3) turn_pair(std::integral_constant<int, PAIRS - 1>{}, s + 1);
            wf[g & 1] = decode(hdr[H], scale[S], odd, g);
        };
        fragments(0);
        if constexpr (BUFS == 2) {
            store_x(S ^ 1);        // the next step's activations; that buffer was last read before the last barrier
            load_x(s + 2);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (EXACT) {
            const floatx16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            floatx16 part[2][TM];   // a block's sums, scaled while the next block is multiplied
            auto fold = [&](int b) __attribute__((always_inline)) {
                const u32 pair = b >> 1 ? scale[S].y : scale[S].x;
                const float d = half_bits_to_float(b & 1 ? pair >> 16 : pair & 0xFFFFu);
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[i][r] = __builtin_fmaf(d, part[b & 1][i][r], acc[i][r]);
            };
#pragma unroll
            for (int g = 0; g < 8; g++) {
                if (g + 1 < 8) fragments(g + 1);
                else if constexpr (TURN) turn_pair(std::integral_constant<int, 0>{}, s + 2);
#pragma unroll
                for (int i = 0; i < TM; i++) part[(g >> 1) & 1][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[g & 1][i], wf[g & 1], g & 1 ? part[(g >> 1) & 1][i] : zero16, 0, 0, 0);
                if (g >= 2 && !(g & 1)) fold((g >> 1) - 1);
            }
            fold(3);
        } else
#pragma unroll
        for (int g = 0; g < 8; g++) {
            if (g + 1 < 8) fragments(g + 1);
            else if constexpr (TURN) turn_pair(std::integral_constant<int, 0>{}, s + 2);
#pragma unroll
            for (int i = 0; i < TM; i++) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[g & 1][i], wf[g & 1], acc[i], 0, 0, 0);
            if (g + 1 < 8) {
#pragma unroll
                for (int i = 0; i < TM; i++) {   // in this order: a product, a read, a share of the unpacking
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, (VALU + TM - 1) / TM, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        scale[S] = load_scales(s + 2);
        if constexpr (FMT == FMT_Q4_K && S == 1) hdr[H] = load_hdr(s + 3);
        __syncthreads();
        if constexpr (BUFS == 1) {
            store_x(0);
            load_x(s + 2);
            __syncthreads();
        }
    };
    int s = 0;
    for (; s + 4 <= own; s += 4) {
        step(std::integral_constant<int, 0>{}, s);
        step(std::integral_constant<int, 1>{}, s + 1);
        step(std::integral_constant<int, 2>{}, s + 2);
        step(std::integral_constant<int, 3>{}, s + 3);
    }
    if (s < own) step(std::integral_constant<int, 0>{}, s);
    if (s + 1 < own) step(std::integral_constant<int, 1>{}, s + 1);
    if (s + 2 < own) step(std::integral_constant<int, 2>{}, s + 2);
    for (s = own; s < a.per; s++) {
        __syncthreads();
        if constexpr (BUFS == 1) __syncthreads();
    }

    auto out_row = [&](int r) { return m0 + tile_row(r, h); };
    constexpr int SHARE = TM * 16 / KW;        // accumulators that a wavefront finishes
    float v[SHARE];
    const int r0 = KW == 1 ? 0 : wk * SHARE;
    share_sums<TM, NW>(acc, reinterpret_cast<float *>(smem), wave, wn, lane, r0, v);
    if (a.swiglu_out) {
#pragma unroll
        for (int k = 0; k < SHARE / 2; k++) {
            const bool odd = lane & 1;
            float g, u;
            gate_and_up(v[2 * k], v[2 * k + 1], odd, g, u);
            const int m = out_row(r0 + 2 * k + (odd ? 1 : 0));
            if (m < a.M && (n | 1) < a.N) {
                a.swiglu_out[(size_t)m * (a.N / 2) + n / 2] = __builtin_bit_cast(uint16_t, (_Float16)__fmul_rn(silu(g), u));
            }
        }
        return;
    }
    float *out = a.splits > 1 ? a.partial + (size_t)split * a.M * a.N : a.y;
    const bool whole = m0 + MT <= a.M && n0 + 32 <= a.N;
    if (a.splits == 1 && a.residual) {
        // requested together: y may be the residual's own memory, and a load behind each store is a trip to memory each
#pragma unroll
        for (int r = 0; r < SHARE; r++) v[r] += a.residual[(size_t)(out_row(r0 + r) < a.M ? out_row(r0 + r) : a.M - 1) * a.N + (n < a.N ? n : a.N - 1)];
    }
    if (whole) {
#pragma unroll
        for (int r = 0; r < SHARE; r++) out[(size_t)out_row(r0 + r) * a.N + n] = v[r];
    } else {
#pragma unroll
        for (int r = 0; r < SHARE; r++) if (out_row(r0 + r) < a.M && n < a.N) out[(size_t)out_row(r0 + r) * a.N + n] = v[r];
    }
}

// TS < TM: two heights of tiles in one launch, the long ones first (no shares of K).
template <int FMT, int TM, int NW, bool EXACT = false, int TS = TM>
__global__ __launch_bounds__(kThreads) void block_gemm_kernel(BlockArgs a) {
    extern __shared__ uint4 smem[];
    if constexpr (TS == TM) {
        const auto [m_tile, n_tile, split] = place_of(a.m_tiles, a.n_tiles);
        block_product<FMT, TM, NW, EXACT>(a, m_tile * 32 * TM, n_tile, split, smem);
    } else {
        const int longs = a.long_tiles * a.n_tiles;
        if ((int)blockIdx.x < longs) {
            const auto [m_tile, n_tile, split] = place_of(a.long_tiles, a.n_tiles, blockIdx.x, longs);
            block_product<FMT, TM, NW, EXACT>(a, m_tile * 32 * TM, n_tile, 0, smem);
        } else {
            const auto [m_tile, n_tile, split] = place_of(a.m_tiles - a.long_tiles, a.n_tiles, blockIdx.x - longs, gridDim.x - longs);
            block_product<FMT, TS, NW, EXACT>(a, a.long_tiles * 32 * TM + m_tile * 32 * TS, n_tile, 0, smem);
        }
    }
}

template <int FMT, int TM, int NW, bool EXACT, int TS = TM>
hipError_t launch(const BlockArgs &a, hipStream_t stream) {
    static std::atomic<uint64_t> raised{0};
    constexpr size_t one = block_lds_bytes<FMT, TM, NW>(), other = block_lds_bytes<FMT, TS, NW>(), lds = one > other ? one : other;
    const hipError_t err = raise_lds_limit(reinterpret_cast<const void *>(block_gemm_kernel<FMT, TM, NW, EXACT, TS>), lds, raised);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL((block_gemm_kernel<FMT, TM, NW, EXACT, TS>), dim3(a.n_tiles * a.m_tiles * a.splits), dim3(kThreads), lds, stream, a);
    return hipGetLastError();
}

template <int FMT, int TM, bool EXACT = false>
hipError_t launch_width(int nw, const BlockArgs &a, hipStream_t stream) {
    if (nw == 8) return launch<FMT, TM, 8, EXACT>(a, stream);
    if (nw == 4) return launch<FMT, TM, 4, EXACT>(a, stream);
    if constexpr (TM < 4) return launch<FMT, TM, 2, EXACT>(a, stream);   // 128 activation rows for each of four groups: more registers than there are
    return hipErrorInvalidValue;
}
template <int FMT>
hipError_t launch_format(int tm, int nw, bool exact, const BlockArgs &a, hipStream_t stream) {
    if (a.long_tiles) return tm == 4 ? launch<FMT, 4, 8, false, 2>(a, stream) : launch<FMT, 3, 8, false, 2>(a, stream);
    if constexpr (FMT == FMT_Q8_0 || FMT == FMT_Q4_0) if (exact) return launch_width<FMT, 1, true>(nw, a, stream);
    switch (tm) {
    case 1: return launch_width<FMT, 1>(nw, a, stream);
    case 2: return launch_width<FMT, 2>(nw, a, stream);
    case 3: return launch_width<FMT, 3>(nw, a, stream);
    default: return launch_width<FMT, 4>(nw, a, stream);
    }
}

struct Form { int tm = 0, nw = 0, per = 0, splits = 0, long_tiles = 0; };   // long_tiles: tiles of tm * 32 rows, tiles of 64 behind them
std::atomic<int> g_block_gemm_form{0};

// The form (rows of a tile, wavefronts along the weights, shares of K) by its expected time: rounds of one workgroup per compute unit, a step of a round growing with the tile's rows and
// with the groups that each stage their own activations, and the bytes of the planes, which the next kernel reads once more (behind a SiLU, and where no
// caller adds them, a launch of its own: 1.6 to 4.3 us; the form that rule chooses is 1 % off the best on average, 11 at worst, 256 x 256).  The
// constants are fitted to 10 000 launches (sixteen shapes of 576 to 32000 weight rows and 768 to 14336 columns, 12 to 512 rows) and are off by 6 % at the
// median; what the rule chooses takes 1.4 % longer than the best form, 4 % at worst.
Form choose_form(const GemmParams &p, bool exact) {
    const int fmt = p.w.format, N = p.w.rows, M = p.rows, unit = fmt == FMT_Q4_K ? 2 : 1, units = p.w.cols / (kStep * unit);
    const float start = 2.25f, fill = 1.34f, step = 0.743f, row_tile = 0.149f, staged = 0.1f, join = 0.383f;
    const float plane_us = 0.28f, again_us = 0.2f;   // per MB
    static const int kSplits[] = {1, 2, 3, 4, 6, 8};
    const int cus = device_compute_units() > 0 ? device_compute_units() : 256;
    Form best;
    float best_us = 0.0f;
    auto group = [&](int per, int tm, int kw) { return per * unit * (step + tm * (row_tile + staged * kw)) + fill + (kw > 1 ? join * tm : 0.0f); };   // one workgroup
    for (int tm = 1; tm <= (exact ? 1 : 4) && tm <= (M + 31) / 32; tm++)
        for (int nw = tm < 4 ? 2 : 4; nw <= 8; nw *= 2)
            for (int want : kSplits) {
                const int kw = kWaves / nw;
                const auto [per, splits] = shares_of(units, nw, want);
                const float mb = (float)splits * (float)M * (float)N * 4e-6f;
                if (splits != want || (splits > 1 && (!p.workspace || (size_t)splits * M * N > p.workspace_floats))) continue;
                const long wgs = (long)((N + 32 * nw - 1) / (32 * nw)) * ((M + 32 * tm - 1) / (32 * tm)) * splits;
                const float rounds = (float)((wgs + cus - 1) / cus);
                float us = start + rounds * group(per, tm, kw) + plane_us * mb;
                if (splits > 1) us += again_us * mb + (p.swiglu_out ? 3.0f : p.deferred_splits ? 1.0f : 1.6f + 0.2f * splits);
                if (!best.tm || us < best_us) { best = Form{tm, nw, per * unit, splits}; best_us = us; }
            }
    // Several rounds of tiles whose last one is nearly empty: tiles of 64 rows at the end, which each compute unit takes as it comes free.  us, one height -> two: 16384 x 3072 Q4_K, 600 / 1200 / 1600 /
    // 1777 rows 100.0 / 174.2 / 224.9 / 233.7 -> 92.2 / 162.1 / 213.2 / 225.4;  28672 x 4096 Q4_0, 300 / 600 / 1200 rows 116.7 / 196.7 / 339.7 -> 104.8 / 184.2 / 327.3;  6144 x 4096 Q4_0, 1400 / 1600 rows
    // 105.5 / 117.8 -> 103.8 / 107.0.  Less than two per cent in the rule's own time is not taken.
    for (int tm = 3; tm <= 4 && !exact && best.splits == 1; tm++) {
        const int n_tiles = (N + 255) / 256;
        const float along = group(units, tm, 1), ashort = group(units, 2, 1);
        for (int longs = 1; 32 * tm * longs < M; longs++) {
            int shorts = n_tiles * ((M - 32 * tm * longs + 63) / 64);
            const int full = n_tiles * longs / cus, ahead = n_tiles * longs % cus;
            float early = full * along, late = (full + (ahead ? 1 : 0)) * along;
            for (; shorts > 0;) {
                const bool at_early = early <= late || !ahead;
                shorts -= at_early ? cus - ahead : ahead;
                (at_early ? early : late) += ashort;
            }
            const float us = start + (early > late ? early : late) + plane_us * (float)M * (float)N * 4e-6f;
            if (us < 0.98f * best_us) { best = Form{tm, 8, units * unit, 1, longs}; best_us = us; }
        }
    }
    return best;
}

}  // namespace

void block_gemm_set_form(int form) {
    const int longs = form / 1000, tm = form / 100 % 10, nw = form / 10 % 10, shares = form % 10;
    const bool known = (longs == 0 || (tm >= 3 && nw == 8 && shares == 1)) && tm >= 1 && tm <= 4 && (nw == 4 || nw == 8 || (nw == 2 && tm < 4)) && shares >= 1;
    g_block_gemm_form.store(known ? form : 0);
}

bool block_gemm_by_size() { return g_block_gemm_form.load() == 0; }

// Products of 2048 columns and more that steps with exact weights ask for, in shares of K that the next kernel adds: up to 32 rows, and what is small (beyond it weights are
// rounded).  Against rows_gemm.hip, whose wavefronts walk more of K each, 2560 x 2048, 4 / 31 / 93 rows: Q8_0 8.0 / 9.5 / 9.9 -> 6.2 / 6.4 / 7.8 us, Q4_0 6.8 / 8.2 / 8.4 -> 5.3 / 5.5 /
// 6.7;  2048 x 2048, 64 / 128 rows: Q8_0 9.6 / 9.9 -> 6.5 / 7.7, Q4_0 8.2 / 8.5 -> 5.8 / 6.8.  Of what the launch gains the next kernel takes 1.5 to 2.5 us for the planes, so whole
// layers decide (q|k|v and wo in shares, a feed-forward of four times the width; us a layer, one launch -> shares): 2048 columns, 12 / 31 / 48 rows Q8_0 65.5 / 74.6 / 75.8 -> 63.3 / 67.6 /
// 71.6, Q4_0 60 / 66 / 67 -> 58 / 60 / 63;  2560 columns Q8_0 87.2 / 96.9 / 98.6 -> 83.5 / 91.2 / 97.0;  3072 columns Q8_0 96.2 / 102.6 / 105.3 -> 94.5 / 97.1 / 104.6.  Rows that are no
// multiple of 512 columns spread better over the memory's channels there and gain up to 32 rows only: 2816 columns Q8_0 88.7 / 96.0 / 99.0 -> 89.7 / 92.7 / 100.0, Q4_0 76.8 / 84.4 / 84.8 ->
// 79.5 / 80.7 / 85.6.
// Behind a SiLU the shares cost a launch, so there only up to 32 rows.  Matrices of fewer weight rows stay where they are beyond 32: the launch alone would be shorter (512 to 1792 rows,
// 40 / 128 rows of 2048 columns: Q8_0 9.3 / 9.5 -> 6.0 to 6.3 / 6.1 to 7.6, Q4_0 7.6 to 8 / 7.8 to 8.2 -> 5.0 to 5.4 / 5.2 to 6.7), but most of it goes into the planes, and calls of 48
// tokens of a six-layer model of 768 columns differ by less than their 3 % noise.
// Where no caller adds the shares, their launch outweighs them as long as the other kernel's workgroups are resident at once (with that launch, 8 rows Q4_0: 2048 x 2048 8.6 us, 6.7
// there; 3072 x 3072 9.4, 7.4; 5632 x 2048 10.3, 6.9; 8192 x 3072 10.5, 9.2; 11264 x 2048 9.8, 12.6).
bool block_gemm_keeps(const GemmParams &p) {
    if ((p.w.format != FMT_Q8_0 && p.w.format != FMT_Q4_0) || p.w.cols < 2048 || p.w.cols % kStep != 0 || !p.unrounded) return false;
    const long row_blocks = (p.rows + 31) / 32, groups = (long)((p.w.rows + 31) / 32) * row_blocks;
    if (block_gemm_alone(p) && groups <= (device_compute_units() > 0 ? device_compute_units() : 256)) return false;
    if (p.w.cols <= 3072 && p.w.cols % 512 != 0 && (p.rows <= 16 || row_blocks > 1)) return false;
    return row_blocks == 1 || (row_blocks <= 4 && !p.swiglu_out && p.w.rows >= 2048 && p.w.cols <= 3072 && groups * (p.w.cols / 64) <= 8192);
}

// Few rows keep their weights exact where a format has one scale per block and the steps they stand for do: the same time for Q8_0, 0 to 12 % more for Q4_0 (12 rows; with shares
// added by the next kernel 2048 x 8192, 4 to 31 rows 7.3 to 7.8 us, in rows_gemm.hip 13 to 17).
bool block_gemm_exact(const GemmParams &p) {
    return (p.w.format == FMT_Q8_0 || p.w.format == FMT_Q4_0) && p.unrounded && (p.rows <= 32 || block_gemm_keeps(p));
}

bool block_gemm_exact(const DeviceMatrix &w, int rows) {
    return w.format == FMT_F16 || ((w.format == FMT_Q8_0 || w.format == FMT_Q4_0) && w.cols % kStep == 0 && rows <= 32);
}

bool block_gemm_takes(const GemmParams &p) {
    const int fmt = p.w.format;
    return (fmt == FMT_Q4_K || fmt == FMT_Q4_0 || fmt == FMT_Q8_0) && p.w.cols % (fmt == FMT_Q4_K ? 256 : kStep) == 0;
}

hipError_t launch_block_gemm(const GemmParams &p, int *splits, hipStream_t stream) {
    bool exact = block_gemm_exact(p);
    Form f = choose_form(p, exact);
    if (const int forced = g_block_gemm_form.load(); forced > 0) {   // long tiles * 1000 + tm * 100 + nw * 10 + shares of K
        f.tm = forced / 100 % 10; f.nw = forced / 10 % 10;
        f.long_tiles = forced / 1000 * 32 * f.tm < p.rows ? forced / 1000 : 0;
        exact = exact && f.tm == 1;   // forms of more row tiles have no exact kernel
        const int unit = p.w.format == FMT_Q4_K ? 2 : 1;
        const Shares shares = shares_of(p.w.cols / (kStep * unit), f.nw, forced % 10);
        f.per = shares.per * unit; f.splits = shares.splits;
        if (f.splits > 1 && (!p.workspace || (size_t)f.splits * p.rows * p.w.rows > p.workspace_floats)) return hipErrorInvalidValue;
    }
    BlockArgs a{p.w.qs, p.w.scales, p.w.qs_row_bytes, p.w.rows, p.w.cols, p.rows, p.x, p.y, p.residual, p.workspace, f.splits == 1 && p.w.rows % 2 == 0 ? p.swiglu_out : nullptr, f.per, f.splits,
                (p.w.rows + 32 * f.nw - 1) / (32 * f.nw), f.long_tiles ? f.long_tiles + (p.rows - 32 * f.tm * f.long_tiles + 63) / 64 : (p.rows + 32 * f.tm - 1) / (32 * f.tm), f.long_tiles};
    *splits = f.splits;
    switch (p.w.format) {
    case FMT_Q4_K: return launch_format<FMT_Q4_K>(f.tm, f.nw, false, a, stream);
    case FMT_Q4_0: return launch_format<FMT_Q4_0>(f.tm, f.nw, exact, a, stream);
    default: return launch_format<FMT_Q8_0>(f.tm, f.nw, exact, a, stream);
    }
}

}  // namespace esp
