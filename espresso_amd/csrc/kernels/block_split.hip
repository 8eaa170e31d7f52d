// y[m][n] = sum_k x[m][k] * W[n][k] for blocks of split rows (SplitRowsView) and Q4_K weights, exact as in gemm_split.hip: integers sc q on the matrix cores, the hi plane against
// them and the lo plane against them / 2048 into one set of sums, d and the minimums' product once per super-block.
//
// The shape is that of block_gemm.hip: eight wavefronts, NW of them along the weights and 8 / NW sharing K, each with 32 weight rows and all 32 TM activation rows; weights go
// from memory into the registers that multiply them, read row by row from the packed matrix (no tiled copy is needed), both planes through LDS.  Two wavefronts on every SIMD, and
// K shared inside a workgroup, are what the narrow forms of gemm_q4k_split_regb_kernel lack: one wavefront per SIMD walks all of K behind a SiLU, which planes cannot split.
// What bounds it: the weights' way from memory for few rows, the matrix cores and the fold (two multiply-adds a sum and super-block, and one product per row tile for the minimums) for many.  Against those forms, us:
//   gate|up 28672 x 4096, 8 / 31 / 60 rows 48 / 48 / 58 -> 29 / 33 / 56;  16384 x 2048, 8 / 31 / 60 / 128 rows 25 / 25 / 26 / 31 -> 13 / 14 / 18 / 28;
//   6144 x 4096, 31 / 256 / 480 rows and their planes 14.1 / 49.9 / 76.9 -> 12.9 / 40.7 / 67.4;  4096 x 14336, 256 rows 82 -> 76.
// Kept out: 128 rows a workgroup and 96 for two groups (264 and 92 bytes of scratch a lane), the activations on their way to LDS as uint4 (they stay in scratch: 8 rows of
// 16384 x 2048 32 us).  With one row tile the activation fragments are read three ahead (one ahead: 42 us for 8 rows of 28672 x 4096 with eight wavefronts along the weights, 62).
#include "../common.h"
#include "block_split.h"
#include "block_tile.h"
#include "silu.h"
#include "split_rows.h"
#include <type_traits>

namespace esp {
namespace {

using split_rows::kScale;
using split_rows::kUnscale;
using namespace block_tile;
typedef u32 quad __attribute__((ext_vector_type(4)));

struct BlockSplitArgs {
    const uint8_t *qs;
    size_t row_bytes;
    int N, K, M;
    const uint16_t *xh, *xl, *xs;
    float *y;
    const float *residual;
    float *partial;
    uint16_t *sw_hi, *sw_lo, *sw_sums;
    int per, splits, n_tiles, m_tiles;   // per: steps of one group of wavefronts, an even number
};

__device__ __forceinline__ u32 dword_of(const uint4 &v, int k) { return k == 0 ? v.x : k == 1 ? v.y : k == 2 ? v.z : v.w; }

constexpr size_t split_tile_bytes(int tm, int nw) { return (size_t)(kWaves / nw) * 2 * 32 * tm * kRow * 2; }   // a step of all groups
constexpr int split_buffers(int tm, int nw) { return 2 * split_tile_bytes(tm, nw) <= 160 * 1024 ? 2 : 1; }
constexpr size_t split_lds_bytes(int tm, int nw) {
    const size_t x = split_buffers(tm, nw) * split_tile_bytes(tm, nw), sums = kWaves / nw > 1 ? (size_t)kWaves * tm * 16 * 64 * 4 : 0, act = 2 * (size_t)32 * tm * (16 * nw + 8) * 2;
    return x > sums ? (x > act ? x : act) : sums > act ? sums : act;
}

template <int TM, int NW>
__global__ __launch_bounds__(kThreads) void block_split_kernel(BlockSplitArgs a) {
    constexpr int KW = kWaves / NW, MT = 32 * TM, GT = 64 * NW, BUFS = split_buffers(TM, NW);
    constexpr int XP = MT * (kStep / 8) / GT;       // sixteen-byte pieces of a plane per thread and step
    static_assert(MT * (kStep / 8) % GT == 0 && XP >= 1, "whole pieces");
    extern __shared__ uint4 smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, col = lane & 31;
    const int wn = wave % NW, wk = wave / NW, gtid = wn * 64 + lane;
    const auto [m_tile, n_tile, split] = place_of(a.m_tiles, a.n_tiles);
    const int m0 = m_tile * MT, n0 = (n_tile * NW + wn) * 32, n = n0 + col;
    const int row0 = n0 < a.N ? n0 : a.N - 1;
    auto row_of = [&](int r) { return row0 + r < a.N ? r : a.N - 1 - row0; };   // rows from row0 on, clamped: those beyond are never stored
    const int all = a.K / kStep, sbs = a.K / 256, s0 = (split * KW + wk) * a.per, own = all - s0 < a.per ? (all > s0 ? all - s0 : 0) : a.per;
    auto at = [&](int s) { return s0 + s < all ? s0 + s : all - 1; };          // steps past the end repeat the last: in bounds, never used

    _Float16 *xt = reinterpret_cast<_Float16 *>(smem) + wk * BUFS * 2 * MT * kRow;   // [BUFS][plane][MT][kRow]
    quad hi_x[XP], lo_x[XP];                   // (as uint4, a structure, they stay in scratch memory)
    u32 xo[XP];                                // elements from row m0 on
#pragma unroll
    for (int i = 0; i < XP; i++) {
        const int piece = gtid + i * GT, r = piece >> 4, part = piece & 15;
        xo[i] = (u32)(m0 + r < a.M ? r : a.M - 1 - m0) * (u32)a.K + part * 8;
    }
    const uint16_t *hbase = a.xh + (size_t)m0 * a.K, *lbase = a.xl + (size_t)m0 * a.K;
    auto load_x = [&](int s) __attribute__((always_inline)) {
        const size_t o = (size_t)at(s) * kStep;
#pragma unroll
        for (int i = 0; i < XP; i++) {
            hi_x[i] = *reinterpret_cast<const quad *>(hbase + o + xo[i]);
            lo_x[i] = *reinterpret_cast<const quad *>(lbase + o + xo[i]);
        }
    };
    auto store_x = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < XP; i++) {
            const int piece = gtid + i * GT, r = piece >> 4, part = piece & 15;
            *reinterpret_cast<quad *>(xt + 2 * buf * MT * kRow + r * kRow + part * 8) = hi_x[i];
            *reinterpret_cast<quad *>(xt + (2 * buf + 1) * MT * kRow + r * kRow + part * 8) = lo_x[i];
        }
    };
    // weights (exchange_rows): the two pieces of the pair of sub-blocks h end up in each lane of the row
    const int piece = lane >> 4;
    const uint8_t *wbase = a.qs + (size_t)row0 * a.row_bytes;
    const u32 wlo = (u32)row_of(lane & 15) * (u32)a.row_bytes + piece * 16, whi = (u32)row_of(16 + (lane & 15)) * (u32)a.row_bytes + piece * 16, ho = (u32)row_of(col) * (u32)a.row_bytes;
    uint4 raw[2], q[2];
    auto load_pair = [&](int s) __attribute__((always_inline)) {
        const uint8_t *from = wbase + (size_t)(at(s) >> 1) * 144 + 16 + (at(s) & 1) * 64;
        raw[0] = *reinterpret_cast<const uint4 *>(from + wlo);
        raw[1] = *reinterpret_cast<const uint4 *>(from + whi);
    };
    auto load_hdr = [&](int s) __attribute__((always_inline)) { return *reinterpret_cast<const uint4 *>(wbase + (size_t)(at(s) >> 1) * 144 + ho); };
    // the rows' sums over the sub-blocks of a super-block: (8 x hi, 8 x lo) of sums
    u32 so[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) so[i] = (u32)(m0 + 32 * i + col < a.M ? 32 * i + col : a.M - 1 - m0) * (u32)(sbs * 16) + 8 * h;
    const uint16_t *sbase = a.xs + (size_t)m0 * sbs * 16;
    half8 fs[TM];
    auto load_sums = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; i++) fs[i] = *reinterpret_cast<const half8 *>(sbase + (size_t)(at(s) >> 1) * 16 + so[i]);
    };
    auto koff = [&](int g) { return 64 * h + 32 * (g & 1) + 8 * (g >> 1); };   // where fragment g (0..7) of a step begins among its 128 k

    const floatx16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    floatx16 tot[TM], acc[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) { tot[i] = zero16; acc[i] = zero16; }
    // constants of the nibble trick, hidden from the optimiser so that (w & mask) | magic stays one v_and_or_b32
    u32 mask_lo = 0x000F000Fu, mask_hi = 0x00F000F0u, magic_lo = 0x64006400u, magic_hi = 0x54005400u;
    asm volatile("" : "+s"(mask_lo), "+s"(mask_hi));
    asm volatile("" : "+v"(magic_lo), "+v"(magic_hi));

    uint4 hdr[2];                                  // of this super-block and the next, by turns
    load_x(0);
    load_pair(0);
    hdr[0] = load_hdr(0); hdr[1] = load_hdr(2);
    store_x(0);
    load_x(1);
    __syncthreads();

    // eight integers sc q of the lane's row, sub-block 4 odd + 2 h + g % 2, in the planes' order inside fours
    auto decode = [&](const uint4 &head, auto odd, int g) __attribute__((always_inline)) {
        const int sh = 16 * h + 8 * (g & 1);
        u32 sc;
        if constexpr (decltype(odd)::value == 0) sc = (head.y >> sh) & 63u;
        else sc = ((head.w >> sh) & 0xFu) | (((head.y >> sh) & 0xC0u) >> 2);
        const _Float16 s1 = (_Float16)(unsigned short)sc;
        const h2 mul = {s1, s1}, add = mul * (g & 1 ? h2{(_Float16)-64.0f, (_Float16)-64.0f} : h2{(_Float16)-1024.0f, (_Float16)-1024.0f});
        const u32 mask = g & 1 ? mask_hi : mask_lo, magic = g & 1 ? magic_hi : magic_lo;
        const uint4 &v = q[g >> 2];
        const u32 w[2] = {g & 2 ? v.z : v.x, g & 2 ? v.w : v.y};
        u32 o[4];
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] = as_u32(__builtin_elementwise_fma(as_h2(((j & 1 ? w[j >> 1] >> 8 : w[j >> 1]) & mask) | magic), mul, add));
        return make_uint4(o[0], o[1], o[2], o[3]);
    };
    auto step = [&](auto slot_c, int s) __attribute__((always_inline)) {   // slot: s % 4: the buffers by turns, half of a super-block, super-blocks by turns
        constexpr int S = decltype(slot_c)::value & 1, H = decltype(slot_c)::value >> 1, B = BUFS == 2 ? S : 0;
        constexpr std::integral_constant<int, S> odd{};
        const _Float16 *xb = xt + B * 2 * MT * kRow + col * kRow;
        constexpr int D = TM == 1 ? 4 : 2;                             // activation fragments are read D - 1 ahead
        half8 xf[D][TM];
        uint4 wq[2];
        auto read = [&](int v) __attribute__((always_inline)) {        // v: fragment v / 2, plane v % 2, whose weights are 2048 times smaller
#pragma unroll
            for (int i = 0; i < TM; i++) xf[v & (D - 1)][i] = *reinterpret_cast<const half8 *>(xb + (v & 1) * MT * kRow + 32 * i * kRow + koff(v >> 1));
        };
        auto unpack = [&](int v) __attribute__((always_inline)) {
            if (v == 0) {
                exchange_rows(raw, q);
                load_pair(s + 1);
            }
            if (!(v & 1)) wq[0] = decode(hdr[H], odd, v >> 1);
            else {
                const h2 k = {(_Float16)kUnscale, (_Float16)kUnscale};
                wq[1] = make_uint4(as_u32(as_h2(wq[0].x) * k), as_u32(as_h2(wq[0].y) * k), as_u32(as_h2(wq[0].z) * k), as_u32(as_h2(wq[0].w) * k));
            }
        };
#pragma unroll
        for (int v = 0; v < D - 1; v++) read(v);
        unpack(0);
        if constexpr (S == 0) load_sums(s);
        if constexpr (BUFS == 2) {
            store_x(S ^ 1);        // the next step's activations; that buffer was last read before the last barrier
            load_x(s + 2);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const half8 w = as_half8(wq[v & 1]);
            if (v + D - 1 < 16) read(v + D - 1);
            if (v + 1 < 16) unpack(v + 1);
#pragma unroll
            for (int i = 0; i < TM; i++) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[v & (D - 1)][i], w, S == 0 && v == 0 ? zero16 : acc[i], 0, 0, 0);
            if (v + 1 < 16) {
#pragma unroll
                for (int i = 0; i < TM; i++) {   // in this order: a product, a read, a share of the unpacking
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, (8 + TM - 1) / TM, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (S == 1) {    // the super-block's fold: d times its sums less dmin sum_j m_j S_j, one product against (m_0..m_7) and (m_0..m_7) / 2048
            const u32 low = hdr[H].z & 0x3F3F3F3Fu, high = ((hdr[H].w >> 4) & 0x0F0F0F0Fu) | ((hdr[H].z >> 2) & 0x30303030u);
            const _Float16 f = (_Float16)(h ? kUnscale : 1.0f);
            const h2 off = {(_Float16)1024.0f, (_Float16)1024.0f}, k = {f, f};
            const uint4 mq = make_uint4(as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, low, 0x04010400u)) - off) * k), as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, low, 0x04030402u)) - off) * k),
                                        as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, high, 0x04010400u)) - off) * k), as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, high, 0x04030402u)) - off) * k));
            const float d = half_bits_to_float(hdr[H].x & 0xFFFFu), dmin = half_bits_to_float(hdr[H].x >> 16);
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const floatx16 am = __builtin_amdgcn_mfma_f32_32x32x16_f16(fs[i], as_half8(mq), zero16, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; r++) tot[i][r] = __builtin_fmaf(-dmin, am[r], __builtin_fmaf(d, acc[i][r], tot[i][r]));
            }
            hdr[H] = load_hdr(s + 3);
        }
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
    if (s < own) {
        step(std::integral_constant<int, 0>{}, s);
        step(std::integral_constant<int, 1>{}, s + 1);
    }
    for (s = own; s < a.per; s++) {   // every group of wavefronts passes the same barriers
        __syncthreads();
        if constexpr (BUFS == 1) __syncthreads();
    }

    constexpr int SHARE = TM * 16 / KW;        // accumulators that a wavefront finishes
    float v[SHARE];
    const int r0 = KW == 1 ? 0 : wk * SHARE;
    share_sums<TM, NW>(tot, reinterpret_cast<float *>(smem), wave, wn, lane, r0, v);
    if (a.sw_hi) {   // the units leave through LDS
        constexpr int LD = 16 * NW + 8, RP = 2 * NW;   // units between rows, sixteen-byte pieces of a row
        uint16_t *hi = reinterpret_cast<uint16_t *>(smem), *lo = hi + MT * LD;
        if constexpr (KW > 1) __syncthreads();
        const bool odd = lane & 1;
        const int u = (32 * wn + col) >> 1, slot = u & 3, at_u = (u & ~3) + (slot == 1 ? 2 : slot == 2 ? 1 : slot);   // the planes' order inside fours: 0, 2, 1, 3
#pragma unroll
        for (int k = 0; k < SHARE / 2; k++) {
            float g, up;
            gate_and_up(v[2 * k], v[2 * k + 1], odd, g, up);
            const float act = __fmul_rn(silu(g), up);
            const int o = tile_row(r0 + 2 * k + (odd ? 1 : 0), h) * LD + at_u;
            const _Float16 top = (_Float16)act;
            hi[o] = __builtin_bit_cast(uint16_t, top);
            lo[o] = __builtin_bit_cast(uint16_t, (_Float16)__fmul_rn(__fsub_rn(act, (float)top), kScale));
        }
        __syncthreads();
        const int units = a.N / 2, unit0 = n_tile * NW * 16;
        for (int p = threadIdx.x; p < MT * RP; p += kThreads) {   // units is a multiple of 32: the four lanes of a sub-block are in or out together
            const int row = p / RP, c8 = (p % RP) * 8, m = m0 + row;
            if (m >= a.M || unit0 + c8 >= units) continue;
            const uint4 hv = *reinterpret_cast<const uint4 *>(hi + row * LD + c8), lv = *reinterpret_cast<const uint4 *>(lo + row * LD + c8);
            const size_t o = (size_t)m * units + unit0 + c8;
            *reinterpret_cast<uint4 *>(a.sw_hi + o) = hv;
            *reinterpret_cast<uint4 *>(a.sw_lo + o) = lv;
            float sum = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const h2 hp = as_h2(dword_of(hv, e)), lp = as_h2(dword_of(lv, e));
                sum += __builtin_fmaf((float)lp.x, kUnscale, (float)hp.x) + __builtin_fmaf((float)lp.y, kUnscale, (float)hp.y);
            }
            split_rows::store_subblock_sum(a.sw_sums, (size_t)m, units, (unit0 + c8) >> 3, sum);
        }
        return;
    }
    float *out = a.splits > 1 ? a.partial + (size_t)split * a.M * a.N : a.y;
    auto out_row = [&](int r) { return m0 + tile_row(r, h); };
    if (a.splits == 1 && a.residual) {
        // requested together: y may be the residual's own memory, and a load behind each store is a trip to memory each
#pragma unroll
        for (int r = 0; r < SHARE; r++) v[r] += a.residual[(size_t)(out_row(r0 + r) < a.M ? out_row(r0 + r) : a.M - 1) * a.N + (n < a.N ? n : a.N - 1)];
    }
#pragma unroll
    for (int r = 0; r < SHARE; r++) if (out_row(r0 + r) < a.M && n < a.N) out[(size_t)out_row(r0 + r) * a.N + n] = v[r];
}

template <int TM, int NW>
hipError_t launch(const BlockSplitArgs &a, hipStream_t stream) {
    static std::atomic<uint64_t> raised{0};
    constexpr size_t lds = split_lds_bytes(TM, NW);
    static_assert(lds <= 160 * 1024, "LDS of a compute unit");
    const hipError_t err = raise_lds_limit(reinterpret_cast<const void *>(block_split_kernel<TM, NW>), lds, raised);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL((block_split_kernel<TM, NW>), dim3(a.n_tiles * a.m_tiles * a.splits), dim3(kThreads), lds, stream, a);
    return hipGetLastError();
}

hipError_t launch_form(int tm, int nw, const BlockSplitArgs &a, hipStream_t stream) {
    switch (tm * 10 + nw) {
    case 12: return launch<1, 2>(a, stream);
    case 14: return launch<1, 4>(a, stream);
    case 18: return launch<1, 8>(a, stream);
    case 24: return launch<2, 4>(a, stream);
    case 28: return launch<2, 8>(a, stream);
    case 38: return launch<3, 8>(a, stream);
    default: return hipErrorInvalidValue;
    }
}
// 64 rows for each of four groups, 96 for each of two and 128 rows do not fit the registers
constexpr struct { int tm, nw; } kForms[] = {{1, 2}, {1, 4}, {1, 8}, {2, 4}, {2, 8}, {3, 8}};

}  // namespace

static std::atomic<int> g_block_split_form{0};
void block_split_set_form(int form) {
    bool known = form < 0;
    for (const auto &f : kForms) known = known || (form / 100 == f.tm && form / 10 % 10 == f.nw && form % 10 >= 1);
    g_block_split_form.store(known ? form : 0);
}

// Expected time, as in block_gemm.hip: rounds of one workgroup per compute unit, a step of a round growing with the tile's rows and with the groups that stage their own activations, planes
// written and read once more.  Fitted to 3300 launches (thirteen shapes of 768 to 28672 weight rows and 768 to 14336 columns, 4 to 480 rows): off by 5 % at the median, 13 at the
// ninetieth percentile.
BlockSplitForm block_split_form(const GemmSplitParams &p) {
    const bool swiglu = p.swiglu.hi != nullptr;
    const int N = p.w.rows, M = p.rows, units = p.w.cols / 256, forced = g_block_split_form.load();
    static const int kSplits[] = {1, 2, 3, 4, 6, 8};
    const int cus = device_compute_units() > 0 ? device_compute_units() : 256;
    BlockSplitForm best;
    if (forced < 0 || (swiglu && (N / 2) % 32 != 0)) return best;
    for (const auto &f : kForms)
        for (int want : kSplits) {
            if (f.tm > 1 && f.tm > (M + 31) / 32) continue;
            const int kw = kWaves / f.nw;
            const auto [per, splits] = shares_of(units, f.nw, want);
            if (forced > 0 && (forced != f.tm * 100 + f.nw * 10 + want || (swiglu && splits > 1))) continue;
            if (forced == 0 && (splits != want || (swiglu && splits > 1))) continue;
            const float mb = (float)splits * (float)M * (float)N * 4e-6f;
            if (splits > 1 && (!p.workspace || (size_t)splits * M * N > p.workspace_floats)) continue;
            const long wgs = (long)((N + 32 * f.nw - 1) / (32 * f.nw)) * ((M + 32 * f.tm - 1) / (32 * f.tm)) * splits;
            float us = 1.4f + (float)((wgs + cus - 1) / cus) * (2 * per * (0.44f + f.tm * (0.433f + 0.227f * kw)) + 1.9f) + 0.363f * mb;
            if (splits > 1) us += 0.2f * mb + 1.0f + 0.3f * splits;
            // what a launch has to win by: the kernel of whole tiles is estimated as well, and large products behind a SiLU take longer here than this says
            us = forced > 0 ? 0.0f : us * (swiglu ? 1.25f : 1.12f);
            if (!best.tm || us < best.us) best = BlockSplitForm{f.tm, f.nw, 2 * per, splits, us};
        }
    return best;
}

hipError_t launch_block_split(const GemmSplitParams &p, const BlockSplitForm &f, hipStream_t stream) {
    BlockSplitArgs a{p.w.qs, p.w.qs_row_bytes, p.w.rows, p.w.cols, p.rows, p.x.hi, p.x.lo, p.x.sums, p.y, p.residual, p.workspace, p.swiglu.hi, p.swiglu.lo, p.swiglu.sums,
                     f.per, f.splits, (p.w.rows + 32 * f.nw - 1) / (32 * f.nw), (p.rows + 32 * f.tm - 1) / (32 * f.tm)};
    return launch_form(f.tm, f.nw, a, stream);
}

}  // namespace esp
