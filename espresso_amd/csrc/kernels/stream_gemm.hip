// y[m][n] = sum_k x[m][k] * W[n][k] for small products of up to 32 activation rows, W in Q4_0 or Q8_0: fp16 activations, weights exact (integers on the matrix cores, a block's scale to its
// sums), fp32 sums.
//
// A workgroup is eight wavefronts that share the K of 32 weight rows and nothing else until their sums meet in LDS: each brings its own share of both operands through a stretch of LDS that is its
// own, so there is no barrier on the way.
//   * Loads cover whole lines: eight neighbouring lanes 128 bytes of an activation row, four lanes 64 bytes of a weight row.  Lanes that are neighbours in the row but not in the wavefront are looked
//     up one by one (fragments straight from memory, lanes of a row sixteen apart: 11264 x 2048 Q8_0, 93 rows 33 us, through LDS 20).  LDS turns them into the operands of
//     v_mfma_f32_32x32x16_f16, sixteen bytes of the lane's own row a read; pieces are placed by row (exclusive or), so that neither side meets its banks twice.
//   * Which k a lane holds, the operands agree on: of each 32, 16 h + 8 f (Q8_0) or 16 f + 8 h (Q4_0, whose bytes hold k and k + 16), h the lane's half of the wavefront, f the fragment.
//   * Weights are two or four units (64 bytes of a row) ahead, activations a step of 64 k; a step asks for its activations before its weights, or the next step would wait for these too.
// What bounds it: launch, the first trip to memory (4 us of 5 to 8) and the chain of a wavefront's steps, which is why the rule below takes it for few of them.
#include "../common.h"
#include "block_gemm.h"
#include "block_tile.h"
#include "rows_gemm.h"
#include "silu.h"
#include "stream_gemm.h"
#include <type_traits>

namespace esp {
namespace {

using namespace block_tile;
typedef u32 uintx4 __attribute__((ext_vector_type(4)));

struct StreamArgs {
    const uint8_t *qs;
    const uint16_t *scales;
    size_t row_bytes;
    int N, K, M;
    const uint16_t *x;
    float *y;
    const float *residual;
    float *partial;
    uint16_t *swiglu_out;
    int per, splits, n_tiles;   // per: units of one wavefront
};

// Sixteen (or fewer) bytes at a uniform base and a lane's own 32-bit offset, hidden from the optimiser where it is used: its widening to 64 bits would leave the loop and take registers.
template <class V>
__device__ __forceinline__ V load_at(const void *base, u32 offset) {
    asm volatile("" : "+v"(offset));
    return *reinterpret_cast<const V *>(static_cast<const uint8_t *>(base) + offset);
}
// Between a wavefront's LDS writes and its reads of what other lanes wrote (or the other way round): LDS operations of a wavefront keep their order, so nothing waits here.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

constexpr int unit_of(int fmt) { return fmt == FMT_Q8_0 ? 64 : 128; }                              // k in 64 bytes of a row
constexpr int ahead(int fmt) { return fmt == FMT_Q8_0 ? 4 : 2; }                                   // units in flight: 256 k
constexpr int kXBytes = 4096, kWaveBytes = kXBytes + 2048;                                         // 32 rows of 128 bytes of activations, 32 rows of 64 bytes of weights

template <int FMT>
__global__ __launch_bounds__(kThreads) void stream_gemm_kernel(StreamArgs a) {
    static_assert(FMT == FMT_Q8_0 || FMT == FMT_Q4_0, "formats of one scale per block");
    constexpr int UNIT = unit_of(FMT), BLOCKS = UNIT / 32, STEPS = UNIT / 64, AHEAD = ahead(FMT);
    extern __shared__ float red[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, col = lane & 31;
    const auto [m_tile, n_tile, split] = place_of(1, a.n_tiles);
    const int n0 = n_tile * 32, n = n0 + col;
    const int all = a.K / UNIT, s0 = (split * kWaves + wave) * a.per, own = all - s0 < a.per ? (all > s0 ? all - s0 : 0) : a.per;

    // Rows past the end repeat the last one, never stored: offsets grow with the row, so the last row's is the most that a piece may have.
    const u32 xrow = (u32)a.K * 2, xlane = (u32)(lane >> 3) * xrow + (lane & 7) * 16, xmost = (u32)(a.M - 1) * xrow + (lane & 7) * 16;
    const u32 wrow = (u32)a.row_bytes, wlane = (u32)(lane >> 2) * wrow + (lane & 3) * 16, wmost = (u32)(a.N - 1 - n0) * wrow + (lane & 3) * 16;
    const u32 so = (u32)(n < a.N ? col : a.N - 1 - n0) * (u32)(a.K / 32) * 2;
    uint8_t *stretch = reinterpret_cast<uint8_t *>(red) + wave * kWaveBytes;
    uint8_t *xin = stretch + (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) * 16), *win = stretch + kXBytes + (lane >> 2) * 64 + (((lane & 3) ^ ((lane >> 3) & 3)) * 16);
    const uint8_t *xout[4], *wout[2];
#pragma unroll
    for (int g = 0; g < 4; g++) xout[g] = stretch + col * 128 + ((4 * (g >> 1) + (FMT == FMT_Q4_0 ? 2 * (g & 1) + h : 2 * h + (g & 1))) ^ (col & 7)) * 16;
#pragma unroll
    for (int p = 0; p < 2; p++) wout[p] = stretch + kXBytes + col * 64 + ((2 * p + h) ^ ((col >> 1) & 3)) * 16;
    const uint8_t *xbase = reinterpret_cast<const uint8_t *>(a.x) + (size_t)s0 * UNIT * 2, *wbase = a.qs + (size_t)n0 * a.row_bytes;
    const uint16_t *sbase = a.scales + (size_t)n0 * (a.K / 32);

    const floatx16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    floatx16 acc[1] = {zero16};

    if (own > 0) {
        typedef std::conditional_t<FMT == FMT_Q8_0, u32, uint2> Scales;
        uintx4 xr[4], wr[AHEAD][2];
        uint4 q[2];
        Scales sc[AHEAD], scale;
        const int last = own - 1, last_step = own * STEPS - 1;   // past the end the last ones are loaded again: in bounds, never used
        auto load_x = [&](int s) __attribute__((always_inline)) {
            const uint8_t *from = xbase + (size_t)(s < last_step ? s : last_step) * 128;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const u32 o = xlane + 8 * t * xrow;
                xr[t] = load_at<uintx4>(from, o < xmost ? o : xmost);
            }
        };
        auto load_w = [&](auto slot, int u) __attribute__((always_inline)) {
            const int at = s0 + (u < last ? u : last);
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const u32 o = wlane + 16 * t * wrow;
                wr[decltype(slot)::value][t] = load_at<uintx4>(wbase + (size_t)at * 64, o < wmost ? o : wmost);
            }
            sc[decltype(slot)::value] = load_at<Scales>(sbase + (size_t)at * BLOCKS, so);
        };
        auto scale_bits = [&](int b) __attribute__((always_inline)) {
            u32 pair;
            if constexpr (FMT == FMT_Q8_0) pair = scale;
            else pair = b >> 1 ? scale.y : scale.x;
            return b & 1 ? pair >> 16 : pair & 0xFFFFu;
        };
        // eight weights of the lane's row, fragment f of block b of the unit: q or q - 8
        auto decode = [&](int b, int f) __attribute__((always_inline)) {
            u32 o[4];
            if constexpr (FMT == FMT_Q8_0) {
                const uint4 &v = q[b];
                const u32 w[2] = {(f ? v.z : v.x) ^ 0x80808080u, (f ? v.w : v.y) ^ 0x80808080u};
                const h2 off = {(_Float16)1152.0f, (_Float16)1152.0f};   // 1024 + 128
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = as_u32(as_h2(__builtin_amdgcn_perm(0x64646464u, w[e >> 1], e & 1 ? 0x04030402u : 0x04010400u)) - off);
            } else {
                const uint4 &v = q[b >> 1];
                const u32 w[2] = {b & 1 ? v.z : v.x, b & 1 ? v.w : v.y}, mask = f ? 0x00F000F0u : 0x000F000Fu, magic = f ? 0x54005400u : 0x64006400u;
                const h2 off = f ? h2{(_Float16)72.0f, (_Float16)72.0f} : h2{(_Float16)1032.0f, (_Float16)1032.0f};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const u32 p = __builtin_amdgcn_perm(w[e >> 1], w[e >> 1], 0x03010200u);   // bytes 0 2 1 3: pairs come out adjacent
                    o[e] = as_u32(as_h2(((e & 1 ? p >> 8 : p) & mask) | magic) - off);
                }
            }
            return as_half8(make_uint4(o[0], o[1], o[2], o[3]));
        };
        auto unit = [&](auto slot, int u) __attribute__((always_inline)) {   // slot: u % AHEAD, the weights' slots by turns
            constexpr int S = decltype(slot)::value;
            wave_sync();
#pragma unroll
            for (int t = 0; t < 2; t++) *reinterpret_cast<uintx4 *>(win + t * 1024) = wr[S][t];
            scale = sc[S];
            wave_sync();
#pragma unroll
            for (int p = 0; p < 2; p++) {
                q[p] = *reinterpret_cast<const uint4 *>(wout[p]);
                if constexpr (FMT == FMT_Q4_0) {   // each half of a wavefront holds blocks h and 2 + h; it needs bytes 8 h .. of all four
                    const auto e0 = __builtin_amdgcn_permlane32_swap(q[p].x, q[p].z, false, false);
                    const auto e1 = __builtin_amdgcn_permlane32_swap(q[p].y, q[p].w, false, false);
                    q[p] = make_uint4(e0[0], e1[0], e0[1], e1[1]);
                }
            }
#pragma unroll
            for (int b = 0; b < BLOCKS; b++) {
                if (b % 2 == 0) {
                    wave_sync();
#pragma unroll
                    for (int t = 0; t < 4; t++) *reinterpret_cast<uintx4 *>(xin + t * 1024) = xr[t];
                    load_x(u * STEPS + b / 2 + 1);
                    if (b + 2 >= BLOCKS) load_w(slot, u + AHEAD);
                    wave_sync();
                    __builtin_amdgcn_sched_barrier(0);
                }
                const half8 x0 = *reinterpret_cast<const half8 *>(xout[2 * (b & 1)]), x1 = *reinterpret_cast<const half8 *>(xout[2 * (b & 1) + 1]);
                const floatx16 low = __builtin_amdgcn_mfma_f32_32x32x16_f16(x0, decode(b, 0), zero16, 0, 0, 0);
                const floatx16 part = __builtin_amdgcn_mfma_f32_32x32x16_f16(x1, decode(b, 1), low, 0, 0, 0);
                const float d = half_bits_to_float(scale_bits(b));
#pragma unroll
                for (int r = 0; r < 16; r++) acc[0][r] = __builtin_fmaf(d, part[r], acc[0][r]);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        typedef std::integral_constant<int, 0> C0;
        typedef std::integral_constant<int, 1> C1;
        typedef std::integral_constant<int, 2> C2;
        typedef std::integral_constant<int, 3> C3;
        load_w(C0{}, 0);
        load_x(0);
        load_w(C1{}, 1);
        if constexpr (AHEAD == 4) { load_w(C2{}, 2); load_w(C3{}, 3); }
        int u = 0;
        for (; u + AHEAD <= own; u += AHEAD) {
            unit(C0{}, u);
            unit(C1{}, u + 1);
            if constexpr (AHEAD == 4) { unit(C2{}, u + 2); unit(C3{}, u + 3); }
        }
        if (u < own) unit(C0{}, u);
        if constexpr (AHEAD == 4) {
            if (u + 1 < own) unit(C1{}, u + 1);
            if (u + 2 < own) unit(C2{}, u + 2);
        }
    }

    constexpr int SHARE = 16 / kWaves;    // accumulators that a wavefront finishes
    const int r0 = wave * SHARE;
    float v[SHARE];
    __syncthreads();                           // everybody has read the operands
    share_sums<1, 1>(acc, red, wave, 0, lane, r0, v);
    if (a.swiglu_out) {
#pragma unroll
        for (int k = 0; k < SHARE / 2; k++) {
            const bool odd = lane & 1;
            float g, up;
            gate_and_up(v[2 * k], v[2 * k + 1], odd, g, up);
            const int m = tile_row(r0 + 2 * k + (odd ? 1 : 0), h);
            if (m < a.M && (n | 1) < a.N) a.swiglu_out[(size_t)m * (a.N / 2) + n / 2] = __builtin_bit_cast(uint16_t, (_Float16)__fmul_rn(silu(g), up));
        }
        return;
    }
    float *out = a.splits > 1 ? a.partial + (size_t)split * a.M * a.N : a.y;
    if (a.splits == 1 && a.residual) {
        // requested together: y may be the residual's own memory, and a load behind each store is a trip to memory each
#pragma unroll
        for (int r = 0; r < SHARE; r++) v[r] += a.residual[(size_t)(tile_row(r0 + r, h) < a.M ? tile_row(r0 + r, h) : a.M - 1) * a.N + (n < a.N ? n : a.N - 1)];
    }
#pragma unroll
    for (int r = 0; r < SHARE; r++) if (tile_row(r0 + r, h) < a.M && n < a.N) out[(size_t)tile_row(r0 + r, h) * a.N + n] = v[r];
}

constexpr size_t kLdsBytes = (size_t)kWaves * kWaveBytes;
static_assert(kLdsBytes >= (size_t)kWaves * 16 * 64 * 4 && kLdsBytes <= 64 * 1024, "the sums; the default limit of dynamic LDS");

std::atomic<int> g_stream_gemm_mode{1};

// As many shares of K as keep every workgroup resident at once; one where no caller adds them, and where rows_gemm.hip would have taken the product, whose bits these are (the same K in a wavefront,
// added in the same order).
Shares stream_shares(const GemmParams &p, bool one_launch) {
    const int units = p.w.cols / unit_of(p.w.format), tiles = (p.w.rows + 31) / 32, cus = device_compute_units() > 0 ? device_compute_units() : 256;
    Shares best = shares_of(units, 1, 1);
    if (one_launch || !p.deferred_splits || p.swiglu_out || !p.workspace) return best;
    for (int want = 2; want <= 4 && tiles * want <= cus; want++) {
        const Shares s = shares_of(units, 1, want);
        if (s.splits == want && (size_t)want * p.rows * p.w.rows <= p.workspace_floats) best = s;
    }
    return best;
}

}  // namespace

void stream_gemm_set_mode(int mode) { g_stream_gemm_mode.store(mode < 0 ? 1 : mode); }

bool stream_gemm_takes(const GemmParams &p) {
    const int mode = g_stream_gemm_mode.load();
    const DeviceMatrix &w = p.w;
    if (mode == 0 || (w.format != FMT_Q8_0 && w.format != FMT_Q4_0) || w.cols % unit_of(w.format) != 0 || p.rows < 3 || p.rows > 32 || (p.swiglu_out && (w.rows % 2 != 0 || p.residual))) return false;
    const bool one_launch = rows_gemm_takes(p);
    if (!one_launch && !(block_gemm_takes(p) && block_gemm_exact(p))) return false;   // weights are kept exactly where they were
    if (mode == 2) return true;
    if (!rows_gemm_by_size() || !block_gemm_by_size()) return false;
    // Where a wavefront has few steps and all workgroups are resident at once; us, in block_gemm.hip -> here, 12 / 16 / 31 rows, shares of K either way: Q4_0 2048 x 2048 6.0 / 6.0 / 6.2 -> 5.9 / 5.0 /
    // 5.2, 2560 x 2048 6.0 / 6.1 / 6.2 -> 5.1 / 5.2 / 5.4, 3072 x 3072 7.4 / 7.4 / 8.2 -> 6.7 / 6.6 / 7.4, 2048 x 5632 7.9 / 8.0 / 9.4 -> 7.2 / 7.3 / 7.6;  31 rows of Q8_0 2048 x 2048 7.1 -> 5.7,
    // 2560 x 2048 8.3 -> 6.8, 2048 x 5632 9.8 -> 8.4.  More steps, or rounds of workgroups: 8 rows of 5120 x 3072 Q8_0 9.3 there, 10.5 here, of 11264 x 2048 13.5, 15.6.  More rows: 48 / 64 of
    // 2048 x 2048 Q4_0 6.7 / 6.5 there, 6.6 / 6.8 here (a form of two row tiles), Q8_0 7.3 / 7.3, 6.8 / 7.5.
    // Q8_0 of up to sixteen rows (2048 columns 7.4 -> 6.9) keeps that kernel's order of sums: short prompts go on to the tokens they went on to where two are equally likely.
    // In rows_gemm.hip -> here, the same bits, 5 / 12 / 16 / 31 rows: Q8_0 2304 x 768 4.8 / 6.0 / 6.6 / 6.2 -> 4.4 / 5.7 / 6.1 / 5.7, Q4_0 768 x 768 4.7 / 5.4 / 5.7 / 6.0 -> 4.1 / 5.4 / 5.3 / 5.4;
    // 576 and 1536 columns, one and three steps, within 10 % either way.
    const Shares s = stream_shares(p, one_launch);
    const int cus = device_compute_units() > 0 ? device_compute_units() : 256, steps = s.per * unit_of(w.format) / 64;
    if (one_launch ? steps != 2 || steps != (w.cols / 64 + kWaves - 1) / kWaves : w.format == FMT_Q8_0 && p.rows <= 16) return false;
    return (w.rows + 31) / 32 * s.splits <= cus && steps <= 4;
}

hipError_t launch_stream_gemm(const GemmParams &p, int *splits, hipStream_t stream) {
    const Shares s = stream_shares(p, rows_gemm_takes(p));
    const StreamArgs a{p.w.qs, p.w.scales, p.w.qs_row_bytes, p.w.rows, p.w.cols, p.rows, p.x, p.y, p.residual, p.workspace, p.swiglu_out, s.per, s.splits, (p.w.rows + 31) / 32};
    *splits = s.splits;
    if (p.w.format == FMT_Q8_0) hipLaunchKernelGGL((stream_gemm_kernel<FMT_Q8_0>), dim3(a.n_tiles * a.splits), dim3(kThreads), kLdsBytes, stream, a);
    else hipLaunchKernelGGL((stream_gemm_kernel<FMT_Q4_0>), dim3(a.n_tiles * a.splits), dim3(kThreads), kLdsBytes, stream, a);
    return hipGetLastError();
}

}  // namespace esp
