// y[m][n] = sum_k x[m][k] * W[n][k], W in fp16: every product of three and more rows of activations with an fp16 matrix, except those of a few steps that rows_gemm.hip takes.  The walk over
// K: wide_tile.h.  Tile and shares of K come from a cost rule (wide_gemm_form).
// Against the kernels these products had before (128 x 128 tiles of four wavefronts, gate|up of up to a tile a compute unit with weights that skip LDS), us, planes of shares counted:
//   16384 x 3072 behind a SiLU, 16 / 64 / 200 / 600 / 1777 rows 22 / 30 / 41 / 123 / 217 -> 20 / 21 / 33 / 74 / 176;  3072 x 8192 17 / 20 / 42 / 69 / 144 -> 12 / 14 / 24 / 43 / 101;
//   2048 x 2048 7.8 / 9.7 / 14.1 / 22.8 / 47.9 -> 5.9 / 7.1 / 9.5 / 14.5 / 23.2;  28672 x 4096 54 / 65 / 126 / 212 / 538 -> 53 / 54 / 77 / 176 / 479;
// 1.34 times as fast on average over fourteen shapes and 3 to 2048 rows.  What bounds it now: few rows, the weights' way from memory (28672 x 4096: 235 MB in 53 us); many rows, power
// (4096^3: 1.16 PFLOP/s with every compute unit at work, a step of 256 x 256 tiles 1.8 us; 1.3 us while a third of them are).  The same walk with packed weights, unpacked on their way to LDS,
// measured 0.94 to 1.03 times block_gemm.hip's kernels, which keep theirs out of LDS: those formats stay there.
#include "../common.h"
#include "silu.h"
#include "wide_gemm.h"
#include "wide_tile.h"
#include <atomic>

namespace esp {
namespace {

using namespace wide;
struct WideArgs {
    const uint16_t *w;
    int N, K, M;
    const uint16_t *x;
    float *y;
    const float *residual;
    float *partial;
    uint16_t *swiglu_out;
    int per, splits, n_tiles, m_tiles;   // per: steps of a share
};

template <int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(kThreads) void wide_gemm_kernel(WideArgs a) {
    using T = Tile<WM, WN, TM, TN>;
    extern __shared__ uint4 smem[];
    uint16_t *lds = reinterpret_cast<uint16_t *>(smem);
    const auto [m_tile, n_tile, split] = place_of(a.m_tiles, a.n_tiles);
    const int m0 = m_tile * T::BM, n0 = n_tile * T::BN, all = a.K / kStep, first = split * a.per, steps = all - first < a.per ? all - first : a.per;
    floatx16 acc[TM][TN];
    Plain<T::BM, T::kDepth> x(a.x, (size_t)a.K, m0, a.M, (size_t)first * kStep, steps);
    Plain<T::BN, T::kDepth> w(a.w, (size_t)a.K, n0, a.N, (size_t)first * kStep, steps);
    walk<false, WM, WN, TM, TN>(x, w, steps, lds, acc);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave / WN, wn = wave % WN, h = lane >> 5, col = lane & 31;
    float *out = a.splits > 1 ? a.partial + (size_t)split * a.M * a.N : a.y;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int n = n0 + (wn * TN + j) * 32 + col, mb = m0 + (wm * TM + i) * 32 + 4 * h;
            auto row = [&](int r) { return mb + 8 * (r >> 2) + (r & 3); };
            if (a.swiglu_out) {   // weight rows as (gate, up) pairs are neighbouring lanes: the even lane finishes rows 2 k of both, the odd lane rows 2 k + 1
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const float even = acc[i][j][2 * k], uneven = acc[i][j][2 * k + 1];
                    const float p0 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, even), 0xB1, 0xF, 0xF, false));   // quad_perm [1,0,3,2]
                    const float p1 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, uneven), 0xB1, 0xF, 0xF, false));
                    const float gate = lane & 1 ? p1 : even, up = lane & 1 ? uneven : p0;
                    const int m = row(2 * k + (lane & 1));
                    if (m < a.M && (n | 1) < a.N) a.swiglu_out[(size_t)m * (a.N / 2) + n / 2] = __builtin_bit_cast(uint16_t, (_Float16)__fmul_rn(silu(gate), up));
                }
                continue;
            }
            if (a.splits == 1 && a.residual) {   // requested together: y may be the residual's own memory, and a load behind each store is a trip to memory each
                float before[16];
#pragma unroll
                for (int r = 0; r < 16; r++) before[r] = a.residual[(size_t)(row(r) < a.M ? row(r) : a.M - 1) * a.N + (n < a.N ? n : a.N - 1)];
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] += before[r];
            }
#pragma unroll
            for (int r = 0; r < 16; r++) if (row(r) < a.M && n < a.N) out[(size_t)row(r) * a.N + n] = acc[i][j][r];
        }
}

template <int WM, int WN, int TM, int TN>
hipError_t launch(const WideArgs &a, hipStream_t stream) {
    using T = Tile<WM, WN, TM, TN>;
    static std::atomic<uint64_t> raised{0};
    const void *kernel = reinterpret_cast<const void *>(wide_gemm_kernel<WM, WN, TM, TN>);
    const hipError_t err = raise_lds_limit(kernel, T::kLdsBytes, raised);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL((wide_gemm_kernel<WM, WN, TM, TN>), dim3(a.n_tiles * a.m_tiles * a.splits), dim3(kThreads), T::kLdsBytes, stream, a);
    return hipGetLastError();
}
hipError_t launch_form(const WideForm &f, const WideArgs &a, hipStream_t stream) {
    switch (f.bm * 1000 + f.bn) {
    case 256256: return launch<4, 2, 2, 4>(a, stream);
    case 192256: return launch<2, 4, 3, 2>(a, stream);
    case 128256: return launch<2, 4, 2, 2>(a, stream);
    case 256128: return launch<4, 2, 2, 2>(a, stream);
    case 192128: return launch<2, 4, 3, 1>(a, stream);
    case 128128: return launch<2, 4, 2, 1>(a, stream);
    case 64256: return launch<2, 4, 1, 2>(a, stream);
    case 64128: return launch<2, 4, 1, 1>(a, stream);
    default: return hipErrorInvalidValue;
    }
}
std::atomic<int> g_wide_gemm_form{0};

}  // namespace

void wide_gemm_set_form(int form) { g_wide_gemm_form.store(wide_form_known(form) ? form : 0); }

// (behind a SiLU, and where no caller adds them, the planes take a launch of their own)
WideForm wide_gemm_form(const GemmParams &p) {
    if (p.w.format != FMT_F16 || p.w.cols % kStep != 0) return WideForm{};
    WideProduct w;
    w.rows = p.rows; w.weight_rows = p.w.rows; w.steps = p.w.cols / kStep; w.compute_units = device_compute_units();
    w.stored_mb = (float)p.rows * (float)p.w.rows * (p.swiglu_out ? 1e-6f : 4e-6f);
    w.plane_floats = p.workspace ? p.workspace_floats : 0;
    w.after = p.swiglu_out ? 3.0f : p.deferred_splits ? 1.0f : 1.6f;
    w.after_share = p.swiglu_out || p.deferred_splits ? 0.0f : 0.2f;
    w.forced = g_wide_gemm_form.load();
    const WideForm f = choose_wide_form(w);
    if (f.bm || w.forced == 0) return f;
    w.forced = 0;   // shares whose planes have no room: by size
    return choose_wide_form(w);
}

hipError_t launch_wide_gemm(const GemmParams &p, const WideForm &f, hipStream_t stream) {
    const WideArgs a{reinterpret_cast<const uint16_t *>(p.w.qs), p.w.rows, p.w.cols, p.rows, p.x, p.y, p.residual, p.workspace, f.splits == 1 && p.w.rows % 2 == 0 ? p.swiglu_out : nullptr,
                     f.per, f.splits, (p.w.rows + f.bn - 1) / f.bn, (p.rows + f.bm - 1) / f.bm};
    return launch_form(f, a, stream);
}

}  // namespace esp
