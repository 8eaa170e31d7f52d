// Blocks of rows against dense matrices on the matrix cores (gfx950): the prompt products of the layered models.
//
//   y[m][n] = sum_k a[m][k] b[n][k],   bf16 operands or fp32 ones, fp32 accumulation
//
// bf16 operands: the walk of wide_tile.h (tiles of 64 x 128 to 256 x 256, by the cost rule of wide_form.h).  Against tiles of 128 x 128 (64, 32) of
// four wavefronts, prompts of six layers, us: Ranavik d768, 40 / 600 / 1700 tokens 498 / 765 / 1250 -> 447 / 596 / 982, d4096, 64 / 300 / 1000 tokens 1330 / 2320 / 4480 -> 1190 / 1860 / 3910,
// Forovik d2048, 60 / 500 / 1100 tokens 649 / 1158 / 1849 -> 591 / 888 / 1543;  steps of 16 sequences of d2048 (prompts and 24 steps) 20470 -> 18940.
// fp32 operands (v_mfma_f32_32x32x2_f32):
//   * a workgroup of four wavefronts owns a BM x BN tile of y and walks k in tiles of 128 bytes per row (64 bf16 or 32 fp32
//     values); LDS holds two tiles of both operands, so one barrier per tile is enough, and two more are on their way in registers;
//   * rows of LDS are 144 bytes apart: the 128-bit fragment reads of eight rows cover all banks;
//   * a bf16 operand of an fp32 product (weights under fp32 activations) is widened on its way to LDS;
//   * block index -> tile: the tiles of y that share rows of b follow each other on the same die (workgroups are dealt round robin
//     over the eight dies), so a tile of weights comes from HBM once and from that die's L2 afterwards;
//   * short grids split k over grid.y and leave partial planes, which launch_residual_norm adds in order.
#include <hip/hip_runtime.h>

#include <type_traits>

#include <atomic>

#include "../common.h"
#include "layer_ops.h"
#include "matrix_ops.h"
#include "wide_form.h"
#include "wide_tile.h"

namespace esp {
namespace {

using matrix::floatx16;
using matrix::Op;

constexpr int kDies = 8;

struct DenseGemmArgs {
    const void *a, *a2, *b;
    int lda, ldb, m, n, tiles, tiles_per_split, m_tiles, n_tiles;
    int out;
    void *y;
    int ldy, mix_cols;
    void *act;
    int ld_act, gate_function, n_store;
    float cap;
};

// Eight consecutive values of an operand row on their way to LDS.
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx8 __attribute__((ext_vector_type(8)));
template <typename T>
struct PieceOf { typedef uintx4 type; };
template <>
struct PieceOf<float> { typedef floatx8 type; };
__device__ __forceinline__ uintx4 fetch_piece(const uint16_t *p) { return *reinterpret_cast<const uintx4 *>(p); }
__device__ __forceinline__ floatx8 fetch_piece(const float *p) {
    const floatx4 a = reinterpret_cast<const floatx4 *>(p)[0], b = reinterpret_cast<const floatx4 *>(p)[1];
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}
__device__ __forceinline__ void store_piece(uintx4 d, uint16_t *lds) { *reinterpret_cast<uintx4 *>(lds) = d; }
__device__ __forceinline__ void store_piece(floatx8 d, float *lds) {
    reinterpret_cast<floatx4 *>(lds)[0] = __builtin_shufflevector(d, d, 0, 1, 2, 3);
    reinterpret_cast<floatx4 *>(lds)[1] = __builtin_shufflevector(d, d, 4, 5, 6, 7);
}
__device__ __forceinline__ void store_piece(uintx4 d, float *lds) {
    const uintx4 lo = d << 16, hi = d & 0xFFFF0000u;
    reinterpret_cast<floatx4 *>(lds)[0] = __builtin_bit_cast(floatx4, __builtin_shufflevector(lo, hi, 0, 4, 1, 5));
    reinterpret_cast<floatx4 *>(lds)[1] = __builtin_bit_cast(floatx4, __builtin_shufflevector(lo, hi, 2, 6, 3, 7));
}

// The 32 rows from m0 on of column n (lane % 32 of its 32).
template <typename E>
__device__ __forceinline__ void store_tile(const DenseGemmArgs &a, const floatx16 &acc, int m0, int n, int lane, int split, bool after_mix) {
    const int half = lane >> 5;
    if (after_mix) {   // even lanes hold gates, their right neighbours the ups: the even lane finishes rows 2 k of both, the odd lane rows 2 k + 1
        const bool odd = lane & 1;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float even = acc[2 * k], uneven = acc[2 * k + 1];
            const float p0 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, even), 0xB1, 0xF, 0xF, false));   // quad_perm [1,0,3,2]
            const float p1 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, uneven), 0xB1, 0xF, 0xF, false));
            const int m = m0 + matrix::accumulator_row(2 * k + (odd ? 1 : 0), half);
            if (m < a.m && (n | 1) < a.n)
                static_cast<E *>(a.act)[(size_t)m * a.ld_act + (n - a.mix_cols) / 2] = Op<E>::from_float(matrix::gated(a.gate_function, odd ? p1 : even, odd ? uneven : p0));
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int m = m0 + matrix::accumulator_row(r, half);
        const float v = acc[r];
        if (m >= a.m || n >= a.n) continue;
        if (a.out == (int)GemmOut::planes) static_cast<float *>(a.y)[((size_t)split * a.m + m) * a.ldy + n] = v;
        else if (a.out == (int)GemmOut::mix_gated) static_cast<float *>(a.y)[(size_t)m * a.ldy + n] = v;
        else if (a.out == (int)GemmOut::elems) static_cast<E *>(a.y)[(size_t)m * a.ldy + n] = Op<E>::from_float(v);
        else if (n < a.n_store) static_cast<float *>(a.y)[(size_t)m * a.ldy + n] = a.cap > 0.0f ? a.cap * tanhf(v / a.cap) : v;
    }
}

template <typename TA, typename TB, int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(64 * WM * WN) void dense_gemm_kernel(DenseGemmArgs a) {
    static_assert(std::is_same<TA, float>::value || std::is_same<TB, float>::value, "bf16 operands have a kernel of their own");
    using E = float;
    constexpr int THREADS = 64 * WM * WN, BM = 32 * WM * TM, BN = 32 * WN * TN;
    constexpr int KT = 128 / sizeof(E), LDK = 144 / sizeof(E), NCH = KT / 8;   // values per tile row, per LDS row; pieces per tile row
    constexpr int XA = BM * NCH / THREADS, XB = BN * NCH / THREADS;
    static_assert(XA >= 1 && XB >= 1, "tile too small for the copy loop");
    __shared__ E at[2][BM * LDK];
    __shared__ E bt[2][BN * LDK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave / WN, wn = wave % WN;
    // the m tiles of one n tile follow each other on one die
    const int die = blockIdx.x % kDies, at_die = blockIdx.x / kDies, mt = at_die % a.m_tiles, nt = at_die / a.m_tiles * kDies + die;
    if (nt >= a.n_tiles) return;
    const int m0 = mt * BM, n0 = nt * BN;
    const int t_begin = blockIdx.y * a.tiles_per_split;
    const int t_end = t_begin + a.tiles_per_split < a.tiles ? t_begin + a.tiles_per_split : a.tiles, t_last = t_end - 1;
    const bool after_mix = a.out == (int)GemmOut::mix_gated && n0 >= a.mix_cols;
    const TA *ap = static_cast<const TA *>(after_mix ? a.a2 : a.a);
    const TB *bp = static_cast<const TB *>(a.b);

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = matrix::zero_accumulator();

    typedef typename PieceOf<TA>::type PA;
    typedef typename PieceOf<TB>::type PB;
    PA pa0[XA], pa1[XA];   // even and odd tiles
    PB pb0[XB], pb1[XB];
    const TA *ar[XA];
    const TB *br[XB];
#pragma unroll
    for (int i = 0; i < XA; i++) {
        const int piece = tid + i * THREADS, row = m0 + piece / NCH;
        ar[i] = ap + (size_t)(row < a.m ? row : a.m - 1) * a.lda + (piece % NCH) * 8;   // rows past the end repeat the last one; never stored
    }
#pragma unroll
    for (int i = 0; i < XB; i++) {
        const int piece = tid + i * THREADS, row = n0 + piece / NCH;
        br[i] = bp + (size_t)(row < a.n ? row : a.n - 1) * a.ldb + (piece % NCH) * 8;
    }
    auto fetch = [&](PA (&pa)[XA], PB (&pb)[XB], int tile) {   // tiles past the end repeat the last one
        const size_t k = (size_t)(tile < t_last ? tile : t_last) * KT;
#pragma unroll
        for (int i = 0; i < XA; i++) pa[i] = fetch_piece(ar[i] + k);
#pragma unroll
        for (int i = 0; i < XB; i++) pb[i] = fetch_piece(br[i] + k);
    };
    auto stage = [&](const PA (&pa)[XA], const PB (&pb)[XB], int buf) {
#pragma unroll
        for (int i = 0; i < XA; i++) {
            const int piece = tid + i * THREADS;
            store_piece(pa[i], at[buf] + piece / NCH * LDK + (piece % NCH) * 8);
        }
#pragma unroll
        for (int i = 0; i < XB; i++) {
            const int piece = tid + i * THREADS;
            store_piece(pb[i], bt[buf] + piece / NCH * LDK + (piece % NCH) * 8);
        }
    };
    fetch(pa0, pb0, t_begin);
    fetch(pa1, pb1, t_begin + 1);
    stage(pa0, pb0, 0);
    fetch(pa0, pb0, t_begin + 2);
    __syncthreads();
    auto multiply = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < KT / 16; ks++) {
            const int kk = ks * 16 + 8 * (lane >> 5);
            typename Op<E>::frag af[TM], bf[TN];
#pragma unroll
            for (int i = 0; i < TM; i++) af[i] = Op<E>::load(at[buf] + ((wm * TM + i) * 32 + (lane & 31)) * LDK + kk);
#pragma unroll
            for (int j = 0; j < TN; j++) bf[j] = Op<E>::load(bt[buf] + ((wn * TN + j) * 32 + (lane & 31)) * LDK + kk);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = Op<E>::mma(af[i], bf[j], acc[i][j]);
        }
    };
    int t0 = t_begin;
    for (; t0 + 1 < t_end; t0 += 2) {
        multiply(0);
        stage(pa1, pb1, 1);
        fetch(pa1, pb1, t0 + 3);
        __syncthreads();
        multiply(1);
        stage(pa0, pb0, 0);
        fetch(pa0, pb0, t0 + 4);
        __syncthreads();
    }
    if (t0 < t_end) multiply(0);

#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) store_tile<E>(a, acc[i][j], m0 + (wm * TM + i) * 32, n0 + (wn * TN + j) * 32 + (lane & 31), lane, blockIdx.y, after_mix);
}

// bf16 operands
template <int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(wide::kThreads) void dense_wide_kernel(DenseGemmArgs a) {
    using T = wide::Tile<WM, WN, TM, TN>;
    extern __shared__ uint4 smem[];
    const auto [m_tile, n_tile, split] = wide::place_of(a.m_tiles, a.n_tiles);
    const int m0 = m_tile * T::BM, n0 = n_tile * T::BN, first = split * a.tiles_per_split, steps = a.tiles - first < a.tiles_per_split ? a.tiles - first : a.tiles_per_split;
    const bool after_mix = a.out == (int)GemmOut::mix_gated && n0 >= a.mix_cols;   // a tile lies on one side
    floatx16 acc[TM][TN];
    wide::Plain<T::BM, T::kDepth> x(static_cast<const uint16_t *>(after_mix ? a.a2 : a.a), (size_t)a.lda, m0, a.m, (size_t)first * wide::kStep, steps);
    wide::Plain<T::BN, T::kDepth> w(static_cast<const uint16_t *>(a.b), (size_t)a.ldb, n0, a.n, (size_t)first * wide::kStep, steps);
    wide::walk<true, WM, WN, TM, TN>(x, w, steps, reinterpret_cast<uint16_t *>(smem), acc);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave / WN, wn = wave % WN;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) store_tile<uint16_t>(a, acc[i][j], m0 + (wm * TM + i) * 32, n0 + (wn * TN + j) * 32 + (lane & 31), lane, split, after_mix);
}

int ceil_div(int a, int b) { return (a + b - 1) / b; }
DenseGemmArgs arguments(const DenseGemm &p, int bm, int bn) {
    DenseGemmArgs a{};
    a.a = p.a; a.a2 = p.a2; a.b = p.b; a.lda = p.lda; a.ldb = p.ldb; a.m = p.m; a.n = p.n;
    a.m_tiles = ceil_div(p.m, bm); a.n_tiles = ceil_div(p.n, bn);
    a.out = (int)p.out; a.y = p.y; a.ldy = p.ldy; a.mix_cols = p.mix_cols; a.act = p.act; a.ld_act = p.ld_act; a.gate_function = (int)p.gate_function; a.n_store = p.n_store; a.cap = p.cap;
    return a;
}

std::atomic<int> g_dense_gemm_form{0};
WideProduct wide_product(int m, int n, int k) {
    WideProduct w;
    w.rows = m; w.weight_rows = n; w.steps = k / wide::kStep; w.compute_units = device_compute_units();
    w.plane_floats = SIZE_MAX;
    return w;
}
template <int WM, int WN, int TM, int TN>
hipError_t launch_wide(const DenseGemm &p, int splits, int per, hipStream_t s) {
    using T = wide::Tile<WM, WN, TM, TN>;
    static std::atomic<uint64_t> raised{0};
    const void *kernel = reinterpret_cast<const void *>(dense_wide_kernel<WM, WN, TM, TN>);
    const hipError_t err = wide::raise_lds_limit(kernel, T::kLdsBytes, raised);
    if (err != hipSuccess) return err;
    DenseGemmArgs a = arguments(p, T::BM, T::BN);
    a.tiles = p.k / wide::kStep;
    a.tiles_per_split = per;
    hipLaunchKernelGGL((dense_wide_kernel<WM, WN, TM, TN>), dim3(a.m_tiles * a.n_tiles * splits), dim3(wide::kThreads), T::kLdsBytes, s, a);
    return hipGetLastError();
}
hipError_t run_wide(const DenseGemm &p, hipStream_t s) {
    WideProduct w = wide_product(p.m, p.n, p.k);
    w.shares = p.splits;
    const bool gated = p.out == GemmOut::mix_gated;
    const float gated_cols = gated && p.n > p.mix_cols ? (float)(p.n - p.mix_cols) : 0.0f, elem = p.out == GemmOut::elems ? 2e-6f : 4e-6f;
    w.stored_mb = (float)p.m * (((float)p.n - gated_cols) * elem + gated_cols * 1e-6f);
    w.wide_weights = !gated || p.mix_cols % 256 == 0 || p.mix_cols >= p.n;
    WideForm f;
    if (const int forced = g_dense_gemm_form.load(); forced > 0) {   // whatever shares it names
        w.forced = forced / 10 * 10 + p.splits;
        f = choose_wide_form(w);
        w.forced = 0;
    }
    if (!f.bm) f = choose_wide_form(w);
    if (f.splits != p.splits) return hipErrorInvalidValue;   // a share without work would leave its plane unwritten
    switch (f.bm * 1000 + f.bn) {
    case 256256: return launch_wide<4, 2, 2, 4>(p, f.splits, f.per, s);
    case 192256: return launch_wide<2, 4, 3, 2>(p, f.splits, f.per, s);
    case 128256: return launch_wide<2, 4, 2, 2>(p, f.splits, f.per, s);
    case 256128: return launch_wide<4, 2, 2, 2>(p, f.splits, f.per, s);
    case 192128: return launch_wide<2, 4, 3, 1>(p, f.splits, f.per, s);
    case 128128: return launch_wide<2, 4, 2, 1>(p, f.splits, f.per, s);
    case 64256: return launch_wide<2, 4, 1, 2>(p, f.splits, f.per, s);
    case 64128: return launch_wide<2, 4, 1, 1>(p, f.splits, f.per, s);
    default: return hipErrorInvalidValue;
    }
}

struct TileShape { int bm, bn; };
// Tall tiles unless they leave compute units without one (a launch that may split k fills the chip that way instead).
TileShape tile_for(int m, int n, bool splits) {
    if (m <= 64 || (!splits && ((m + 127) / 128) * ((n + 127) / 128) < 200)) return TileShape{64, 128};
    return TileShape{128, 128};
}
template <typename TA, typename TB>
hipError_t run(const DenseGemm &p, hipStream_t s) {
    constexpr int KT = 32;
    const TileShape t = tile_for(p.m, p.n, p.out == GemmOut::planes);
    DenseGemmArgs a = arguments(p, t.bm, t.bn);
    a.tiles = p.k / KT;
    a.tiles_per_split = ceil_div(a.tiles, p.splits);
    if ((p.splits - 1) * a.tiles_per_split >= a.tiles) return hipErrorInvalidValue;   // a split without work would leave its plane unwritten
    const dim3 grid(ceil_div(a.n_tiles, kDies) * kDies * a.m_tiles, p.splits);
    if (t.bm == 64) hipLaunchKernelGGL((dense_gemm_kernel<TA, TB, 2, 2, 1, 2>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((dense_gemm_kernel<TA, TB, 2, 2, 2, 2>), grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace

void dense_gemm_set_form(int form) { g_dense_gemm_form.store(wide_form_known(form) ? form : 0); }

// bf16: as many shares of K as the product and the kernel that adds them take the least time with.  fp32: enough workgroups for two per compute unit, at least four tiles of 64 per share.
// Planes stay within the workspace.
int gemm_planes_splits(int m, int n, int k, Precision type, size_t workspace_floats) {
    if (type == Precision::bf16) {
        WideProduct w = wide_product(m, n, k);
        w.stored_mb = (float)m * (float)n * 4e-6f;
        w.plane_floats = workspace_floats;
        w.after = -0.2f * w.stored_mb;   // that kernel reads one plane in any case
        return choose_wide_form(w).splits;
    }
    const TileShape t = tile_for(m, n, true);
    const int tiles = ceil_div(m, t.bm) * ceil_div(n, t.bn), k_tiles = k / 64;
    int splits = 1;
    for (int s = 2; s <= 16; s++) {
        const int per = ceil_div(k_tiles, s);
        if (tiles * s > 640 || per < 4 || (size_t)s * m * n > workspace_floats) break;
        if ((s - 1) * per < k_tiles) splits = s;
    }
    return splits;
}

hipError_t launch_dense_gemm(const DenseGemm &p, hipStream_t s) {
    const bool gated_only = p.out == GemmOut::mix_gated && p.mix_cols == 0;
    if (!p.a || !p.b || (!p.y && !gated_only) || p.m < 1 || p.n < 1 || p.k < 64 || p.k % 64 || p.splits < 1 || p.lda < p.k || p.ldb < p.k || p.lda % 8 || p.ldb % 8) return hipErrorInvalidValue;
    if (p.out != GemmOut::planes && p.splits != 1) return hipErrorInvalidValue;
    if (p.out == GemmOut::mix_gated && (p.mix_cols % 128 || p.n % 2 || (p.n > p.mix_cols && (!p.a2 || !p.act)))) return hipErrorInvalidValue;
    if (p.a_type == Precision::bf16 && p.b_type == Precision::bf16) return run_wide(p, s);
    if (p.a_type == Precision::f32 && p.b_type == Precision::bf16) return run<float, uint16_t>(p, s);
    if (p.a_type == Precision::bf16 && p.b_type == Precision::f32) return run<uint16_t, float>(p, s);
    return hipErrorInvalidValue;
}

}  // namespace esp
