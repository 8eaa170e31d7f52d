// Dequant-fused MFMA GEMM for more than two activation rows (prompt prefill, batched verify, batch-8
// microbenchmarks):   y[m][n] = sum_k x[m][k] * dequant(W)[n][k],   fp16 operands, fp32 accumulation.
//
// Replaces the per-token vDSP_mmul calls the reference issues while it walks a prompt
// (RealModelInferenceEngine.swift:6674-6697 inside the prefill loop :6365-6375) by one pass over the
// packed weights per block of rows.
//
// launch_gemm chooses: few rows or small matrices with exact weights (rows_gemm.hip), fp16 matrices (wide_gemm.hip), up to eight rows of Q4_K (gemm_rows_kernel below), blocks of rows
// (block_gemm.hip), and for what is left - columns that are no multiple of 128 - gemm_kernel:
//   * a workgroup of four wavefronts owns 128 weight rows (n) x MT activation rows (m) and walks K in
//     tiles of 64;
//   * per K tile every thread fetches the packed bytes of (one weight row, one half of the tile) with
//     128-bit loads, turns them into 32 fp16 weights in registers (nibble / byte exponent tricks, one
//     packed fp16 multiply-add with the block's scale and minimum) and writes them to LDS; the fp16
//     activations of the tile are copied to LDS next to them;
//   * every weight reaches the matrix core as its dequantised value rounded to fp16 exactly once
//     (one exact packed fp16 product);
//   * the Q4_0 / Q8_0 exponent tricks yield elements in (0,2,1,3) order inside every group of four; the
//     activations are stored with the same swap, which costs nothing because a dot product does not care
//     about the order of k as long as both operands agree;
//   * v_mfma_f32_32x32x16_f16: activations are the A operand (rows m), weights the B operand (columns
//     n), so a lane's 16 accumulators belong to one weight row and 16 activation rows;
//   * the global loads of several tiles ahead are in flight while the matrix cores work on tile t;
//   * when the (n, m) grid is too small to fill the chip, K is split over grid.y and a small kernel
//     adds the partial sums in split order (deterministic, no atomics).
#include "../common.h"
#include "decode_ops.h"
#include "block_gemm.h"
#include "wide_gemm.h"
#include "rows_gemm.h"
#include "stream_gemm.h"
#include <atomic>
#include <type_traits>

namespace esp {
namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32;

constexpr int KT = 64;        // k per tile
constexpr int LDK = KT + 8;   // fp16 per LDS row: 144 bytes, so eight rows cover all banks
constexpr int NT = 128;       // weight rows per workgroup: two threads per row

struct GemmArgs {
    const uint8_t *qs;
    const uint16_t *scales;
    size_t qs_row_bytes;
    int N, K, M;
    const uint16_t *x;      // [M][K] fp16
    float *y;               // [M][N]
    const float *residual;  // [M][N] or null
    float *partial;         // [splits][M][N] when gridDim.y > 1
    int tiles_per_split;
    uint16_t *swiglu_out;   // tile kernel without split-K only: fp16 [M][N / 2] instead of y
};

__device__ __forceinline__ h2 as_h2(u32 v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ u32 as_u32(h2 v) { return __builtin_bit_cast(u32, v); }
__device__ __forceinline__ float half_bits_to_float(u32 bits16) { return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16); }
__device__ __forceinline__ half8 as_half8(const uint4 &v) { return __builtin_bit_cast(half8, v); }
__device__ __forceinline__ h2 splat(float v) { const _Float16 h = (_Float16)v; return h2{h, h}; }
__device__ __forceinline__ u32 dword_of(const uint4 &v, int k) { return k == 0 ? v.x : k == 1 ? v.y : k == 2 ? v.z : v.w; }
__device__ __forceinline__ uint4 swap_middle(const uint4 &v) {
    uint4 p;
    p.x = __builtin_amdgcn_perm(v.y, v.x, 0x05040100u);
    p.y = __builtin_amdgcn_perm(v.y, v.x, 0x07060302u);
    p.z = __builtin_amdgcn_perm(v.w, v.z, 0x05040100u);
    p.w = __builtin_amdgcn_perm(v.w, v.z, 0x07060302u);
    return p;
}

// The packed bytes one thread holds for (weight row, half h of a K tile), per format.
template <int FMT>
struct Raw;
template <>
struct Raw<FMT_Q4_0> { uint4 q; u32 d; };        // one block
template <>
struct Raw<FMT_Q8_0> { uint4 q0, q1; u32 d; };   // one block

template <int FMT>
__device__ __forceinline__ Raw<FMT> fetch_raw(const GemmArgs &a, int row, int tile, int h) {
    Raw<FMT> r;
    const uint8_t *base = a.qs + (size_t)row * a.qs_row_bytes;
    if constexpr (FMT == FMT_Q4_0) {
        const int block = tile * 2 + h;
        r.q = *reinterpret_cast<const uint4 *>(base + (size_t)block * 16);
        r.d = a.scales[(size_t)row * (a.K / 32) + block];
    } else {
        const int block = tile * 2 + h;
        const uint4 *q = reinterpret_cast<const uint4 *>(base + (size_t)block * 32);
        r.q0 = q[0];
        r.q1 = q[1];
        r.d = a.scales[(size_t)row * (a.K / 32) + block];
    }
    return r;
}

// Byte `idx` (0..11) of the twelve scale bytes that follow d and dmin in a Q4_K header.
__device__ __forceinline__ u32 scale_byte(const uint4 &hdr, int idx) {
    const u32 word = idx < 4 ? hdr.y : idx < 8 ? hdr.z : hdr.w;
    return (word >> ((idx & 3) * 8)) & 0xFFu;
}
// ggml's get_scale_min_k4
__device__ __forceinline__ void q4k_scale_min(const uint4 &hdr, int j, float &sc, float &m) {
    if (j < 4) {
        sc = (float)(scale_byte(hdr, j) & 63u);
        m = (float)(scale_byte(hdr, j + 4) & 63u);
    } else {
        sc = (float)((scale_byte(hdr, j + 4) & 0xFu) | ((scale_byte(hdr, j - 4) >> 6) << 4));
        m = (float)((scale_byte(hdr, j + 4) >> 4) | ((scale_byte(hdr, j) >> 6) << 4));
    }
}

// Four weights of dword `w` per call: nibbles at bits 0..3 (offset 1024) or 4..7 (offset 64) become exact
// fp16 integers, then w = n * s - dm in packed fp16 (one rounding per weight).
__device__ __forceinline__ uint2 nibbles_to_half(u32 w, bool high, h2 s, h2 dm) {
    const u32 mask = high ? 0x00F000F0u : 0x000F000Fu, magic = high ? 0x54005400u : 0x64006400u;
    const h2 off = high ? h2{(_Float16)64.0f, (_Float16)64.0f} : h2{(_Float16)1024.0f, (_Float16)1024.0f};
    const h2 n02 = as_h2((w & mask) | magic) - off, n13 = as_h2(((w >> 8) & mask) | magic) - off;
    return make_uint2(as_u32(__builtin_elementwise_fma(n02, s, -dm)), as_u32(__builtin_elementwise_fma(n13, s, -dm)));
}

// Writes the thread's 32 fp16 weights into its LDS row (`wrow` points at k = 0 of the tile).
// Element order inside each group of four is (0,2,1,3).
template <int FMT>
__device__ __forceinline__ void dequant_to_lds(const Raw<FMT> &r, int h, _Float16 *wrow) {
    if constexpr (FMT == FMT_Q4_0) {
        // byte j: low nibble = element j, high nibble = element j + 16; w = (n - 8) * d
        const h2 s = splat(half_bits_to_float(r.d)), dm = splat(8.0f * half_bits_to_float(r.d));
        uint2 lo[4], hi[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            lo[k] = nibbles_to_half(dword_of(r.q, k), false, s, dm);
            hi[k] = nibbles_to_half(dword_of(r.q, k), true, s, dm);
        }
        uint4 *p = reinterpret_cast<uint4 *>(wrow + 32 * h);
        p[0] = make_uint4(lo[0].x, lo[0].y, lo[1].x, lo[1].y);
        p[1] = make_uint4(lo[2].x, lo[2].y, lo[3].x, lo[3].y);
        p[2] = make_uint4(hi[0].x, hi[0].y, hi[1].x, hi[1].y);
        p[3] = make_uint4(hi[2].x, hi[2].y, hi[3].x, hi[3].y);
    } else {
        const h2 s = splat(half_bits_to_float(r.d)), off = h2{(_Float16)1152.0f, (_Float16)1152.0f};   // 1024 + 128
        uint4 *p = reinterpret_cast<uint4 *>(wrow + 32 * h);
#pragma unroll
        for (int half = 0; half < 2; half++) {
            const uint4 &q = half ? r.q1 : r.q0;
            u32 out[8];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const u32 t = dword_of(q, k) ^ 0x80808080u;   // signed -> biased
                const h2 f02 = as_h2(__builtin_amdgcn_perm(0x64646464u, t, 0x04020400u)) - off;
                const h2 f13 = as_h2(__builtin_amdgcn_perm(0x64646464u, t, 0x04030401u)) - off;
                out[2 * k] = as_u32(f02 * s);
                out[2 * k + 1] = as_u32(f13 * s);
            }
            p[2 * half] = make_uint4(out[0], out[1], out[2], out[3]);
            p[2 * half + 1] = make_uint4(out[4], out[5], out[6], out[7]);
        }
    }
}

// WM x WN wavefronts, each TM x TN MFMA tiles of 32 x 32: the workgroup covers 32*WM*TM rows of x and
// 32*WN*TN = 128 weight rows.  DEPTH tiles of packed weights and activations are in flight in registers
// (a slot is refilled as soon as its tile has gone to LDS), and LDS holds two tiles so that one barrier
// per tile is enough: tile t+1 is written while other wavefronts still read tile t.
template <int FMT, int WM, int WN, int TM, int TN, int DEPTH>
__global__ __launch_bounds__(64 * WM * WN) void gemm_kernel(GemmArgs a) {
    constexpr int THREADS = 64 * WM * WN, NTILE = 32 * WN * TN;   // two threads per weight row dequantise
    static_assert(2 * NTILE == THREADS, "one (weight row, half tile) per thread");
    constexpr int MT = 32 * WM * TM;
    constexpr int XV = MT * KT / 8 / THREADS;   // 128-bit pieces of x per thread per tile
    static_assert(XV >= 1, "tile too small for the copy loop");
    __shared__ _Float16 xt[2][MT * LDK];
    __shared__ _Float16 wt[2][NTILE * LDK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int n0 = blockIdx.x * NTILE, m0 = blockIdx.z * MT;
    const int tiles = a.K / KT;
    const int t_begin = blockIdx.y * a.tiles_per_split;
    const int t_end = t_begin + a.tiles_per_split < tiles ? t_begin + a.tiles_per_split : tiles;

    // dequantisation role: weight row and half of the tile
    const int wr = tid >> 1, wh = tid & 1;
    const int w_row = n0 + wr < a.N ? n0 + wr : a.N - 1;   // clamped, the result is never stored

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    auto fetch_x = [&](int tile, uint4 (&xv)[XV]) {
#pragma unroll
        for (int i = 0; i < XV; i++) {
            const int piece = tid + i * THREADS, row = piece >> 3, part = piece & 7;   // eight pieces per row
            const int m = m0 + row < a.M ? m0 + row : a.M - 1;   // rows beyond M repeat the last one; their results are never stored
            xv[i] = reinterpret_cast<const uint4 *>(a.x + (size_t)m * a.K + (size_t)tile * KT)[part];
        }
    };

    // Slot j % DEPTH holds the packed bytes and activations of tile t_begin + j.  Staging a tile (dequantise into LDS,
    // copy the activations, refill the slot DEPTH tiles ahead) sits in the same barrier interval as the matrix-core work
    // on the tile before it, so the vector ALU and the LDS writes run in the shadow of the MFMAs of the same wavefront.
    // Tile indices beyond the last are clamped: the extra stage of the last interval is in bounds and never read.
    Raw<FMT> raw[DEPTH];
    uint4 xv[DEPTH][XV];
    const int t_last = t_end - 1;
#pragma unroll
    for (int d = 0; d < DEPTH; d++) {
        const int tile = t_begin + d < t_last ? t_begin + d : t_last;
        raw[d] = fetch_raw<FMT>(a, w_row, tile, wh);
        fetch_x(tile, xv[d]);
    }
    static_assert(4 % DEPTH == 0, "the main loop is unrolled by four");
    auto stage = [&](int S, int tile, int buf) {   // S is a constant after unrolling
        dequant_to_lds<FMT>(raw[S], wh, wt[buf] + wr * LDK);
#pragma unroll
        for (int i = 0; i < XV; i++) {
            const int piece = tid + i * THREADS, row = piece >> 3, part = piece & 7;
            *reinterpret_cast<uint4 *>(xt[buf] + row * LDK + part * 8) = swap_middle(xv[S][i]);
        }
        const int ahead = tile + DEPTH < t_last ? tile + DEPTH : t_last;
        raw[S] = fetch_raw<FMT>(a, w_row, ahead, wh);
        fetch_x(ahead, xv[S]);
    };
    stage(0, t_begin, 0);
    __syncthreads();
    for (int t0 = t_begin; t0 < t_end; t0 += 4) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int t = t0 + u, buf = u & 1;
            if (t < t_end) {
#pragma unroll
                for (int ks = 0; ks < KT / 16; ks++) {
                    const int kk = ks * 16 + 8 * (lane >> 5);
                    half8 af[TM], bf[TN];
#pragma unroll
                    for (int i = 0; i < TM; i++)
                        af[i] = *reinterpret_cast<const half8 *>(xt[buf] + ((wm * TM + i) * 32 + (lane & 31)) * LDK + kk);
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        bf[j] = *reinterpret_cast<const half8 *>(wt[buf] + ((wn * TN + j) * 32 + (lane & 31)) * LDK + kk);
#pragma unroll
                    for (int i = 0; i < TM; i++)
#pragma unroll
                        for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
                }
                stage((u + 1) % DEPTH, t + 1, buf ^ 1);
                __syncthreads();
            }
        }
    }

    // accumulator r of lane l: row 8*(r/4) + 4*(l/32) + r%4, column l%32 of the 32 x 32 tile
    if (a.swiglu_out) {   // rows of W are (gate, up) pairs: even lanes hold gate, their right neighbours up (:6825-6827, :6337)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int n = n0 + (wn * TN + j) * 32 + (lane & 31);
                // a pair of lanes holds (gate, up) of one unit for 16 rows; the even lane finishes the even accumulators, the
                // odd lane the odd ones, so that no lane idles through the tanh
                const bool odd = lane & 1;
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const float a0 = acc[i][j][2 * k], a1 = acc[i][j][2 * k + 1];
                    const float p0 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, a0), 0xB1, 0xF, 0xF, false));   // quad_perm [1,0,3,2]
                    const float p1 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, a1), 0xB1, 0xF, 0xF, false));
                    const float g = odd ? p1 : a0, u = odd ? a1 : p0;
                    const int r = 2 * k + (odd ? 1 : 0);
                    const int m = m0 + (wm * TM + i) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    if (m < a.M && (n | 1) < a.N) {
                        const float silu = g * __builtin_amdgcn_rcpf(1.0f + __expf(-g));   // = 0.5 g (1 + tanh(0.5 g)), a fifth of tanhf's instructions
                        a.swiglu_out[(size_t)m * (a.N / 2) + n / 2] = __builtin_bit_cast(uint16_t, (_Float16)__fmul_rn(silu, u));
                    }
                }
            }
        return;
    }
    const bool split = gridDim.y > 1;
    float *out = split ? a.partial + (size_t)blockIdx.y * a.M * a.N : a.y;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int n = n0 + (wn * TN + j) * 32 + (lane & 31);
            auto row_of = [&](int r) { return m0 + (wm * TM + i) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); };
            if (!split && a.residual) {
                float res[16];   // requested together: y may be the residual's own memory, and a load behind each store is a trip to memory each
#pragma unroll
                for (int r = 0; r < 16; r++) res[r] = a.residual[(size_t)(row_of(r) < a.M ? row_of(r) : a.M - 1) * a.N + (n < a.N ? n : a.N - 1)];
#pragma unroll
                for (int r = 0; r < 16; r++) if (row_of(r) < a.M && n < a.N) out[(size_t)row_of(r) * a.N + n] = res[r] + acc[i][j][r];
            } else {
#pragma unroll
                for (int r = 0; r < 16; r++) if (row_of(r) < a.M && n < a.N) out[(size_t)row_of(r) * a.N + n] = acc[i][j][r];
            }
        }
}

constexpr int CK = 256;        // k per activation stage of the kernel below

// ---------------------------------------------------------------------------------------------
// Up to eight activation rows against Q4_K weights without dequantising them (three vector operations per weight however few rows
// there are).  The weights never touch LDS: a lane of the B operand of v_mfma_f32_32x32x16_f16 holds eight consecutive k of ONE column, so a lane loads packed bytes of its
// own weight row; lanes 0..31 and 32..63 of a wavefront take the two halves of each 64-k tile of the same 32 weight rows.  The B operand is the nibble itself under an fp16 exponent, as in the GEMV kernels: one
// v_and_or_b32 turns two low nibbles into (64 + n/16, 64 + n/16) and two high nibbles into (4 + n/16, 4 + n/16),
// exactly; two MFMAs contract a 32-weight sub-block into sum (offset + n/16) x with exact products, and scale and
// minimum of the sub-block are folded into the few accumulator registers that hold real rows afterwards:
//     sum_k (d sc n_k - dmin m) x_k = (16 d sc) raw - (16 d sc offset + dmin m) sum_k x_k,
// with the sums of the activations over each sub-block computed once per workgroup while they are staged.
// Only the activations go through LDS, in (0,2,1,3) order inside fours, which is how the masked nibble pairs come out; the rows 0..7 are
// accumulator registers 0..3 of a lane.
__device__ __forceinline__ float quad_sum(float v) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false));   // quad_perm [1,0,3,2]
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, false));   // quad_perm [2,3,0,1]
    return v;
}

// The workgroup owns 32 weight rows and its WAVES wavefronts split K between them, so a launch has one workgroup per 32 rows
// whatever K is, needs no split-K workspace and no reduce launch; the wavefronts' partial results meet in LDS and are added
// in wavefront order.  The activations are staged a span of SPAN chunks (of 256 k) at a time into one of two LDS buffers: the
// next span's are loaded into registers before the current span is computed and written after it, one barrier per span.
// Inside a span wavefront w takes chunks w, w + WAVES, ...; the packed weights of its chunks of the next two spans are always
// in flight (they do not wait for the staging).  Short spans measure faster than long ones (one chunk per wavefront and span:
// 15.7 us for 14336 x 4096 against 18.2 us with two and 17.9 us with all of K staged at once), and eight wavefronts
// faster than four when the rows fill no more than one workgroup per compute unit.
constexpr int kRowsMaxRows = 8;
template <int WAVES, int SPAN> constexpr size_t rows_lds_bytes() {
    return 2 * ((size_t)kRowsMaxRows * (SPAN * CK + 8) * 2 + (size_t)SPAN * 8 * kRowsMaxRows * 4) + (size_t)WAVES * 4 * 64 * 4;
}

struct RowsChunk { uint4 hdr, q[4]; };
__device__ __forceinline__ RowsChunk fetch_rows_chunk(const GemmArgs &a, int row, int chunk, int h) {
    RowsChunk c;
    const uint8_t *blk = a.qs + (size_t)row * a.qs_row_bytes + (size_t)chunk * 144;
    c.hdr = *reinterpret_cast<const uint4 *>(blk);
#pragma unroll
    for (int t = 0; t < 4; t++) c.q[t] = *reinterpret_cast<const uint4 *>(blk + 16 + t * 32 + h * 16);
    return c;
}

template <int WAVES, int SPAN>
__global__ __launch_bounds__(WAVES * 64, WAVES == 4 ? 2 : 1) void gemm_rows_kernel(GemmArgs a) {
    constexpr int MR = kRowsMaxRows, THREADS = WAVES * 64, LDW = SPAN * CK + 8;
    constexpr int CPW = SPAN / WAVES;                     // chunks per wavefront and span
    constexpr int PIECES = MR * SPAN * 32 / THREADS;      // 128-bit pieces of x per thread and span
    extern __shared__ uint4 rows_smem[];
    _Float16 *xt_base = reinterpret_cast<_Float16 *>(rows_smem);               // [2][MR][LDW]
    float *xsum_base = reinterpret_cast<float *>(xt_base + 2 * MR * LDW);      // [2][SPAN * 8 groups of 32][MR]
    float *red = xsum_base + 2 * SPAN * 8 * MR;                                // [WAVES][4][64]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5;
    const int n = blockIdx.x * 32 + (lane & 31);
    const int w_row = n < a.N ? n : a.N - 1;     // clamped, the result is never stored
    const int chunks = a.K / CK, spans = (chunks + SPAN - 1) / SPAN;
    // constants of the nibble trick, hidden from the optimiser so that (w & mask) | magic stays one v_and_or_b32
    u32 mask_lo = 0x000F000Fu, mask_hi = 0x00F000F0u, magic_lo = 0x54005400u, magic_hi = 0x44004400u;
    asm volatile("" : "+s"(mask_lo), "+s"(mask_hi));
    asm volatile("" : "+v"(magic_lo), "+v"(magic_hi));
    auto pattern_lo = [&](u32 w0, u32 w1) { return as_half8(make_uint4((w0 & mask_lo) | magic_lo, ((w0 >> 8) & mask_lo) | magic_lo, (w1 & mask_lo) | magic_lo, ((w1 >> 8) & mask_lo) | magic_lo)); };
    auto pattern_hi = [&](u32 w0, u32 w1) { return as_half8(make_uint4((w0 & mask_hi) | magic_hi, ((w0 >> 8) & mask_hi) | magic_hi, (w1 & mask_hi) | magic_hi, ((w1 >> 8) & mask_hi) | magic_hi)); };

    float total[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    auto chunk_of = [&](int sp, int j) { return sp * SPAN + j * WAVES + wave; };
    RowsChunk ring[2 * CPW];
#pragma unroll
    for (int q = 0; q < 2 * CPW; q++)
        if (chunk_of(q / CPW, q % CPW) < chunks) ring[q] = fetch_rows_chunk(a, w_row, chunk_of(q / CPW, q % CPW), h);

    uint4 xv[PIECES];
    auto load_x = [&](int sp) {
#pragma unroll
        for (int i = 0; i < PIECES; i++) {
            const int piece = tid + i * THREADS, row = piece / (SPAN * 32), part = piece % (SPAN * 32);
            const int k0 = sp * SPAN * CK + part * 8;
            xv[i] = row < a.M && k0 < a.K ? *reinterpret_cast<const uint4 *>(a.x + (size_t)row * a.K + k0) : make_uint4(0, 0, 0, 0);
        }
    };
    // (0,2,1,3) order inside fours; alongside, per group of 32, the sum of the activations
    auto store_x = [&](int buf) {
        _Float16 *xt = xt_base + buf * MR * LDW;
        float *xsum = xsum_base + buf * SPAN * 8 * MR;
#pragma unroll
        for (int i = 0; i < PIECES; i++) {
            const int piece = tid + i * THREADS, row = piece / (SPAN * 32), part = piece % (SPAN * 32);
            *reinterpret_cast<uint4 *>(xt + row * LDW + part * 8) = swap_middle(xv[i]);
            const h2 p0 = as_h2(xv[i].x), p1 = as_h2(xv[i].y), p2 = as_h2(xv[i].z), p3 = as_h2(xv[i].w);
            float sum = (((float)p0.x + (float)p0.y) + ((float)p1.x + (float)p1.y)) + (((float)p2.x + (float)p2.y) + ((float)p3.x + (float)p3.y));
            sum = quad_sum(sum);                 // the four pieces of a group of 32 sit in one quad of lanes
            if ((part & 3) == 0) xsum[(part >> 2) * MR + row] = sum;
        }
    };
    auto compute_span = [&](int sp, auto parity) {
        constexpr int P = decltype(parity)::value;
        const _Float16 *xt = xt_base + P * MR * LDW;
        const float *xsum = xsum_base + P * SPAN * 8 * MR;
#pragma unroll
        for (int j = 0; j < CPW; j++) {
            const int c = chunk_of(sp, j);
            if (c < chunks) {
                const RowsChunk r = ring[P * CPW + j];
                if (chunk_of(sp + 2, j) < chunks) ring[P * CPW + j] = fetch_rows_chunk(a, w_row, chunk_of(sp + 2, j), h);
                const int local = j * WAVES + wave;   // chunk index inside the span
                // rows of x beyond MR alias real ones: they only reach accumulator registers that are never read
                const _Float16 *xchunk = xt + ((lane & 31) & (MR - 1)) * LDW + local * CK;
                const float dd = half_bits_to_float(r.hdr.x & 0xFFFFu), dmin = half_bits_to_float(r.hdr.x >> 16);
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    float sc_lo, m_lo, sc_hi, m_hi;
                    q4k_scale_min(r.hdr, 2 * t, sc_lo, m_lo);
                    q4k_scale_min(r.hdr, 2 * t + 1, sc_hi, m_hi);
                    const float a_lo = 16.0f * dd * sc_lo, b_lo = 64.0f * a_lo + dmin * m_lo;
                    const float a_hi = 16.0f * dd * sc_hi, b_hi = 4.0f * a_hi + dmin * m_hi;
                    const u32 w0 = r.q[t].x, w1 = r.q[t].y, w2 = r.q[t].z, w3 = r.q[t].w;
                    const half8 f0 = pattern_lo(w0, w1), f1 = pattern_lo(w2, w3), f2 = pattern_hi(w0, w1), f3 = pattern_hi(w2, w3);
                    const _Float16 *xrow = xchunk + t * KT;
                    floatx16 lo, hi;
#pragma unroll
                    for (int i = 0; i < 16; i++) lo[i] = hi[i] = 0.0f;
                    lo = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8 *>(xrow + 16 * h), f0, lo, 0, 0, 0);
                    hi = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8 *>(xrow + 32 + 16 * h), f2, hi, 0, 0, 0);
                    lo = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8 *>(xrow + 16 * h + 8), f1, lo, 0, 0, 0);
                    hi = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8 *>(xrow + 40 + 16 * h), f3, hi, 0, 0, 0);
                    const float4 xs_lo = *reinterpret_cast<const float4 *>(xsum + (local * 8 + 2 * t) * MR + 4 * h);
                    const float4 xs_hi = *reinterpret_cast<const float4 *>(xsum + (local * 8 + 2 * t + 1) * MR + 4 * h);
                    const float sl[4] = {xs_lo.x, xs_lo.y, xs_lo.z, xs_lo.w}, sh[4] = {xs_hi.x, xs_hi.y, xs_hi.z, xs_hi.w};
#pragma unroll
                    for (int i = 0; i < 4; i++) {   // accumulator registers 0..3 of a lane: rows 4 (lane / 32) + i
                        float acc = total[i];
                        acc = __builtin_fmaf(lo[i], a_lo, acc);
                        acc = __builtin_fmaf(-b_lo, sl[i], acc);
                        acc = __builtin_fmaf(hi[i], a_hi, acc);
                        acc = __builtin_fmaf(-b_hi, sh[i], acc);
                        total[i] = acc;
                    }
                    __builtin_amdgcn_sched_barrier(0);   // one sub-block pair at a time keeps the accumulators few
                }
            }
        }
    };
    auto span_step = [&](int sp, auto parity) {
        constexpr int P = decltype(parity)::value;
        const bool more = sp + 1 < spans;
        if (more) load_x(sp + 1);
        compute_span(sp, parity);
        if (more) store_x(1 - P);
        __syncthreads();
    };

    load_x(0);
    store_x(0);
    __syncthreads();
    for (int sp = 0; sp < spans; sp += 2) {
        span_step(sp, std::integral_constant<int, 0>{});
        if (sp + 1 < spans) span_step(sp + 1, std::integral_constant<int, 1>{});
    }

    // ---- the wavefronts' shares of K meet in LDS; wavefront 0 adds them in order and writes the rows ----
#pragma unroll
    for (int i = 0; i < 4; i++) red[(wave * 4 + i) * 64 + lane] = total[i];
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float v = red[i * 64 + lane];
#pragma unroll
            for (int w = 1; w < WAVES; w++) v += red[(w * 4 + i) * 64 + lane];
            const int m = 4 * h + i;
            if (m < a.M && n < a.N) {
                const size_t o = (size_t)m * a.N + n;
                a.y[o] = a.residual ? a.residual[o] + v : v;
            }
        }
    }
}

// y = (residual +) sum over splits of partial, in split order
__global__ void gemm_reduce_kernel(const float *partial, int splits, size_t count, const float *residual, float *y) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    float s = partial[i];
    for (int k = 1; k < splits; k++) s += partial[(size_t)k * count + i];
    y[i] = residual ? residual[i] + s : s;
}

template <int FMT, int WM, int WN, int TM, int TN, int DEPTH>
hipError_t launch_tile(const GemmArgs &a, int splits, hipStream_t stream) {
    constexpr int MT = 32 * WM * TM;
    constexpr int NTILE = 32 * WN * TN;
    dim3 grid((a.N + NTILE - 1) / NTILE, splits, (a.M + MT - 1) / MT);
    hipLaunchKernelGGL((gemm_kernel<FMT, WM, WN, TM, TN, DEPTH>), grid, dim3(64 * WM * WN), 0, stream, a);
    return hipGetLastError();
}

hipError_t launch_reduce(const GemmArgs &a, int splits, hipStream_t stream) {
    const size_t count = (size_t)a.M * a.N;
    hipLaunchKernelGGL(gemm_reduce_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, stream, a.partial, splits, count, a.residual, a.y);
    return hipGetLastError();
}

// splits so that about `target` workgroups exist, each with at least `min_units` units of K
int choose_splits(int blocks, int units, int min_units, int target, const GemmArgs &a, size_t workspace_floats) {
    if (!a.partial || blocks >= target) return 1;
    int splits = (target + blocks - 1) / blocks;
    if (splits > units / min_units) splits = units / min_units;
    if (splits < 1) splits = 1;
    while (splits > 1 && (size_t)splits * a.M * a.N > workspace_floats) splits--;
    return splits;
}

// Up to eight rows of Q4_K: one workgroup per 32 weight rows, K split over its wavefronts.  The kernels' LDS (above 64 KB) is dynamic: the limit is raised once per kernel and device.
hipError_t launch_few_rows(const GemmArgs &a, hipStream_t stream) {
    const int groups = (a.N + 31) / 32;
    auto go = [&](auto kernel, int waves, size_t lds, std::atomic<uint64_t> &raised) {
        int device = 0;
        hipError_t err = hipGetDevice(&device);
        if (err != hipSuccess) return err;
        const uint64_t bit = 1ull << (device & 63);
        if (!(raised.load(std::memory_order_acquire) & bit)) {
            err = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (err != hipSuccess) return err;
            raised.fetch_or(bit, std::memory_order_release);
        }
        hipLaunchKernelGGL(kernel, dim3(groups), dim3(waves * 64), lds, stream, a);
        return hipGetLastError();
    };
    static std::atomic<uint64_t> raised8{0}, raised4{0};
    if (groups <= 256) return go(gemm_rows_kernel<8, 8>, 8, rows_lds_bytes<8, 8>(), raised8);
    return go(gemm_rows_kernel<4, 4>, 4, rows_lds_bytes<4, 4>(), raised4);
}

// gemm_kernel by size.  (Eight wavefronts on a 128 x 256 tile measure 2-5 % faster at 4096 and more weight rows and 10 % slower at 1024; a 256 x 256 tile is 25 % slower: not instantiated.)
template <int FMT>
hipError_t launch_tiles(const GemmParams &p, GemmArgs a, int *used_splits, hipStream_t stream) {
    const int tiles = a.K / KT, mt = a.M <= 32 ? 32 : a.M <= 64 ? 64 : 128;
    int splits = choose_splits((a.N + NT - 1) / NT * ((a.M + mt - 1) / mt), tiles, 8, 1024, a, p.workspace_floats);
    a.tiles_per_split = ((tiles + splits - 1) / splits + 3) & ~3;   // every split starts on a multiple of four tiles
    *used_splits = splits = (tiles + a.tiles_per_split - 1) / a.tiles_per_split;
    if (splits == 1 && a.N % 2 == 0) a.swiglu_out = p.swiglu_out;
    if (mt == 32) return launch_tile<FMT, 1, 4, 1, 1, 4>(a, splits, stream);
    if (mt == 64) return launch_tile<FMT, 1, 4, 2, 1, 4>(a, splits, stream);
    return launch_tile<FMT, 2, 2, 2, 2, 2>(a, splits, stream);
}

// p.swiglu_out (may be null) is written by a kernel that runs without shares of K; *fused tells the caller.  Partial sums are added by gemm_reduce_kernel, or left to the caller's next kernel
// when it asked for that.
template <int FMT>
hipError_t launch_format(const GemmParams &p, GemmArgs a, bool *fused, int *deferred_splits, hipStream_t stream) {
    if (FMT == FMT_Q4_K && a.M <= kRowsMaxRows) return launch_few_rows(a, stream);
    a.partial = p.workspace;
    int splits = 1;
    hipError_t e;
    if constexpr (FMT == FMT_F16) {
        const WideForm f = wide_gemm_form(p);
        if (!f.bm) return hipErrorInvalidValue;
        splits = f.splits;
        e = launch_wide_gemm(p, f, stream);
    } else {
        if (block_gemm_takes(p)) e = launch_block_gemm(p, &splits, stream);
        else if constexpr (FMT == FMT_Q4_K) return hipErrorInvalidValue;   // whole super-blocks: block_gemm.hip takes them all
        else e = launch_tiles<FMT>(p, a, &splits, stream);
    }
    *fused = splits == 1 && p.swiglu_out && a.N % 2 == 0;
    if (e != hipSuccess || splits == 1) return e;
    if (deferred_splits) { *deferred_splits = splits; return hipSuccess; }
    return launch_reduce(a, splits, stream);
}

}  // namespace

bool gemm_keeps_weights(const GemmParams &p) {
    return p.w.format == FMT_F16 || rows_gemm_takes(p) || (p.w.format == FMT_Q4_K ? p.rows <= kRowsMaxRows : block_gemm_takes(p) && block_gemm_exact(p));
}

hipError_t launch_gemm(const GemmParams &params, hipStream_t stream) {
    GemmParams p = params;
    const DeviceMatrix &w = p.w;
    if (!w.qs || !p.x || !p.y || p.rows <= 0 || w.rows <= 0 || w.cols <= 0 || w.cols % KT != 0 || w.qs_row_bytes % 16 != 0) return hipErrorInvalidValue;
    if ((w.format == FMT_Q8_0 || w.format == FMT_Q4_0) && !w.scales) return hipErrorInvalidValue;
    if (w.format == FMT_Q4_K && w.cols % 256 != 0) return hipErrorInvalidValue;
    if (p.deferred_splits) *p.deferred_splits = 1;
    // single products of up to eight rows of Q4_0 keep their weights, whoever asks, and so may take either kernel that does (8 rows, in rows_gemm.hip -> with shares of K and
    // their sum: 768 x 768 3.9 -> 6.9 us, 2048 x 2048 6.7 -> 8.6, 2048 x 5632 10.3 -> 9.6)
    if (w.format == FMT_Q4_0 && p.rows <= 8 && w.cols % 128 == 0) p.unrounded = true;
    if (stream_gemm_takes(p)) {
        int shares = 1;
        const hipError_t e = launch_stream_gemm(p, &shares, stream);
        if (p.deferred_splits) *p.deferred_splits = shares;
        return e;
    }
    if (rows_gemm_takes(p)) return launch_rows_gemm(p, stream);
    GemmArgs a{};
    a.qs = w.qs; a.scales = w.scales; a.qs_row_bytes = w.qs_row_bytes; a.N = w.rows; a.K = w.cols; a.M = p.rows;
    a.x = p.x; a.y = p.y; a.residual = p.residual;
    bool fused = false;
    // SiLU(gate) * up outside the epilogue adds split-K partial sums itself: one launch less (93 rows of 11264 gate|up rows: a reduction of 5.3 us)
    int splits = 1;
    int *const deferred = p.swiglu_out ? &splits : p.deferred_splits;
    hipError_t e;
    switch (w.format) {
    case FMT_Q4_K: e = launch_format<FMT_Q4_K>(p, a, &fused, deferred, stream); break;
    case FMT_Q4_0: e = launch_format<FMT_Q4_0>(p, a, &fused, deferred, stream); break;
    case FMT_Q8_0: e = launch_format<FMT_Q8_0>(p, a, &fused, deferred, stream); break;
    case FMT_F16: e = launch_format<FMT_F16>(p, a, &fused, deferred, stream); break;
    default: return hipErrorInvalidValue;   // fp32 matrices stay on the GEMV path
    }
    if (e != hipSuccess || !p.swiglu_out || fused) return e;
    if (w.rows % 2 != 0 || p.residual) return hipErrorInvalidValue;
    return launch_swiglu(splits > 1 ? p.workspace : p.y, splits, (size_t)p.rows * w.rows, p.rows, w.rows / 2, p.swiglu_out, stream);
}

}  // namespace esp
