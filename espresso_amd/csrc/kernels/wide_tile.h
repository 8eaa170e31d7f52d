// Products of three and more rows of activations on the matrix cores, y[m][n] = sum_k x[m][k] w[n][k], both operands in sixteen bits: the walk over K that wide_gemm.hip (fp16) and
// dense_gemm.hip (bf16) share.
//
// A workgroup is eight wavefronts, WM x WN of them, each with TM x TN products of 32 x 32; it walks K in steps of 64 through two LDS buffers that hold both operands as sixteen-bit values.
// What bounds a product of many rows is neither memory nor the matrix cores alone but how long a wavefront waits for its fragments, so
//   * tiles are as large as the registers allow (256 x 256: six fragments of LDS for eight products; 64 x 64 a wavefront, as in the 128 x 128 tiles of four wavefronts, reads eight for eight);
//   * small tiles, which few rows take, keep four steps on their way from memory in registers (8 rows of 10368 x 2048, 81 workgroups: 22 us with one step, 16.3);
//   * fragments of the next sixteen k are read while these are multiplied, also across the step: the barrier stands before the step's last sixteen k, whose fragments are in registers
//     by then, so one barrier a step suffices and the first fragments behind it are on their way before the products end;
//   * writes to the other buffer and loads of a later step are spread over the step (sched_group_barrier: product, read, write, load by turns; left to the compiler 4 to 8 % slower).
// Rows of LDS are 144 bytes apart, so that reads of eight rows fall on all banks.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <atomic>
#include <type_traits>

namespace esp {
namespace wide {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 512, kStep = 64, kPitch = 72;   // k of a step; sixteen-bit values between the rows in LDS

template <int WM, int WN, int TM, int TN>
struct Tile {
    static_assert(WM * WN == 8, "eight wavefronts");
    static constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN, kBuffer = (BM + BN) * kPitch;
    static constexpr size_t kLdsBytes = (size_t)2 * kBuffer * 2;
    static_assert(kLdsBytes <= 160 * 1024, "LDS of a compute unit");
    // Steps in registers on their way to LDS: small tiles are bound by the weights' way from memory, and what is in flight is all that shortens it
    static constexpr int kDepth = BM + BN <= 192 ? 4 : BM + BN <= 384 ? 2 : 1;
};

// The workgroup's place: workgroups of one die take neighbouring output tiles, the row tiles of one block of weights first.
struct Place { int m_tile, n_tile, split; };
__device__ __forceinline__ Place place_of(int m_tiles, int n_tiles, int block, int total) {
    const int die = block & 7, q8 = total >> 3, r8 = total & 7;
    const int unit = die * q8 + (die < r8 ? die : r8) + (block >> 3);
    const int rest = unit / m_tiles;
    return {unit % m_tiles, rest % n_tiles, rest / n_tiles};
}
__device__ __forceinline__ Place place_of(int m_tiles, int n_tiles) { return place_of(m_tiles, n_tiles, blockIdx.x, gridDim.x); }

// The limit of dynamic LDS, raised once per kernel and device (`raised`: the kernel's own).
inline hipError_t raise_lds_limit(const void *kernel, size_t lds, std::atomic<uint64_t> &raised) {
    int device = 0;
    hipError_t err = hipGetDevice(&device);
    if (err != hipSuccess) return err;
    const uint64_t bit = 1ull << (device & 63);
    if (raised.load(std::memory_order_acquire) & bit) return hipSuccess;
    err = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err == hipSuccess) raised.fetch_or(bit, std::memory_order_release);
    return err;
}

// Sixteen (or eight) bytes at a uniform base and a lane's own 32-bit offset, one load without vector arithmetic: the offset is hidden from the optimiser where it is used, or its widening
// to 64 bits leaves the loop, takes two registers and an addition for each load.
template <class V>
__device__ __forceinline__ V load_at(const uint8_t *base, uint32_t offset) {
    asm volatile("" : "+v"(offset));
    return *reinterpret_cast<const V *>(base + offset);
}

// Rows of sixteen-bit values on their way to LDS, 64 k a step: the activations, and weights that need no unpacking.
template <int ROWS, int DEPTH>
struct Plain {
    static constexpr int kPieces = ROWS * 8 / kThreads;
    static_assert(ROWS * 8 % kThreads == 0 && kPieces >= 1, "whole pieces");
    const uint8_t *base;
    uint32_t offset[kPieces];   // bytes from base on
    uintx4 raw[DEPTH][kPieces];
    int last, at_lds;
    // rows row0 .. of a matrix of `count`: those beyond repeat the last one, never stored
    __device__ __forceinline__ Plain(const uint16_t *m, size_t ld, int row0, int count, size_t k0, int steps) : base(reinterpret_cast<const uint8_t *>(m + (size_t)row0 * ld + k0)), last(steps - 1) {
#pragma unroll
        for (int i = 0; i < kPieces; i++) {
            const int piece = threadIdx.x + i * kThreads, r = piece >> 3;
            offset[i] = (uint32_t)(row0 + r < count ? r : count - 1 - row0) * (uint32_t)(2 * ld) + (piece & 7) * 16;
        }
        at_lds = (threadIdx.x >> 3) * kPitch + (threadIdx.x & 7) * 8;
    }
    __device__ __forceinline__ void load_piece(int slot, int i, int s) { raw[slot][i] = load_at<uintx4>(base + (size_t)(s < last ? s : last) * (2 * kStep), offset[i]); }
    __device__ __forceinline__ void load(int slot, int s) {
#pragma unroll
        for (int i = 0; i < kPieces; i++) load_piece(slot, i, s);
    }
    // part PART of three of the step in slot SLOT to LDS, and step `next` on its way there
    template <int PART, int SLOT>
    __device__ __forceinline__ void stage(uint16_t *lds, int next) {
#pragma unroll
        for (int i = 0; i < kPieces; i++)
            if (i * 3 / kPieces == PART) {
                *reinterpret_cast<uintx4 *>(lds + at_lds + i * (kThreads / 8) * kPitch) = raw[SLOT][i];
                load_piece(SLOT, i, next);
            }
    }
};

template <bool BF16>
__device__ __forceinline__ floatx16 multiply(const uintx4 &a, const uintx4 &b, const floatx16 &c) {
    if constexpr (BF16) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
}

// acc[i][j] = rows 32 (wm TM + i) .. of the tile against weight rows 32 (wn TN + j) ..; a lane's accumulator r is row 8 (r / 4) + 4 (lane / 32) + r % 4, weight row lane % 32.
template <bool BF16, int WM, int WN, int TM, int TN, class Rows, class Weights>
__device__ __forceinline__ void walk(Rows &x, Weights &w, int steps, uint16_t *lds, floatx16 (&acc)[TM][TN]) {
    using T = Tile<WM, WN, TM, TN>;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave / WN, wn = wave % WN;
    const int fx = (wm * TM * 32 + (lane & 31)) * kPitch + 8 * (lane >> 5), fw = (T::BM + wn * TN * 32 + (lane & 31)) * kPitch + 8 * (lane >> 5);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;
    uintx4 xf[2][TM], wf[2][TN];
    auto fragments = [&](int slot, int buf, int ks) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < TN; j++) wf[slot][j] = *reinterpret_cast<const uintx4 *>(lds + buf * T::kBuffer + fw + j * 32 * kPitch + ks * 16);
#pragma unroll
        for (int i = 0; i < TM; i++) xf[slot][i] = *reinterpret_cast<const uintx4 *>(lds + buf * T::kBuffer + fx + i * 32 * kPitch + ks * 16);
    };
    constexpr int D = T::kDepth, U = D < 2 ? 2 : D;   // U steps are written out: buffers and slots by turns
    auto stage = [&](auto part, auto slot, int buf, int next) __attribute__((always_inline)) {
        x.template stage<decltype(part)::value, decltype(slot)::value>(lds + buf * T::kBuffer, next);
        w.template stage<decltype(part)::value, decltype(slot)::value>(lds + buf * T::kBuffer + T::BM * kPitch, next);
    };
    typedef std::integral_constant<int, 0> C0;
    typedef std::integral_constant<int, 1> C1;
    typedef std::integral_constant<int, 2> C2;
    typedef std::integral_constant<int, 3> C3;
#pragma unroll
    for (int i = 0; i < D; i++) {
        x.load(i, i);
        w.load(i, i);
    }
    stage(C0{}, C0{}, 0, D);
    stage(C1{}, C0{}, 0, D);
    stage(C2{}, C0{}, 0, D);
    __syncthreads();
    fragments(0, 0, 0);
    auto step = [&](auto turn, int s) __attribute__((always_inline)) {
        constexpr int B = decltype(turn)::value & 1;
        constexpr std::integral_constant<int, (decltype(turn)::value + 1) % D> slot{};   // of the next step
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            if (ks < 3) {
                fragments((ks + 1) & 1, B, ks + 1);
                if (ks == 0) stage(C0{}, slot, B ^ 1, s + 1 + D);
                else if (ks == 1) stage(C1{}, slot, B ^ 1, s + 1 + D);
                else stage(C2{}, slot, B ^ 1, s + 1 + D);
            } else {
                __syncthreads();   // everybody has read this buffer, and written the other one
                fragments(0, B ^ 1, 0);
            }
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int jj = 0; jj < TN; jj++) acc[i][jj] = multiply<BF16>(xf[ks & 1][i], wf[ks & 1][jj], acc[i][jj]);
#pragma unroll
            for (int n = 0; n < TM * TN; n++) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);     // a product
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // an LDS read
                __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);   // an LDS write
                __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);    // a load
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int s = 0;
    for (; s + U <= steps; s += U) {
        step(C0{}, s);
        step(C1{}, s + 1);
        if constexpr (U == 4) {
            step(C2{}, s + 2);
            step(C3{}, s + 3);
        }
    }
    if (s < steps) step(C0{}, s);
    if constexpr (U == 4) {
        if (s + 1 < steps) step(C1{}, s + 1);
        if (s + 2 < steps) step(C2{}, s + 2);
    }
}

}  // namespace wide
}  // namespace esp
