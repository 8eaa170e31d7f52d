// What the kernels of block_gemm.hip and block_split.hip share.  A workgroup is eight wavefronts: NW of them side by side along 32 NW weight rows, 8 / NW groups that share K, each
// wavefront with 32 weight rows and all 32 TM activation rows of the workgroup's tile.
#pragma once

#include "../common.h"
#include <atomic>

namespace esp {
namespace block_tile {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32;

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kStep = 128;        // k per step: four blocks of Q8_0 / Q4_0, half a super-block of Q4_K
constexpr int kRow = kStep + 8;   // fp16 between the staged activation rows: 272 bytes, sixteen-byte reads of neighbouring rows fall on different banks

__device__ __forceinline__ h2 as_h2(u32 v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ u32 as_u32(h2 v) { return __builtin_bit_cast(u32, v); }
__device__ __forceinline__ half8 as_half8(const uint4 &v) { return __builtin_bit_cast(half8, v); }
__device__ __forceinline__ float half_bits_to_float(u32 bits16) { return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16); }

// The workgroup's place among tiles of activation rows, tiles of weight rows and shares of K: workgroups of one die take neighbouring output tiles, the row tiles of one block of
// weights first.
struct Place { int m_tile, n_tile, split; };
__device__ __forceinline__ Place place_of(int m_tiles, int n_tiles, int block, int total) {
    const int die = block & 7, q8 = total >> 3, r8 = total & 7;
    const int unit = die * q8 + (die < r8 ? die : r8) + (block >> 3);
    const int m_tile = unit % m_tiles, rest = unit / m_tiles, n_tile = rest % n_tiles, split = rest / n_tiles;
    return {m_tile, n_tile, split};
}
__device__ __forceinline__ Place place_of(int m_tiles, int n_tiles) { return place_of(m_tiles, n_tiles, blockIdx.x, gridDim.x); }

// Lane 16 p + r loaded piece p of row r (raw[0]) and of row 16 + r (raw[1]), so that four lanes cover 64 bytes of a row; afterwards each lane holds two pieces of row lane % 32.
__device__ __forceinline__ void exchange_rows(const uint4 (&raw)[2], uint4 (&q)[2]) {
    auto swap = [](u32 x, u32 y, u32 &u, u32 &v) __attribute__((always_inline)) { const auto p = __builtin_amdgcn_permlane16_swap(x, y, false, false); u = p[0]; v = p[1]; };
    swap(raw[0].x, raw[1].x, q[0].x, q[1].x);
    swap(raw[0].y, raw[1].y, q[0].y, q[1].y);
    swap(raw[0].z, raw[1].z, q[0].z, q[1].z);
    swap(raw[0].w, raw[1].w, q[0].w, q[1].w);
}

// The accumulators r0 .. r0 + TM * 16 / KW - 1 (r0: the group times their number) that a wavefront finishes.  With several groups their sums meet in LDS, in the groups' order: the caller's last barrier is behind
// everybody's last read of it.
template <int TM, int NW>
__device__ __forceinline__ void share_sums(const floatx16 (&acc)[TM], float *red, int wave, int wn, int lane, int r0, float (&v)[TM * 16 / (kWaves / NW)]) {
    constexpr int KW = kWaves / NW, SHARE = TM * 16 / KW;
    if constexpr (KW == 1) {
#pragma unroll
        for (int r = 0; r < SHARE; r++) v[r] = acc[r >> 4][r & 15];
    } else {
#pragma unroll
        for (int r = 0; r < TM * 16; r++) red[((size_t)wave * TM * 16 + r) * 64 + lane] = acc[r >> 4][r & 15];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < SHARE; r++) {
            float sum = red[((size_t)wn * TM * 16 + r0 + r) * 64 + lane];
#pragma unroll
            for (int g = 1; g < KW; g++) sum += red[((size_t)(g * NW + wn) * TM * 16 + r0 + r) * 64 + lane];
            v[r] = sum;
        }
    }
}

// Accumulator r of a lane is activation row 8 (r / 4) + 4 h + r % 4 of its 32, weight row lane % 32.
__device__ __forceinline__ int tile_row(int r, int h) { return 32 * (r >> 4) + 8 * ((r & 15) >> 2) + 4 * h + (r & 3); }

// Weight rows as (gate, up) pairs are neighbouring lanes: the even lane takes accumulator `even` of both, the odd lane accumulator `uneven`.
__device__ __forceinline__ void gate_and_up(float even, float uneven, bool odd, float &gate, float &up) {
    const float p0 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, even), 0xB1, 0xF, 0xF, false));   // quad_perm [1,0,3,2]
    const float p1 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, uneven), 0xB1, 0xF, 0xF, false));
    gate = odd ? p1 : even;
    up = odd ? uneven : p0;
}

// The limit of dynamic LDS, raised once per kernel and device (`raised`: the kernel's own).
inline hipError_t raise_lds_limit(const void *kernel, size_t lds, std::atomic<uint64_t> &raised) {
    if (lds <= 64 * 1024) return hipSuccess;
    int device = 0;
    hipError_t err = hipGetDevice(&device);
    if (err != hipSuccess) return err;
    const uint64_t bit = 1ull << (device & 63);
    if (raised.load(std::memory_order_acquire) & bit) return hipSuccess;
    err = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err == hipSuccess) raised.fetch_or(bit, std::memory_order_release);
    return err;
}

// Steps of a group, and the shares of K that leaves, where `want` shares of `units` indivisible pieces of K are asked for.
struct Shares { int per, splits; };
inline Shares shares_of(int units, int nw, int want) {
    const int kw = kWaves / nw, per = (units + want * kw - 1) / (want * kw);
    return {per, (units + per * kw - 1) / (per * kw)};
}

}  // namespace block_tile
}  // namespace esp
