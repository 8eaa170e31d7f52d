// y[b][n] = sum_k x[b][k] * W[n][k] for up to sixteen rows of fp16 activations and the tiled copy of Q4_K weights (tiles of sixteen rows x 256 columns: gemv.hip), exact products as in
// gemv_q4k_wide_kernel: the integer sc q as the B operand, the minimums' sum from a second chain against the lane's own minimum, both folded into fp32 per super-block.
//
// A wavefront has ONE super-block of columns and takes the BLOCKS row blocks of its workgroup through it, one after the other: its activations are read once, and stay in registers as fragments;
// there is no loop over K, and every wavefront asks for its first weights in its first instructions.  The wavefronts' sums meet in LDS, once, in wavefront order, and as many wavefronts as there are row blocks finish them.
// With more than sixteen super-blocks K is shared by workgroups, whose planes the next kernel adds.  What bounds it is the weights' way from memory and the launch; gemv_q4k_wide_kernel, which these
// products had before, reads a tile of activations, 8 KB, for every 2.3 KB of weights.  Sixteen rows, weights that no cache holds, us:
//   28672 x 4096 with SiLU 28.1 -> 17.7 (3.9 TB/s), 4096 x 14336 15.4 -> 10.8, 6144 x 4096 9.2 -> 7.0, 4096 x 4096 6.4 -> 5.6;  16384 x 2048 9.7 -> 7.7, 2048 x 8192 8.6 -> 5.6;  128256 x 4096 97 -> 68.
#include "batch_gemv.h"
#include "gemv_device.h"
#include <atomic>

namespace esp {
namespace {

using namespace detail;
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr size_t kTileBytes = 2304;
constexpr int kMaxBlocks = 8, kRowBytes = 512 + 16, kWaveBytes = 16 * kRowBytes;   // LDS of a wavefront: its activations, then up to kMaxBlocks kilobytes of sums
static_assert(kWaveBytes >= kMaxBlocks * 1024, "the sums take the activations' place");

struct BatchArgs {
    const uint8_t *tiled;
    const uint16_t *x;
    int N, K, batch, shares, waves, epilogue;
    float *y;
    const float *residual;
    float *partial;
    uint16_t *out_f16;
    QkvEpilogue qkv;
};

struct Tile { uint4 hdr, q0, q1; };

// Where a row's keys and values go, and the RoPE factors of a pair: requested before the sums meet.
struct Place { int pos, seq; float c, s; };
__device__ __forceinline__ void rope_factors(const BatchArgs &a, int r0, Place &e) {
    const QkvEpilogue &q = a.qkv;
    const int half = q.head_dim / 2, ad = q.n_head * q.head_dim, kd = q.n_kv_head * q.head_dim, j = r0 < ad + kd ? (r0 < ad ? r0 : r0 - ad) / 2 % half : 0;
    e.c = q.rope_cos[(size_t)e.pos * half + j];
    e.s = q.rope_sin[(size_t)e.pos * half + j];
}

// rows r0, r0 + 1 of activation row b
__device__ __forceinline__ void finish_pair(const BatchArgs &a, int b, int r0, float v0, float v1, const Place &e) {
    if (r0 + 1 >= a.N) return;
    if (a.epilogue == EPI_SWIGLU_F16) {   // (gate, up): silu_tanh(gate) * up (RealModelInferenceEngine.swift:6825-6827, :6337)
        const float hg = __fmul_rn(0.5f, v0);
        a.out_f16[(size_t)b * (a.N / 2) + r0 / 2] = __builtin_bit_cast(uint16_t, (_Float16)__fmul_rn(__fmul_rn(hg, __fadd_rn(1.0f, tanhf(hg))), v1));
        return;
    }
    // q and k as RoPE pairs (j, j + half), v in natural order (:6745-6772, :6297-6300)
    const QkvEpilogue &q = a.qkv;
    const int half = q.head_dim / 2, ad = q.n_head * q.head_dim, kd = q.n_kv_head * q.head_dim;
    const size_t base = (size_t)e.seq * q.cache_seq_stride + (size_t)e.pos * kd;
    auto keep = [&](void *cache, size_t at, float v) {
        if (q.kv_f16) reinterpret_cast<uint16_t *>(cache)[at] = __builtin_bit_cast(uint16_t, (_Float16)v);
        else reinterpret_cast<float *>(cache)[at] = v;
    };
    if (r0 >= ad + kd) {
        keep(q.v_cache, base + (r0 - ad - kd), v0);
        keep(q.v_cache, base + (r0 - ad - kd) + 1, v1);
        return;
    }
    const bool is_q = r0 < ad;
    const int pr = (is_q ? r0 : r0 - ad) / 2, h = pr / half, j = pr - h * half;
    const float o0 = __fsub_rn(__fmul_rn(v0, e.c), __fmul_rn(v1, e.s)), o1 = __fadd_rn(__fmul_rn(v0, e.s), __fmul_rn(v1, e.c));
    if (is_q) {
        float *dst = q.q_out + (size_t)b * ad + (size_t)h * q.head_dim + j;
        dst[0] = o0;
        dst[half] = o1;
    } else {
        keep(q.k_cache, base + (size_t)h * q.head_dim + j, o0);
        keep(q.k_cache, base + (size_t)h * q.head_dim + j + half, o1);
    }
}

template <int BLOCKS>
__global__ __launch_bounds__(1024) void batch_gemv_kernel(const uint8_t *tiled, const uint16_t *x, int N, int K, int batch, int shares, BatchArgs rest) {
    constexpr int DEPTH = BLOCKS < 4 ? BLOCKS : 4;    // tiles in flight
    BatchArgs a = rest;
    a.N = N;
    extern __shared__ uint4 smem[];
    uint8_t *lds = reinterpret_cast<uint8_t *>(smem);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6, n = lane & 15, g = lane >> 4;
    const int share = blockIdx.x % shares, rb0 = blockIdx.x / shares * BLOCKS, row_blocks = (N + 15) >> 4, nsb = K >> 8, mine = share * waves + wave;
    const int sb = mine < nsb ? mine : nsb - 1;       // (a share's last wavefronts may have none: they add nothing)
    uint8_t *own = lds + wave * kWaveBytes;

    // activations: two rows of 512 bytes an instruction (rows past the batch repeat the last one)
    uint4 xr[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int r = 2 * j + (lane >> 5);
        xr[j] = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint8_t *>(x) + (size_t)(r < batch ? r : batch - 1) * K * 2 + (size_t)sb * 512 + 16 * (lane & 31));
    }
    Tile ring[DEPTH];
    auto load = [&](Tile &t, int i) __attribute__((always_inline)) {
        const int rb = rb0 + i < row_blocks ? rb0 + i : row_blocks - 1;
        const uint8_t *p = tiled + ((size_t)rb * nsb + sb) * kTileBytes;
        t.hdr = *reinterpret_cast<const uint4 *>(p + 16 * n);
        t.q0 = *reinterpret_cast<const uint4 *>(p + 256 + 16 * lane);
        t.q1 = *reinterpret_cast<const uint4 *>(p + 1280 + 16 * lane);
    };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < DEPTH; i++) load(ring[i], i);
    __builtin_amdgcn_sched_barrier(0);
    // a pair's lanes finish activation rows 4 g + 2 k + n % 2
    const bool odd = n & 1;
    Place place[2] = {};
    auto row_of = [&](int k) { return 4 * g + 2 * k + (odd ? 1 : 0); };
    if (a.epilogue == EPI_QKV_ROPE) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int b = row_of(k) < batch ? row_of(k) : batch - 1;
            place[k].pos = a.qkv.pos[b];
            place[k].seq = a.qkv.seq[b];
        }
    }
    // to fragments: lane (i = n, g) has chunk g of row i, fours in the order in which nibbles unpack (0, 2, 1, 3); nobody else uses this stretch, and a wavefront's LDS operations keep their order
#pragma unroll
    for (int j = 0; j < 8; j++) {
        uint4 t;
        t.x = __builtin_amdgcn_perm(xr[j].y, xr[j].x, 0x05040100u);
        t.y = __builtin_amdgcn_perm(xr[j].y, xr[j].x, 0x07060302u);
        t.z = __builtin_amdgcn_perm(xr[j].w, xr[j].z, 0x05040100u);
        t.w = __builtin_amdgcn_perm(xr[j].w, xr[j].z, 0x07060302u);
        *reinterpret_cast<uint4 *>(own + (2 * j + (lane >> 5)) * kRowBytes + 16 * (lane & 31)) = t;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    half8 xf[8];
#pragma unroll
    for (int j = 0; j < 8; j++) xf[j] = *reinterpret_cast<const half8 *>(own + n * kRowBytes + 128 * g + 16 * j);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();

    const Q4KLane L = q4k_chunk_constants(g);
    u32 mask_lo = 0x000F000Fu, mask_hi = 0x00F000F0u, magic_lo = 0x64006400u, magic_hi = 0x54005400u;
    asm volatile("" : "+s"(mask_lo), "+s"(mask_hi));
    asm volatile("" : "+v"(magic_lo), "+v"(magic_hi));
#pragma unroll
    for (int i = 0; i < BLOCKS; i++) {
        const Tile &it = ring[i % DEPTH];
        const u32 qd[8] = {it.q0.x, it.q0.y, it.q0.z, it.q0.w, it.q1.x, it.q1.y, it.q1.z, it.q1.w};
        const u32 src_sc = L.upper ? it.hdr.w : it.hdr.y, src_min = L.upper ? it.hdr.w : it.hdr.z;
        const u32 scp = ((src_sc >> L.sh_sc) & L.mask_low) | ((it.hdr.y >> L.sh_top) & L.mask_top);
        const u32 mp = ((src_min >> L.sh_min) & L.mask_low) | ((it.hdr.z >> L.sh_top) & L.mask_top);
        const _Float16 s0 = (_Float16)(unsigned short)(scp & 0xFFu), s1 = (_Float16)(unsigned short)((scp >> 8) & 0xFFu);
        const _Float16 m0 = (_Float16)(unsigned short)(mp & 0xFFu), m1 = (_Float16)(unsigned short)((mp >> 8) & 0xFFu);
        const h2 s_lo = {s0, s0}, s_hi = {s1, s1}, o_lo = s_lo * (h2){(_Float16)-1024.0f, (_Float16)-1024.0f}, o_hi = s_hi * (h2){(_Float16)-64.0f, (_Float16)-64.0f};
        const half8 bm_lo = {m0, m0, m0, m0, m0, m0, m0, m0}, bm_hi = {m1, m1, m1, m1, m1, m1, m1, m1};
        floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, accm = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
            uint4 pl, ph;
            auto four = [&](u32 w, u32 mask, u32 magic, const h2 &s, const h2 &o) { return __builtin_bit_cast(u32, __builtin_elementwise_fma(as_h2((w & mask) | magic), s, o)); };
            pl.x = four(qd[2 * jj], mask_lo, magic_lo, s_lo, o_lo); pl.y = four(qd[2 * jj] >> 8, mask_lo, magic_lo, s_lo, o_lo);
            pl.z = four(qd[2 * jj + 1], mask_lo, magic_lo, s_lo, o_lo); pl.w = four(qd[2 * jj + 1] >> 8, mask_lo, magic_lo, s_lo, o_lo);
            ph.x = four(qd[2 * jj], mask_hi, magic_hi, s_hi, o_hi); ph.y = four(qd[2 * jj] >> 8, mask_hi, magic_hi, s_hi, o_hi);
            ph.z = four(qd[2 * jj + 1], mask_hi, magic_hi, s_hi, o_hi); ph.w = four(qd[2 * jj + 1] >> 8, mask_hi, magic_hi, s_hi, o_hi);
            // low nibbles of the chunk: columns 8 jj .. 8 jj + 7 of its first half, high nibbles: of its second half
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[jj], __builtin_bit_cast(half8, pl), acc, 0, 0, 0);
            accm = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[jj], bm_lo, accm, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[4 + jj], __builtin_bit_cast(half8, ph), acc, 0, 0, 0);
            accm = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[4 + jj], bm_hi, accm, 0, 0, 0);
        }
        const float d = half_bits_to_float(it.hdr.x & 0xFFFFu), dmin = half_bits_to_float(it.hdr.x >> 16);
        float4 v;
        float *out = &v.x;
#pragma unroll
        for (int r = 0; r < 4; r++) out[r] = mine < nsb ? d * acc[r] - dmin * accm[r] : 0.0f;
        *reinterpret_cast<float4 *>(own + i * 1024 + 16 * lane) = v;
        if (i + DEPTH < BLOCKS) load(ring[i % DEPTH], i + DEPTH);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (a.epilogue == EPI_QKV_ROPE) {
#pragma unroll
        for (int k = 0; k < 2; k++) rope_factors(a, (rb0 + wave) * 16 + (n & ~1) < N ? (rb0 + wave) * 16 + (n & ~1) : 0, place[k]);
    }
    __syncthreads();
    // lane (n, g) holds weight row n of its block for activation rows 4 g .. 4 g + 3
    for (int i = wave; i < BLOCKS; i += waves) {
        const int rb = rb0 + i, row = rb * 16 + n;
        float4 t = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        for (int w = 0; w < waves; w++) {
            const float4 p = *reinterpret_cast<const float4 *>(lds + w * kWaveBytes + i * 1024 + 16 * lane);
            t.x += p.x; t.y += p.y; t.z += p.z; t.w += p.w;
        }
        if (rb >= row_blocks) return;
        const float out[4] = {t.x, t.y, t.z, t.w};
        if (a.epilogue == EPI_SWIGLU_F16 || a.epilogue == EPI_QKV_ROPE) {
            // rows n and n + 1 (n even) are a pair
            float other[4];
#pragma unroll
            for (int r = 0; r < 4; r++) other[r] = dpp_term<0xB1, 0xF>(out[r]);   // the neighbouring lane's row
#pragma unroll
            for (int k = 0; k < 2; k++) {
                if (i != wave && a.epilogue == EPI_QKV_ROPE) rope_factors(a, (row & ~1) < N ? row & ~1 : 0, place[k]);
                if (row_of(k) < batch) finish_pair(a, row_of(k), row & ~1, odd ? other[2 * k + 1] : out[2 * k], odd ? out[2 * k + 1] : other[2 * k], place[k]);
            }
            continue;
        }
        if (row < N) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int b = 4 * g + r;
                if (b >= batch) continue;
                const size_t o = (size_t)b * N + row;
                if (shares > 1) a.partial[(size_t)share * batch * N + o] = out[r];
                else a.y[o] = a.epilogue == EPI_ADD_RESIDUAL ? a.residual[o] + out[r] : out[r];
            }
        }
    }
}

template <int BLOCKS>
hipError_t launch(const BatchArgs &a, hipStream_t stream) {
    const size_t lds = (size_t)a.waves * kWaveBytes;
    static std::atomic<uint64_t> raised{0};
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    if (const uint64_t bit = 1ull << (device & 63); !(raised.load(std::memory_order_acquire) & bit)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(batch_gemv_kernel<BLOCKS>), hipFuncAttributeMaxDynamicSharedMemorySize, 16 * kWaveBytes);
        if (e != hipSuccess) return e;
        raised.fetch_or(bit, std::memory_order_release);
    }
    const int row_blocks = (a.N + 15) / 16;
    hipLaunchKernelGGL(batch_gemv_kernel<BLOCKS>, dim3((row_blocks + BLOCKS - 1) / BLOCKS * a.shares), dim3(64 * a.waves), lds, stream, a.tiled, a.x, a.N, a.K, a.batch, a.shares, a);
    return hipGetLastError();
}
std::atomic<int> g_batch_gemv_form{0};

}  // namespace

void batch_gemv_set_form(int form) { g_batch_gemv_form.store(form > 0 && form / 10 <= kMaxBlocks && form / 10 >= 1 && form % 10 >= 1 ? form : 0); }

// By the busiest compute unit's bytes, or all of them at what the card reads; a share of K is a plane that the next kernel reads.  Forms that are asked for and cannot be fall back to the rule.
BatchGemvForm batch_gemv_form(const GemvParams &p) {
    BatchGemvForm best, asked;
    const DeviceMatrix &w = p.w;
    const int forced = g_batch_gemv_form.load(), cus = device_compute_units() > 0 ? device_compute_units() : 256;
    const bool planes = p.workspace && p.deferred_splits && (p.epilogue == EPI_STORE_F32 || p.epilogue == EPI_ADD_RESIDUAL);
    if (w.format != FMT_Q4_K || !w.tiled || w.cols % 256 != 0 || w.rows <= 0 || p.batch < 1 || p.batch > 16 || !p.x || p.epilogue == EPI_ARGMAX) return best;
    const int nsb = w.cols / 256, row_blocks = (w.rows + 15) / 16;
    for (int want = 1; want <= 8; want++) {
        const int waves = (nsb + want - 1) / want, shares = (nsb + waves - 1) / waves;
        if (waves > 16 || shares != want || (shares > 1 && (!planes || (size_t)shares * p.batch * w.rows > p.workspace_floats))) continue;
        for (int blocks = 1; blocks <= kMaxBlocks; blocks++) {
            const long wgs = (long)((row_blocks + blocks - 1) / blocks) * shares, at_once = (long)cus * (16 / waves), rounds = (wgs + at_once - 1) / at_once;
            const float on_one = (float)((wgs + cus - 1) / cus);   // workgroups of the busiest compute unit
            const float on_unit = on_one * (float)waves * ((float)blocks * 2304.0f + 4096.0f) / 24000.0f, all = (float)row_blocks * (float)nsb * 2304.0f / 5.4e6f;
            float us = 1.0f + (float)rounds + (on_unit > all ? on_unit : all);
            if (shares > 1) us += 0.5f + 0.25f * (float)shares;
            if (!best.blocks || us < best.us) best = BatchGemvForm{blocks, shares, waves, us};
            if (forced == 10 * blocks + shares) asked = best, asked.blocks = blocks, asked.shares = shares, asked.waves = waves;
        }
    }
    return asked.blocks ? asked : best;
}

hipError_t launch_batch_gemv(const GemvParams &p, const BatchGemvForm &f, hipStream_t stream) {
    const BatchArgs a{p.w.tiled, p.x, p.w.rows, p.w.cols, p.batch, f.shares, f.waves, p.epilogue, p.y, p.residual, p.workspace, p.out_f16, p.qkv};
    if (f.shares > 1) *p.deferred_splits = f.shares;
    switch (f.blocks) {
    case 1: return launch<1>(a, stream);
    case 2: return launch<2>(a, stream);
    case 3: return launch<3>(a, stream);
    case 4: return launch<4>(a, stream);
    case 5: return launch<5>(a, stream);
    case 6: return launch<6>(a, stream);
    case 7: return launch<7>(a, stream);
    case 8: return launch<8>(a, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace esp
