// Attention with grouped heads over a ring of cached keys and values, a sliding window, root-mean-square norms over the whole query and
// key projections, and rotation of the first dimensions of a head (gfx950).
//
//   mixed row   [q: heads | k: kv_heads | v: kv_heads], heads padded; a layer that reads another one's cache has q alone
//   cached row  [k: kv_heads x dim_p | v: kv_heads x vdim_p], one per token, at position % ring, keys normed and rotated
//
// A decode step of one row or a few with a short window is one launch (attention_window_kernel).  Otherwise it is two.  partial: a workgroup takes a slice of the window for the query heads of one key head; it norms and
// rotates their queries itself (the norm's sum runs over the whole projection, which every workgroup reads), and the workgroup whose
// slice holds the row's own token puts its key and value into the cache first.  Eight lanes share a key, so a key is read once for all
// query heads of the group.  merge: the slices' (maximum, sum, weighted values) joined.
//
// A prompt block is three: prepare (queries, and keys and values into the ring), gather (the visible span, values transposed), and
// attention in tiles of 64 keys (block_attention.hip).
#include <hip/hip_runtime.h>

#include "gemv_device.h"
#include "layer_ops.h"
#include "matrix_ops.h"

namespace esp {
namespace {

using matrix::Op;

__host__ __device__ __forceinline__ int cached_row(const AttentionShape &l) { return l.kv_heads * (l.dim_p + l.vdim_p); }
__device__ __forceinline__ int first_seen(int pos, int window) { return pos - window + 1 > 0 ? pos - window + 1 : 0; }

// Element d of a head x, normed (scale inv, weights w) and rotated: pairs (i, i + dims / 2) of the first dims elements.
__device__ __forceinline__ float normed_rotated(const float *x, const float *w, float inv, int d, int dims, const float *cos, const float *sin) {
    if (d >= dims) return x[d] * inv * w[d];
    const int half = dims / 2, i = d < half ? d : d - half;
    const float c = cos[i], s = sin[i], u = x[i] * inv * w[i], v = x[i + half] * inv * w[i + half];
    return d < half ? u * c - v * s : v * c + u * s;
}

__device__ __forceinline__ float squares(const float *x, int count) {   // this thread's share; count is a multiple of four
    float s = 0.0f;
    for (int i = threadIdx.x * 4; i < count; i += 256 * 4) {
        const float4 v = *reinterpret_cast<const float4 *>(x + i);
        s += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
    }
    return s;
}

// Eight consecutive cached elements.
__device__ __forceinline__ void load8(const uint16_t *p, float (&f)[8]) { matrix::unpack_bf16(*reinterpret_cast<const uint4 *>(p), f); }
__device__ __forceinline__ void load8(const float *p, float (&f)[8]) {
    const float4 a = reinterpret_cast<const float4 *>(p)[0], b = reinterpret_cast<const float4 *>(p)[1];
    f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
}

// The same eight as they are loaded, to be unpacked later.
template <typename T>
struct Piece;
template <>
struct Piece<uint16_t> {
    uint4 v;
    __device__ __forceinline__ void load(const uint16_t *p) { v = *reinterpret_cast<const uint4 *>(p); }
    __device__ __forceinline__ void unpack(float (&f)[8]) const { matrix::unpack_bf16(v, f); }
};
template <>
struct Piece<float> {
    float4 a, b;
    __device__ __forceinline__ void load(const float *p) { a = reinterpret_cast<const float4 *>(p)[0]; b = reinterpret_cast<const float4 *>(p)[1]; }
    __device__ __forceinline__ void unpack(float (&f)[8]) const { f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w; }
};

constexpr int meeting_heads(int q) { return q < 4 ? q : 4; }   // query heads whose sums meet in LDS together
constexpr int kTile = 32;   // keys per pass of a workgroup: eight lanes each

constexpr int kKeyPieces = 4, kValuePieces = 2;   // pieces of eight per thread that are requested ahead; longer heads read the rest when needed

// grid (splits, key heads x chunks of Q query heads, rows).  LDS: queries [Q][dim_p], scores [Q][kTile], running (maximum, sum, rescale)
// [Q][4], the row's own key [dim_p] and value [vdim_p], and for the end the value sums [parts][vdim_p].  A tile's keys and values are
// requested a tile ahead, the first ones before the norms.
template <typename T, int Q>
__global__ __launch_bounds__(256) void attention_partial_kernel(AttentionShape l, AttentionStep p) {
    extern __shared__ float lds[];
    __shared__ float red[8];
    float *q = lds, *scores = q + Q * l.dim_p, *running = scores + Q * kTile, *own_key = running + Q * 4, *own_value = own_key + l.dim_p, *meet = own_value + l.vdim_p;
    const int tid = threadIdx.x, lane = tid & 63, split = blockIdx.x, m = blockIdx.z, pos = p.pos[m], seq = p.seq[m];
    const int share = l.heads / l.kv_heads, chunks = (share + Q - 1) / Q, kv = blockIdx.y / chunks, h0 = kv * share + blockIdx.y % chunks * Q;
    const int live = (kv + 1) * share - h0 < Q ? (kv + 1) * share - h0 : Q;
    const int lo = first_seen(pos, l.window), tiles = (pos - lo) / kTile + 1;
    if (split >= tiles) return;
    const float *row = p.mixed + (size_t)m * l.ld_mix;
    const float *cos = l.cos + (size_t)pos * (l.rot_dims / 2), *sin = l.sin + (size_t)pos * (l.rot_dims / 2);
    const int width = cached_row(l);
    T *cache = static_cast<T *>(l.cache) + (size_t)seq * l.ring * width;
    const bool owner = l.k_at >= 0 && split == (tiles - 1) % p.splits;   // the last tile holds the row's own token
    const int e = tid & 7, key_in = tid >> 3;
    const int pieces = l.vdim_p / 8, parts = 256 / pieces < kTile ? 256 / pieces : kTile, piece = tid % pieces, part = tid / pieces;   // value phase: eight values, every parts-th key
    const T *keys = cache + kv * l.dim_p, *values = cache + l.kv_heads * l.dim_p + kv * l.vdim_p + piece * 8;
    auto row_of = [&](int key) { return (size_t)((key < pos ? key : pos) % l.ring) * width; };   // keys past the query repeat it and weigh nothing
    Piece<T> key_ahead[kKeyPieces], value_ahead[kValuePieces];
    auto request = [&](int t) {
        const int k0 = lo + t * kTile;
        const T *from = keys + row_of(k0 + key_in);
#pragma unroll
        for (int i = 0; i < kKeyPieces; i++) key_ahead[i].load(from + (e * 8 + i * 64 < l.dim_p ? e * 8 + i * 64 : 0));
#pragma unroll
        for (int i = 0; i < kValuePieces; i++) value_ahead[i].load(values + row_of(k0 + (part + i * parts < kTile ? part + i * parts : 0)));
    };
    {
        float sq = squares(row, l.heads * l.dim_p), sk = owner ? squares(row + l.k_at, l.kv_heads * l.dim_p) : 0.0f;
        request(split);
        sq = detail::wave_sum(sq);
        sk = detail::wave_sum(sk);
        if (lane == 0) { red[tid >> 6] = sq; red[4 + (tid >> 6)] = sk; }
        __syncthreads();
        sq = (red[0] + red[1]) + (red[2] + red[3]);
        sk = (red[4] + red[5]) + (red[6] + red[7]);
        const float inv_q = 1.0f / sqrtf(sq / ((float)l.heads * (float)l.dim) + l.eps), inv_k = 1.0f / sqrtf(sk / ((float)l.kv_heads * (float)l.dim) + l.eps);
        for (int i = tid; i < Q * l.dim_p; i += 256) {
            const int r = i / l.dim_p, d = i - r * l.dim_p, at = (h0 + (r < live ? r : 0)) * l.dim_p;   // heads past the group repeat its first
            q[i] = l.scale * normed_rotated(row + at, l.q_norm + at, inv_q, d, l.rot_dims, cos, sin);
        }
        if (owner) {   // every chunk of the group's heads writes the same; here they are read from LDS
            T *own = cache + (size_t)(pos % l.ring) * width;
            for (int d = tid; d < l.dim_p; d += 256) {
                const int at = kv * l.dim_p;
                const T k = Op<T>::from_float(normed_rotated(row + l.k_at + at, l.k_norm + at, inv_k, d, l.rot_dims, cos, sin));
                own[at + d] = k;
                own_key[d] = Op<T>::to_float(k);
            }
            const float *v = row + l.k_at + l.kv_heads * l.dim_p + kv * l.vdim_p;
            for (int d = tid; d < l.vdim_p; d += 256) {
                const T x = Op<T>::from_float(v[d]);
                own[l.kv_heads * l.dim_p + kv * l.vdim_p + d] = x;
                own_value[d] = Op<T>::to_float(x);
            }
        }
        if (tid < Q) { running[tid * 4] = -INFINITY; running[tid * 4 + 1] = 0.0f; }
    }
    __syncthreads();
    float acc[Q][8];
#pragma unroll
    for (int r = 0; r < Q; r++)
#pragma unroll
        for (int i = 0; i < 8; i++) acc[r][i] = 0.0f;
    for (int t = split; t < tiles; t += p.splits) {
        const int k0 = lo + t * kTile;
        const bool in = k0 + key_in <= pos, mine = owner && k0 + key_in >= pos;
        float s[Q];
#pragma unroll
        for (int r = 0; r < Q; r++) s[r] = 0.0f;
        auto score = [&](float (&k)[8], int d) {
            if (mine) load8(own_key + d, k);
#pragma unroll
            for (int r = 0; r < Q; r++) {
                float x[8];
                load8(q + r * l.dim_p + d, x);
#pragma unroll
                for (int i = 0; i < 8; i++) s[r] = __builtin_fmaf(k[i], x[i], s[r]);
            }
        };
#pragma unroll
        for (int i = 0; i < kKeyPieces; i++) {
            float k[8];
            key_ahead[i].unpack(k);
            if (e * 8 + i * 64 < l.dim_p) score(k, e * 8 + i * 64);
        }
        for (int d = e * 8 + kKeyPieces * 64; d < l.dim_p; d += 64) {
            float k[8];
            load8(keys + row_of(k0 + key_in) + d, k);
            score(k, d);
        }
#pragma unroll
        for (int r = 0; r < Q; r++) {   // the eight lanes of a key
            s[r] += detail::dpp_term<0xB1, 0xF>(s[r]);
            s[r] += detail::dpp_term<0x4E, 0xF>(s[r]);
            s[r] += detail::dpp_term<0x141, 0xF>(s[r]);
            if (e == 0) scores[r * kTile + key_in] = in ? s[r] : -INFINITY;
        }
        __syncthreads();
        for (int r = tid / kTile; r < Q; r += 256 / kTile) {   // 32 lanes per head
            const float x = scores[r * kTile + (tid & 31)], was = running[r * 4];
            float top = fmaxf(x, was);
#pragma unroll
            for (int d = 16; d >= 1; d >>= 1) top = fmaxf(top, __shfl_xor(top, d));
            const float w = matrix::weight_exp<T>(x - top), keep = matrix::weight_exp<T>(was - top);
            float sum = w;
#pragma unroll
            for (int d = 16; d >= 1; d >>= 1) sum += __shfl_xor(sum, d);
            scores[r * kTile + (tid & 31)] = w;
            if ((tid & 31) == 0) { running[r * 4] = top; running[r * 4 + 1] = running[r * 4 + 1] * keep + sum; running[r * 4 + 2] = keep; }
        }
        __syncthreads();
        if (part < parts) {
#pragma unroll
            for (int r = 0; r < Q; r++) {
                const float keep = running[r * 4 + 2];
#pragma unroll
                for (int i = 0; i < 8; i++) acc[r][i] *= keep;
            }
            auto add = [&](float (&v)[8], int k) {
                if (owner && k0 + k >= pos) load8(own_value + piece * 8, v);
#pragma unroll
                for (int r = 0; r < Q; r++) {
                    const float w = scores[r * kTile + k];
#pragma unroll
                    for (int i = 0; i < 8; i++) acc[r][i] = __builtin_fmaf(w, v[i], acc[r][i]);
                }
            };
#pragma unroll
            for (int i = 0; i < kValuePieces; i++) {
                float v[8];
                value_ahead[i].unpack(v);
                if (part + i * parts < kTile) add(v, part + i * parts);
            }
            for (int k = part + kValuePieces * parts; k < kTile; k += parts) {
                float v[8];
                load8(values + row_of(k0 + k), v);
                add(v, k);
            }
        }
        if (t + p.splits < tiles) request(t + p.splits);
        __syncthreads();
    }
    const size_t first = ((size_t)m * p.splits + split) * l.heads + h0;
    // the parts' sums of up to four heads meet in LDS at once (head by head, two barriers each, the launch took 8.9 us instead of 8.0 with a window of 256)
#pragma unroll
    for (int r0 = 0; r0 < Q; r0 += meeting_heads(Q)) {
        if (r0 >= live) break;
        if (part < parts) {
#pragma unroll
            for (int i = 0; i < meeting_heads(Q); i++) {
                float4 *to = reinterpret_cast<float4 *>(meet + (i * parts + part) * l.vdim_p + piece * 8);
                to[0] = make_float4(acc[r0 + i][0], acc[r0 + i][1], acc[r0 + i][2], acc[r0 + i][3]);
                to[1] = make_float4(acc[r0 + i][4], acc[r0 + i][5], acc[r0 + i][6], acc[r0 + i][7]);
            }
        }
        __syncthreads();
        const int heads = live - r0 < meeting_heads(Q) ? live - r0 : meeting_heads(Q);
        for (int v = tid; v < heads * l.vdim_p; v += 256) {
            const int r = v / l.vdim_p, d = v - r * l.vdim_p;
            float s = 0.0f;
            for (int i = 0; i < parts; i++) s += meet[(r * parts + i) * l.vdim_p + d];
            p.partial[(first + r0 + r) * l.vdim_p + d] = s;
        }
        if (tid < heads) *reinterpret_cast<float2 *>(p.partial_ml + (first + r0 + tid) * 2) = make_float2(running[(r0 + tid) * 4], running[(r0 + tid) * 4 + 1]);
        if (r0 + meeting_heads(Q) < Q) __syncthreads();
    }
}

// grid (heads, rows).  splits <= 64: a lane of the first wavefront each.
template <typename T>
__global__ __launch_bounds__(256) void attention_merge_kernel(AttentionShape l, AttentionStep p) {
    __shared__ float weight[64];
    const int tid = threadIdx.x, h = blockIdx.x, m = blockIdx.y, pos = p.pos[m];
    const int tiles = (pos - first_seen(pos, l.window)) / kTile + 1, live = tiles < p.splits ? tiles : p.splits;
    const size_t first = (size_t)m * p.splits * l.heads + h;   // slice s: first + s * heads
    if (tid < 64) {
        const float2 ml = *reinterpret_cast<const float2 *>(p.partial_ml + (first + (size_t)(tid < live ? tid : 0) * l.heads) * 2);
        float top = ml.x;
#pragma unroll
        for (int x = 32; x >= 1; x >>= 1) top = fmaxf(top, __shfl_xor(top, x));
        const float w = tid < live ? expf(ml.x - top) : 0.0f;
        weight[tid] = w / detail::wave_sum(w * ml.y);
    }
    __syncthreads();
    for (int v = tid; v < l.vdim_p; v += 256) {
        float o = 0.0f;
        for (int s0 = 0; s0 < live; s0 += 8) {   // eight slices in flight
            float x[8];
#pragma unroll
            for (int u = 0; u < 8; u++) x[u] = p.partial[(first + (size_t)(s0 + u < live ? s0 + u : 0) * l.heads) * l.vdim_p + v];
#pragma unroll
            for (int u = 0; u < 8; u++) o += s0 + u < live ? weight[s0 + u] * x[u] : 0.0f;
        }
        if (p.mix) p.mix[(size_t)m * l.heads * l.vdim_p + h * l.vdim_p + v] = o;
        else static_cast<T *>(p.act)[(size_t)m * p.ld_act + h * l.vdim_p + v] = Op<T>::from_float(o);
    }
}

// One element of a head before its norm is known: what normed_rotated reads.
struct Element {
    float u, v, wu, wv, c, s;
    __device__ __forceinline__ void load(const float *x, const float *w, int d, int dims, const float *cos, const float *sin) {
        const int half = dims / 2, i = d < dims && d >= half ? d - half : d, j = d < dims ? i + half : d;
        u = x[i]; v = x[j]; wu = w[i]; wv = w[j];
        c = d < dims ? cos[i] : 1.0f;
        s = d < dims ? sin[i] : 0.0f;
    }
    __device__ __forceinline__ float value(float inv, int d, int dims) const {
        if (d >= dims) return u * inv * wu;
        const float x = u * inv * wu, y = v * inv * wv;
        return d < dims / 2 ? x * c - y * s : y * c + x * s;
    }
};

constexpr int kWindowHead = 128, kWindowSlice = 32, kWindowKeys = 128;   // longest key; values of a workgroup, keys of a pass
// A short window in one launch: grid (heads x slices of 32 values, rows).  Bound by its chain of memory trips, position -> keys and values -> store, so sixteen wavefronts ask for all of the window's keys (eight lanes a
// key) and their slice of its values (four lanes a key) at once, together with what the norms and the rotation read; a workgroup needs every score of its head, which is why keys are read once per slice, from the cache
// after the first.  No state passes between workgroups, and no sum is rescaled: maximum, weights and sum are taken over the whole window.  Window of 256, heads of 128: 7 us instead of 8.7 + 4.7 for slices and their merge.
template <typename T, int PASSES>
__global__ __launch_bounds__(1024) void attention_window_kernel(AttentionShape l, AttentionStep p) {
    constexpr int VP = PASSES / 2;   // passes over the values: 256 keys each
    static_assert(PASSES % 2 == 0, "whole passes over the values");
    __shared__ float q[kWindowHead], own_key[kWindowHead], own_value[kWindowSlice], scores[256 * VP], red[2][16], meet[64][kWindowSlice];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, slices = l.vdim_p / kWindowSlice, h = blockIdx.x / slices, slice = blockIdx.x % slices, m = blockIdx.y;
    const int share = l.heads / l.kv_heads, kv = h / share, width = cached_row(l), count_q = l.heads * l.dim_p, count_k = l.k_at >= 0 ? l.kv_heads * l.dim_p : 0;
    const float *row = p.mixed + (size_t)m * l.ld_mix, *row_k = row + (l.k_at >= 0 ? l.k_at : 0);
    // whatever the position: the norms' first values
    const float4 first_q = *reinterpret_cast<const float4 *>(row + (tid * 4 < count_q ? tid * 4 : 0)), first_k = *reinterpret_cast<const float4 *>(row_k + (tid * 4 < count_k ? tid * 4 : 0));
    const int pos = p.pos[m], seq = p.seq[m];
    const int lo = first_seen(pos, l.window), keys = pos - lo + 1;
    const float *cos = l.cos + (size_t)pos * (l.rot_dims / 2), *sin = l.sin + (size_t)pos * (l.rot_dims / 2);
    T *cache = static_cast<T *>(l.cache) + (size_t)seq * l.ring * width;
    auto row_of = [&](int i) { return (size_t)((i < keys ? lo + i : pos) % l.ring) * width; };   // keys past the query repeat it and weigh nothing
    const int e = tid & 7, key_in = tid >> 3, piece = tid & 3, value_in = tid >> 2;
    Piece<T> key_piece[PASSES][2], value_piece[VP];
#pragma unroll
    for (int k = 0; k < PASSES; k++) {
        const T *from = cache + kv * l.dim_p + row_of(k * kWindowKeys + key_in);
#pragma unroll
        for (int i = 0; i < 2; i++) key_piece[k][i].load(from + (e * 8 + i * 64 < l.dim_p ? e * 8 + i * 64 : 0));
    }
#pragma unroll
    for (int k = 0; k < VP; k++) value_piece[k].load(cache + l.kv_heads * l.dim_p + kv * l.vdim_p + slice * kWindowSlice + piece * 8 + row_of(k * 256 + value_in));
    const int d = tid & 127;
    const bool makes_q = tid < l.dim_p, makes_k = tid >= 128 && tid < 128 + l.dim_p && count_k > 0, makes_v = tid >= 256 && tid < 256 + kWindowSlice && count_k > 0;
    const bool keeps = count_k > 0 && h % share == 0 && slice == 0;   // one workgroup of a key head puts the row's own key and value into the cache
    const float *row_v = row_k + count_k + kv * l.vdim_p;
    Element x = {};
    float v = 0.0f;
    if (makes_q) x.load(row + h * l.dim_p, l.q_norm + h * l.dim_p, d, l.rot_dims, cos, sin);
    if (makes_k) x.load(row_k + kv * l.dim_p, l.k_norm + kv * l.dim_p, d, l.rot_dims, cos, sin);
    if (makes_v) v = row_v[slice * kWindowSlice + tid - 256];
    __builtin_amdgcn_sched_barrier(0);   // all of it is requested before anything is waited for
    auto dot4 = [](const float4 &f) { return f.x * f.x + f.y * f.y + f.z * f.z + f.w * f.w; };
    float sq = tid * 4 < count_q ? dot4(first_q) : 0.0f, sk = tid * 4 < count_k ? dot4(first_k) : 0.0f;
    for (int i = 4096 + tid * 4; i < count_q; i += 4096) sq += dot4(*reinterpret_cast<const float4 *>(row + i));
    for (int i = 4096 + tid * 4; i < count_k; i += 4096) sk += dot4(*reinterpret_cast<const float4 *>(row_k + i));
    sq = detail::wave_sum(sq);
    sk = detail::wave_sum(sk);
    if (lane == 0) { red[0][wave] = sq; red[1][wave] = sk; }
    __syncthreads();
    sq = 0.0f;
    sk = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i++) { sq += red[0][i]; sk += red[1][i]; }
    if (makes_q) q[d] = l.scale * x.value(1.0f / sqrtf(sq / ((float)l.heads * (float)l.dim) + l.eps), d, l.rot_dims);
    T *own = cache + (size_t)(pos % l.ring) * width;
    if (makes_k) {
        const T k = Op<T>::from_float(x.value(1.0f / sqrtf(sk / ((float)l.kv_heads * (float)l.dim) + l.eps), d, l.rot_dims));
        if (keeps) own[kv * l.dim_p + d] = k;
        own_key[d] = Op<T>::to_float(k);
    }
    if (makes_v) own_value[tid - 256] = Op<T>::to_float(Op<T>::from_float(v));
    if (keeps)
        for (int i = tid - 512; i < l.vdim_p; i += 512)
            if (i >= 0) own[l.kv_heads * l.dim_p + kv * l.vdim_p + i] = Op<T>::from_float(row_v[i]);
    __syncthreads();
    auto own_or = [&](const Piece<T> &from, bool own_row, const float *own_at, float (&f)[8]) __attribute__((always_inline)) {
        from.unpack(f);
        if (own_row) load8(own_at, f);
    };
#pragma unroll
    for (int k = 0; k < PASSES; k++) {
        const int i = k * kWindowKeys + key_in;
        float s = 0.0f;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int at = e * 8 + c * 64;
            if (at < l.dim_p) {
                float f[8], y[8];
                own_or(key_piece[k][c], count_k > 0 && i >= keys - 1, own_key + at, f);
                load8(q + at, y);
#pragma unroll
                for (int j = 0; j < 8; j++) s = __builtin_fmaf(f[j], y[j], s);
            }
        }
        s += detail::dpp_term<0xB1, 0xF>(s);
        s += detail::dpp_term<0x4E, 0xF>(s);
        s += detail::dpp_term<0x141, 0xF>(s);
        if (e == 0) scores[i] = i < keys ? s : -INFINITY;
    }
    __syncthreads();
    // every wavefront has the maximum and the sum by itself
    float top = -INFINITY, sum = 0.0f;
#pragma unroll
    for (int k = 0; k < 4 * VP; k++) top = fmaxf(top, scores[k * 64 + lane]);
#pragma unroll
    for (int k = 32; k >= 1; k >>= 1) top = fmaxf(top, __shfl_xor(top, k));
#pragma unroll
    for (int k = 0; k < 4 * VP; k++) sum += matrix::weight_exp<T>(scores[k * 64 + lane] - top);
    sum = detail::wave_sum(sum);
    float acc[8] = {};
#pragma unroll
    for (int k = 0; k < VP; k++) {
        const int i = k * 256 + value_in;
        const float w = matrix::weight_exp<T>(scores[i] - top);
        float f[8];
        own_or(value_piece[k], count_k > 0 && i >= keys - 1, own_value + piece * 8, f);
#pragma unroll
        for (int j = 0; j < 8; j++) acc[j] = __builtin_fmaf(w, f[j], acc[j]);
    }
    // lanes of a row of sixteen with the same values, then the 64 rows in LDS
#pragma unroll
    for (int j = 0; j < 8; j++) {
        acc[j] += detail::dpp_term<0x128, 0xF>(acc[j]);   // row_ror 8
        acc[j] += detail::dpp_term<0x124, 0xF>(acc[j]);   // row_ror 4
    }
    if ((lane & 15) < 4) {
        float4 *to = reinterpret_cast<float4 *>(&meet[tid >> 4][piece * 8]);
        to[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
        to[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
    }
    __syncthreads();
    if (wave) return;
    float o = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; i++) o += meet[(lane >> 5) * 32 + i][lane & 31];
    o += __shfl_xor(o, 32);
    if (lane >= kWindowSlice) return;
    o /= sum;
    const int at = h * l.vdim_p + slice * kWindowSlice + lane;
    if (p.mix) p.mix[(size_t)m * l.heads * l.vdim_p + at] = o;
    else static_cast<T *>(p.act)[(size_t)m * p.ld_act + at] = Op<T>::from_float(o);
}

// ---- prompt blocks ---------------------------------------------------------------------------------------
// One workgroup per row: queries normed and rotated to [heads][rows_p][dim_p] (rows past the block are zero), keys and values to the ring.
template <typename T>
__global__ __launch_bounds__(256) void attention_prepare_kernel(AttentionShape l, AttentionBlock p, int rows_p) {
    __shared__ float red[8];
    const int m = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    T *out = static_cast<T *>(p.q) + (size_t)m * l.dim_p;
    if (m >= p.rows) {
        for (int i = tid; i < l.heads * l.dim_p; i += 256) out[(size_t)(i / l.dim_p) * rows_p * l.dim_p + i % l.dim_p] = Op<T>::from_float(0.0f);
        return;
    }
    const int pos = p.base + m, kv = l.kv_heads * l.dim_p;
    const float *row = p.mixed + (size_t)m * l.ld_mix;
    const float *cos = l.cos + (size_t)pos * (l.rot_dims / 2), *sin = l.sin + (size_t)pos * (l.rot_dims / 2);
    float sq = detail::wave_sum(squares(row, l.heads * l.dim_p)), sk = l.k_at >= 0 ? detail::wave_sum(squares(row + l.k_at, kv)) : 0.0f;
    if (lane == 0) { red[tid >> 6] = sq; red[4 + (tid >> 6)] = sk; }
    __syncthreads();
    sq = (red[0] + red[1]) + (red[2] + red[3]);
    sk = (red[4] + red[5]) + (red[6] + red[7]);
    const float inv_q = 1.0f / sqrtf(sq / ((float)l.heads * (float)l.dim) + l.eps), inv_k = 1.0f / sqrtf(sk / ((float)l.kv_heads * (float)l.dim) + l.eps);
    for (int i = tid; i < l.heads * l.dim_p; i += 256) {
        const int h = i / l.dim_p, d = i - h * l.dim_p, at = h * l.dim_p;
        out[(size_t)h * rows_p * l.dim_p + d] = Op<T>::from_float(normed_rotated(row + at, l.q_norm + at, inv_q, d, l.rot_dims, cos, sin));
    }
    if (l.k_at < 0) return;
    T *own = static_cast<T *>(l.cache) + ((size_t)p.seq * l.ring + pos % l.ring) * cached_row(l);
    for (int i = tid; i < kv; i += 256) {
        const int at = i / l.dim_p * l.dim_p;
        own[i] = Op<T>::from_float(normed_rotated(row + l.k_at + at, l.k_norm + at, inv_k, i - at, l.rot_dims, cos, sin));
    }
    for (int i = tid; i < l.kv_heads * l.vdim_p; i += 256) own[kv + i] = Op<T>::from_float(row[l.k_at + kv + i]);
}

// The keys a block sees as rows, their values transposed; grid (tiles of 64 keys, slabs of 32 elements: keys, then values).
template <typename T>
__global__ __launch_bounds__(256) void attention_gather_kernel(AttentionShape l, AttentionBlock p) {
    __shared__ T slab[32][64 + 8];
    const int tid = threadIdx.x, i0 = blockIdx.x * 64, c0 = blockIdx.y * 32, kv = l.kv_heads * l.dim_p, width = cached_row(l);
    const T *cache = static_cast<const T *>(l.cache) + (size_t)p.seq * l.ring * width;
    const bool values = c0 >= kv;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int i = (tid >> 5) + 8 * k, c = tid & 31;
        const T x = i0 + i < p.keys ? cache[(size_t)((p.first_key + i0 + i) % l.ring) * width + c0 + c] : (T)0;
        if (values) slab[c][i] = x;
        else static_cast<T *>(p.k)[(size_t)(i0 + i) * kv + c0 + c] = x;
    }
    if (!values) return;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int c = (tid >> 6) + 4 * k, i = tid & 63;
        static_cast<T *>(p.vt)[(size_t)(c0 - kv + c) * p.keys_p + i0 + i] = slab[c][i];
    }
}

bool shape_ok(const AttentionShape &l) {
    return l.heads > 0 && l.kv_heads > 0 && l.heads % l.kv_heads == 0 && l.dim_p % 32 == 0 && l.vdim_p % 32 == 0 && l.dim > 0 && l.vdim > 0 && l.dim <= l.dim_p && l.vdim <= l.vdim_p &&
           l.rot_dims >= 0 && l.rot_dims <= l.dim && l.rot_dims % 2 == 0 && l.window >= 1 && l.ring >= 1 && l.cache && l.vdim_p <= kAttentionMaxHead && l.dim_p <= kAttentionMaxHead &&
           (l.k_at < 0 || (l.k_at >= l.heads * l.dim_p && l.k_norm && l.k_at + cached_row(l) <= l.ld_mix)) && l.q_norm && l.heads * l.dim_p <= l.ld_mix;
}

int heads_together(const AttentionShape &l) {
    const int share = l.heads / l.kv_heads;
    return share <= 1 ? 1 : share <= 2 ? 2 : share <= 4 ? 4 : 8;
}

template <typename T, int Q>
hipError_t run_partial(const AttentionShape &l, const AttentionStep &p, hipStream_t s) {
    const int chunks = (l.heads / l.kv_heads + Q - 1) / Q, parts = 256 / (l.vdim_p / 8) < kTile ? 256 / (l.vdim_p / 8) : kTile;
    const size_t rows = (size_t)(Q * (l.dim_p + kTile + 4) + l.dim_p + l.vdim_p) * 4, sums = (size_t)parts * l.vdim_p * 4, lds = rows + meeting_heads(Q) * sums;
    if (rows + sums > 62 * 1024) return hipErrorInvalidValue;
    if (lds > 62 * 1024) {   // four heads' sums beside eight long queries: 86 KB at most
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&attention_partial_kernel<T, Q>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((attention_partial_kernel<T, Q>), dim3(p.splits, l.kv_heads * chunks, p.rows), dim3(256), lds, s, l, p);
    return hipGetLastError();
}

template <typename T>
hipError_t run_step(const AttentionShape &l, const AttentionStep &p, hipStream_t s) {
    hipError_t e;
    const int span = l.window < l.max_seq ? l.window : l.max_seq;
    // Windows that a workgroup's registers hold, and as many workgroups as there are compute units: every one of them reads all keys of its head.  Layers of 16 heads of 128, four key heads (64 workgroups a row), us a
    // layer and step, two launches / one: window 256, one row 13.4 / 7, 512 bf16 13.4 / 9 (1024, two spans of registers: 13.4 / 15; 512 fp32: the same); a generation of 4 rows 11.4 / 11.2 ms, of 16 rows 20.2 / 20.5.
    if (const dim3 grid(l.heads * (l.vdim_p / kWindowSlice), p.rows); l.dim_p <= kWindowHead && (long)grid.x * grid.y <= 256 && span <= (sizeof(T) == 2 ? 512 : 256)) {
        if (span <= 256) hipLaunchKernelGGL((attention_window_kernel<T, 2>), grid, dim3(1024), 0, s, l, p);
        else if constexpr (sizeof(T) == 2) hipLaunchKernelGGL((attention_window_kernel<T, 4>), grid, dim3(1024), 0, s, l, p);
        return hipGetLastError();
    }
    switch (heads_together(l)) {
        case 1: e = run_partial<T, 1>(l, p, s); break;
        case 2: e = run_partial<T, 2>(l, p, s); break;
        case 4: e = run_partial<T, 4>(l, p, s); break;
        default: e = run_partial<T, 8>(l, p, s); break;
    }
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((attention_merge_kernel<T>), dim3(l.heads, p.rows), dim3(256), 0, s, l, p);
    return hipGetLastError();
}

template <typename T>
hipError_t run_block(const AttentionShape &l, const AttentionBlock &p, hipStream_t s) {
    const int rows_p = (p.rows + 31) / 32 * 32;
    hipLaunchKernelGGL((attention_prepare_kernel<T>), dim3(rows_p), dim3(256), 0, s, l, p, rows_p);
    hipLaunchKernelGGL((attention_gather_kernel<T>), dim3(p.keys_p / 64, cached_row(l) / 32), dim3(256), 0, s, l, p);
    return hipGetLastError();
}

}  // namespace

int attention_step_splits(const AttentionShape &l) {
    const int span = l.window < l.max_seq ? l.window : l.max_seq, tiles = (span + kTile - 1) / kTile;
    const int groups = l.kv_heads * ((l.heads / l.kv_heads + heads_together(l) - 1) / heads_together(l)), wanted = (512 + groups - 1) / groups, most = wanted < 64 ? wanted : 64;
    return tiles < most ? tiles : most;
}

hipError_t launch_attention_step(const AttentionShape &l, const AttentionStep &p, Precision type, hipStream_t s) {
    if (!shape_ok(l) || p.rows < 1 || p.splits < 1 || p.splits > 64 || (!p.mix && !p.act)) return hipErrorInvalidValue;
    return type == Precision::bf16 ? run_step<uint16_t>(l, p, s) : run_step<float>(l, p, s);
}

hipError_t launch_attention_block(const AttentionShape &l, const AttentionBlock &p, Precision type, hipStream_t s) {
    if (!shape_ok(l) || p.rows < 1 || p.base < 0 || p.base + p.rows > l.max_seq || p.first_key < 0 || p.first_key > p.base || p.keys != p.base + p.rows - p.first_key || p.keys > l.ring ||
        p.keys_p % 64 || p.keys_p < p.keys)
        return hipErrorInvalidValue;
    const hipError_t e = type == Precision::bf16 ? run_block<uint16_t>(l, p, s) : run_block<float>(l, p, s);
    if (e != hipSuccess) return e;
    BlockAttention b;
    b.heads = l.heads; b.kv_heads = l.kv_heads; b.dim_p = l.dim_p; b.vdim_p = l.vdim_p; b.window = l.window; b.scale = l.scale;
    b.rows = p.rows; b.before = p.base - p.first_key; b.keys_p = p.keys_p; b.q = p.q; b.k = p.k; b.vt = p.vt; b.act = p.act; b.ld_act = p.ld_act;
    return launch_block_attention(b, type, s);
}

}  // namespace esp
