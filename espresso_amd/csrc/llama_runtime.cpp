#include "llama_runtime.h"

#include "kernels/block_gemm.h"
#include "kernels/rows_gemm.h"
#include "kernels/span_attention.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>

namespace esp {
namespace {

// fp16 bits -> float on the host (weights arrive as raw bytes)
float half_to_float_host(uint16_t h) {
    uint32_t sign = ((uint32_t)h & 0x8000u) << 16, exp = (h >> 10) & 0x1Fu, mant = h & 0x3FFu, f;
    if (exp == 0) {
        if (mant == 0) f = sign;
        else {
            int e = -1;
            do { mant <<= 1; e++; } while ((mant & 0x400u) == 0);
            f = sign | ((uint32_t)(127 - 15 - e) << 23) | ((mant & 0x3FFu) << 13);
        }
    } else if (exp == 31) f = sign | 0x7F800000u | (mant << 13);
    else f = sign | ((exp + 112u) << 23) | (mant << 13);
    float out;
    std::memcpy(&out, &f, 4);
    return out;
}

}  // namespace

int LlamaRuntime::create(const LlamaConfig &c, LlamaRuntime **out) {
    *out = nullptr;
    // validateRuntimeConfig (RealModelInferenceEngine.swift:7615-7634)
    if (c.n_layer <= 0 || c.n_head <= 0 || c.n_kv_head <= 0 || c.d_model <= 0 || c.head_dim <= 0 ||
        c.hidden_dim <= 0 || c.vocab <= 0 || c.max_seq <= 0)
        return fail(ESP_ERR_INVALID_ARGUMENT, "llama config: every dimension must be positive");
    if (c.n_head % c.n_kv_head != 0)
        return fail(ESP_ERR_INVALID_ARGUMENT, "llama config: nHead %d is not a multiple of nKVHead %d", c.n_head, c.n_kv_head);
    if (c.head_dim % 2 != 0) return fail(ESP_ERR_INVALID_ARGUMENT, "llama config: headDim %d must be even", c.head_dim);
    if (c.kv_format != FMT_F32 && c.kv_format != FMT_F16)
        return fail(ESP_ERR_INVALID_ARGUMENT, "llama config: KV cache format must be f32 or f16");
    if (c.max_sequences < 1 || c.max_sequences > kMaxStepRows)
        return fail(ESP_ERR_INVALID_ARGUMENT, "llama config: max_sequences must be 1..%d", kMaxStepRows);
    int rc = ensure_init();
    if (rc != ESP_OK) return rc;
    LlamaRuntime *rt = new LlamaRuntime();
    rt->c_ = c;
    rt->h_layers_.resize(c.n_layer);
    *out = rt;
    return ESP_OK;
}

LlamaRuntime::~LlamaRuntime() {
    free_device(embedding_);
    free_device(final_norm_);
    matrix_release(&lm_head_);
    for (Layer &L : layers_) {
        free_device(L.rms_att); free_device(L.rms_ffn); free_device(L.q_norm); free_device(L.k_norm);
        matrix_release(&L.wqkv); matrix_release(&L.wo); matrix_release(&L.w13); matrix_release(&L.w2);
        free_device(L.k_cache); free_device(L.v_cache);
    }
    free_device(rope_cos_); free_device(rope_sin_);
    free_device(qkv_); free_device(q_); free_device(gu_);
    free_device(xn_); free_device(ctx_); free_device(act_);
    free_device(xn_lo_); free_device(ctx_lo_); free_device(act_lo_); free_device(xn_sums_); free_device(ctx_sums_); free_device(act_sums_);
    free_device(attn_scratch_);
    free_device(gemm_workspace_);
    free_device(d_tiles_);
    release_loop_session();
}

// Launches the GEMV of one class for every layer in turn (the head: the same matrix), `iters` rounds, between
// two events: back-to-back dependent launches at the real shapes over the real weights, which no cache can hold
// across a round.  The epilogues write into the step's buffers, so sequence state is garbage afterwards.
// The decode step (one or two rows) runs attention as a single launch that leaves per-head partial states, and
// the wo GEMV merges them while staging, when the head size and the matrix allow it.
bool LlamaRuntime::wo_merges_attention(const Layer &L, int rows) const {
    return merged_attention_ && c_.n_head % c_.n_kv_head == 0 && rows <= 2 &&
           L.wo.cols == c_.attention_dim() && gemv_merges_attention_partials(L.wo, rows, c_.head_dim);
}

// Small models, one row or two: five launches a layer are four.  Both counts, so that a row is the same alone and beside another.
bool LlamaRuntime::projects_attention(const Layer &L, int rows) const {
    return merged_attention_ && rows <= 2 && attention_project_supported(L.wo, c_.n_head, c_.n_kv_head, c_.head_dim, c_.max_seq) && gemv_adds_planes(L.w13) && L.w13.cols == L.wo.rows &&
           (size_t)rows * (c_.n_head + 1) * c_.d_model <= gemm_workspace_floats_;
}

int LlamaRuntime::time_kernel_class(int kernel_class, int iters, double *mean_us, double *kernel_only_us) {
    if (!finalized_ || iters < 1 || !mean_us) return fail(ESP_ERR_INVALID_ARGUMENT, "time_kernel_class: bad argument");
    if (kernel_class < K_QKV || kernel_class > K_HEAD) return fail(ESP_ERR_INVALID_ARGUMENT, "time_kernel_class: class %d", kernel_class);
    hipStream_t s = context().stream;
    const int kd = c_.kv_dim();
    const bool kv16 = c_.kv_format == FMT_F16;
    auto launch = [&](const Layer *L, hipEvent_t start = nullptr, hipEvent_t stop = nullptr) -> hipError_t {
        GemvParams g;
        g.batch = 1;
        g.start_event = start;
        g.stop_event = stop;
        switch (kernel_class) {
        case K_QKV:
            if (L->q_norm) { g.w = L->wqkv; g.norm_x = hidden_; g.norm_w = L->rms_att; g.norm_eps = c_.norm_eps; g.y = qkv_; g.epilogue = EPI_STORE_F32; break; }
            g.w = L->wqkv; g.norm_x = hidden_; g.norm_w = L->rms_att; g.norm_eps = c_.norm_eps; g.epilogue = EPI_QKV_ROPE;
            g.qkv.n_head = c_.n_head; g.qkv.n_kv_head = c_.n_kv_head; g.qkv.head_dim = c_.head_dim; g.qkv.max_seq = c_.max_seq;
            g.qkv.rope_cos = rope_cos_; g.qkv.rope_sin = rope_sin_; g.qkv.pos = d_pos_; g.qkv.seq = d_seq_;
            g.qkv.q_out = q_; g.qkv.k_cache = L->k_cache; g.qkv.v_cache = L->v_cache;
            g.qkv.cache_seq_stride = (size_t)kd * c_.max_seq; g.qkv.kv_f16 = kv16 ? 1 : 0;
            break;
        case K_WO:
            g.w = L->wo; g.x = ctx_; g.y = hidden_; g.residual = hidden_; g.epilogue = EPI_ADD_RESIDUAL;
            if (wo_merges_attention(*L, 1)) { g.x = nullptr; g.merge_partials = attn_scratch_; g.merge_head_dim = c_.head_dim; }
            break;
        case K_GATE_UP:
            g.w = L->w13; g.norm_w = L->rms_ffn; g.norm_eps = c_.norm_eps; g.out_f16 = act_; g.epilogue = EPI_SWIGLU_F16;
            if (projects_attention(*L, 1)) { g.norm_planes = gemm_workspace_; g.norm_plane_count = c_.n_head; g.norm_sum = gemm_workspace_ + (size_t)c_.n_head * c_.d_model; }
            else g.norm_x = hidden_;
            g.split_out = split_activations_ && gemv_splits_activations(L->w2, 1);
            break;
        case K_DOWN: g.w = L->w2; g.x = act_; g.y = hidden_; g.residual = hidden_; g.epilogue = EPI_ADD_RESIDUAL; break;
        default:
            g.w = lm_head_; g.norm_x = hidden_; g.norm_w = final_norm_; g.norm_eps = c_.norm_eps; g.y = logits_; g.epilogue = EPI_STORE_F32;
            if (head_fuses_argmax()) {   // what a greedy step launches
                g.y = nullptr; g.epilogue = EPI_ARGMAX;
                g.argmax_value = argmax_scratch_.part_value; g.argmax_index = argmax_scratch_.part_index; g.argmax_capacity = head_partial_capacity_;
            }
            break;
        }
        // what the decode step launches: split activations wherever the GEMV takes them (not for fp16 rows given unsplit)
        g.split_x = kernel_class != K_HEAD && !(g.x == ctx_ && kernel_class == K_WO) && split_activations_ && gemv_splits_activations(g.w, 1);
        return launch_gemv(g, s);
    };
    std::vector<const Layer *> round;   // the class's launches of a step
    if (kernel_class == K_HEAD) round.push_back(nullptr);
    else
        for (const Layer &L : layers_)
            if (kernel_class != K_WO || !projects_attention(L, 1)) round.push_back(&L);
    *mean_us = 0.0;
    if (kernel_only_us) *kernel_only_us = 0.0;
    if (round.empty()) return ESP_OK;
    StepRows rows{};
    rows.count = 1;
    ESP_HIP_TRY(launch_set_rows(rows, d_tokens_, d_pos_, d_seq_, s));
    hipEvent_t t0 = take_event(), t1 = take_event();
    if (!t0 || !t1) return fail(ESP_ERR_OUT_OF_MEMORY, "time_kernel_class: events");
    const int per_round = (int)round.size();
    for (const Layer *L : round) ESP_HIP_TRY(launch(L));   // warm-up round
    ESP_HIP_TRY(hipEventRecord(t0, s));
    for (int r = 0; r < iters; r++)
        for (const Layer *L : round) ESP_HIP_TRY(launch(L));
    ESP_HIP_TRY(hipEventRecord(t1, s));
    ESP_HIP_TRY(hipEventSynchronize(t1));
    float ms = 0.0f;
    ESP_HIP_TRY(hipEventElapsedTime(&ms, t0, t1));
    event_pool_.push_back(t0);
    event_pool_.push_back(t1);
    *mean_us = (double)ms * 1e3 / ((double)iters * per_round);
    if (kernel_only_us) {
        // the same launches again, each with events of its own that take the kernel's start and end
        std::vector<hipEvent_t> ev((size_t)iters * per_round * 2, nullptr);
        for (hipEvent_t &e : ev) if (!(e = take_event())) return fail(ESP_ERR_OUT_OF_MEMORY, "time_kernel_class: events");
        for (int r = 0, k = 0; r < iters; r++)
            for (int i = 0; i < per_round; i++, k += 2)
                ESP_HIP_TRY(launch(round[(size_t)i], ev[(size_t)k], ev[(size_t)k + 1]));
        ESP_HIP_TRY(hipStreamSynchronize(s));
        double total = 0.0;
        for (size_t k = 0; k < ev.size(); k += 2) {
            ESP_HIP_TRY(hipEventElapsedTime(&ms, ev[k], ev[k + 1]));
            total += ms;
        }
        for (hipEvent_t e : ev) event_pool_.push_back(e);
        *kernel_only_us = total * 1e3 / ((double)iters * per_round);
    }
    return ESP_OK;
}

size_t LlamaRuntime::kernel_bytes(int kernel_class) const {
    if (!finalized_ || layers_.empty()) return 0;
    const Layer &L = layers_[0];
    auto io = [](const DeviceMatrix &m) { return m.bytes() + (size_t)m.cols * 2 + (size_t)m.rows * 4; };
    switch (kernel_class) {
    case K_QKV: return io(L.wqkv);
    case K_WO: return projects_attention(L, 1) ? 0 : io(L.wo);   // (no launch of its own there)
    case K_GATE_UP: return io(L.w13);
    case K_DOWN: return io(L.w2);
    case K_HEAD: return io(lm_head_) - (head_fuses_argmax() ? (size_t)lm_head_.rows * 4 : 0);   // the fused head stores no logits
    default: return 0;
    }
}

LlamaRuntime::HostTensor *LlamaRuntime::host_slot(int layer, int slot) {
    switch (slot) {
    case SLOT_TOKEN_EMBEDDING: return &h_embedding_;
    case SLOT_FINAL_NORM: return &h_final_norm_;
    case SLOT_LM_HEAD: return &h_lm_head_;
    default: break;
    }
    if (layer < 0 || layer >= c_.n_layer) return nullptr;
    HostLayer &L = h_layers_[layer];
    switch (slot) {
    case SLOT_RMS_ATT: return &L.rms_att;
    case SLOT_WQ: return &L.wq;
    case SLOT_WK: return &L.wk;
    case SLOT_WV: return &L.wv;
    case SLOT_WO: return &L.wo;
    case SLOT_RMS_FFN: return &L.rms_ffn;
    case SLOT_W1: return &L.w1;
    case SLOT_W2: return &L.w2;
    case SLOT_W3: return &L.w3;
    case SLOT_Q_NORM: return &L.q_norm;
    case SLOT_K_NORM: return &L.k_norm;
    default: return nullptr;
    }
}

int LlamaRuntime::set_weight(int layer, int slot, int format, const void *data, size_t bytes) {
    if (finalized_) return fail(ESP_ERR_INVALID_ARGUMENT, "set_weight after finalize");
    HostTensor *t = host_slot(layer, slot);
    if (!t) return fail(ESP_ERR_INVALID_ARGUMENT, "set_weight: no slot %d in layer %d", slot, layer);
    if (!data || !format_supported(format)) return fail(ESP_ERR_INVALID_ARGUMENT, "set_weight: null data or unknown format %d", format);
    const size_t d = c_.d_model, ad = c_.attention_dim(), kd = c_.kv_dim(), hd = c_.hidden_dim;
    size_t elems = 0;
    switch (slot) {
    case SLOT_TOKEN_EMBEDDING: case SLOT_LM_HEAD: elems = (size_t)c_.vocab * d; break;
    case SLOT_FINAL_NORM: case SLOT_RMS_ATT: case SLOT_RMS_FFN: elems = d; break;
    case SLOT_WQ: case SLOT_WO: elems = ad * d; break;
    case SLOT_WK: case SLOT_WV: elems = kd * d; break;
    case SLOT_W1: case SLOT_W2: case SLOT_W3: elems = hd * d; break;
    case SLOT_Q_NORM: case SLOT_K_NORM: elems = (size_t)c_.head_dim; break;
    }
    const bool is_vector = slot == SLOT_FINAL_NORM || slot == SLOT_RMS_ATT || slot == SLOT_RMS_FFN ||
                           slot == SLOT_Q_NORM || slot == SLOT_K_NORM || slot == SLOT_TOKEN_EMBEDDING;
    if (is_vector && format != FMT_F32 && format != FMT_F16)
        return fail(ESP_ERR_UNSUPPORTED, "set_weight: slot %d takes f32 or f16 values", slot);
    if (elems % format_block_elems(format) != 0 || bytes != format_bytes(format, elems))
        return fail(ESP_ERR_INVALID_ARGUMENT, "set_weight: slot %d expects %zu elements (%zu bytes in format %d), got %zu bytes",
                    slot, elems, format_bytes(format, elems), format, bytes);
    t->format = format;
    t->bytes.assign(static_cast<const uint8_t *>(data), static_cast<const uint8_t *>(data) + bytes);
    return ESP_OK;
}

int LlamaRuntime::upload_vector(const HostTensor &t, size_t count, float **out, const char *what) {
    if (t.format < 0) return fail(ESP_ERR_INVALID_ARGUMENT, "finalize: missing weight %s", what);
    std::vector<float> v(count);
    if (t.format == FMT_F32) std::memcpy(v.data(), t.bytes.data(), count * 4);
    else for (size_t i = 0; i < count; i++) v[i] = half_to_float_host((uint16_t)(t.bytes[2 * i] | (t.bytes[2 * i + 1] << 8)));
    int rc = device_alloc(out, count);
    if (rc != ESP_OK) return rc;
    ESP_HIP_TRY(hipMemcpy(*out, v.data(), count * 4, hipMemcpyHostToDevice));
    return ESP_OK;
}

int LlamaRuntime::finalize() {
    if (finalized_) return ESP_OK;
    const int d = c_.d_model, ad = c_.attention_dim(), kd = c_.kv_dim(), hd = c_.hidden_dim, half = c_.head_dim / 2;
    int rc;
    // ---- top level ----
    if (h_embedding_.format < 0) return fail(ESP_ERR_INVALID_ARGUMENT, "finalize: missing token embedding");
    embedding_f16_ = h_embedding_.format == FMT_F16;
    {
        uint8_t *p = nullptr;
        if ((rc = device_alloc(&p, h_embedding_.bytes.size())) != ESP_OK) return rc;
        embedding_ = p;
        ESP_HIP_TRY(hipMemcpy(embedding_, h_embedding_.bytes.data(), h_embedding_.bytes.size(), hipMemcpyHostToDevice));
    }
    if ((rc = upload_vector(h_final_norm_, d, &final_norm_, "rms_final")) != ESP_OK) return rc;
    if (h_lm_head_.format < 0) return fail(ESP_ERR_INVALID_ARGUMENT, "finalize: missing lm_head");
    if ((rc = matrix_upload(h_lm_head_.format, h_lm_head_.bytes.data(), c_.vocab, d, &lm_head_)) != ESP_OK) return rc;
    weight_bytes_ = lm_head_.bytes();
    resident_weight_bytes_ = lm_head_.resident_bytes() + h_embedding_.bytes.size();

    // ---- layers ----
    layers_.resize(c_.n_layer);
    const size_t cache_elems = (size_t)c_.max_sequences * kd * c_.max_seq;
    const size_t cache_bytes = cache_elems * (c_.kv_format == FMT_F16 ? 2 : 4);
    std::vector<uint8_t> fused;
    for (int l = 0; l < c_.n_layer; l++) {
        HostLayer &H = h_layers_[l];
        Layer &L = layers_[l];
        const HostTensor *need[] = {&H.wq, &H.wk, &H.wv, &H.wo, &H.w1, &H.w2, &H.w3};
        for (const HostTensor *t : need)
            if (t->format < 0) return fail(ESP_ERR_INVALID_ARGUMENT, "finalize: layer %d is missing a projection weight", l);
        if (H.wq.format != H.wk.format || H.wq.format != H.wv.format)
            return fail(ESP_ERR_UNSUPPORTED, "finalize: layer %d wq/wk/wv must share one format", l);
        if (H.w1.format != H.w3.format) return fail(ESP_ERR_UNSUPPORTED, "finalize: layer %d w1/w3 must share one format", l);
        if ((rc = upload_vector(H.rms_att, d, &L.rms_att, "rms_att")) != ESP_OK) return rc;
        if ((rc = upload_vector(H.rms_ffn, d, &L.rms_ffn, "rms_ffn")) != ESP_OK) return rc;
        // q_norm/k_norm are optional and only used when both exist (:6585-6607)
        if (H.q_norm.format >= 0 && H.k_norm.format >= 0) {
            if ((rc = upload_vector(H.q_norm, c_.head_dim, &L.q_norm, "q_norm")) != ESP_OK) return rc;
            if ((rc = upload_vector(H.k_norm, c_.head_dim, &L.k_norm, "k_norm")) != ESP_OK) return rc;
        }
        // fused QKV: q and k rows reordered so that the two rows of a RoPE pair (j, j + half) are
        // adjacent; v rows in natural order.
        {
            const size_t rb = format_bytes(H.wq.format, d);
            fused.resize((size_t)(ad + 2 * kd) * rb);
            size_t o = 0;
            auto put_rope_rows = [&](const HostTensor &t, int heads) {
                for (int h = 0; h < heads; h++)
                    for (int j = 0; j < half; j++) {
                        std::memcpy(&fused[o], &t.bytes[(size_t)(h * c_.head_dim + j) * rb], rb); o += rb;
                        std::memcpy(&fused[o], &t.bytes[(size_t)(h * c_.head_dim + j + half) * rb], rb); o += rb;
                    }
            };
            put_rope_rows(H.wq, c_.n_head);
            put_rope_rows(H.wk, c_.n_kv_head);
            std::memcpy(&fused[o], H.wv.bytes.data(), (size_t)kd * rb);
            if ((rc = matrix_upload(H.wq.format, fused.data(), ad + 2 * kd, d, &L.wqkv)) != ESP_OK) return rc;
        }
        // fused gate/up: rows interleaved (g0, u0, g1, u1, ...)
        {
            const size_t rb = format_bytes(H.w1.format, d);
            fused.resize((size_t)2 * hd * rb);
            for (int i = 0; i < hd; i++) {
                std::memcpy(&fused[(size_t)(2 * i) * rb], &H.w1.bytes[(size_t)i * rb], rb);
                std::memcpy(&fused[(size_t)(2 * i + 1) * rb], &H.w3.bytes[(size_t)i * rb], rb);
            }
            if ((rc = matrix_upload(H.w1.format, fused.data(), 2 * hd, d, &L.w13)) != ESP_OK) return rc;
        }
        if ((rc = matrix_upload(H.wo.format, H.wo.bytes.data(), d, ad, &L.wo)) != ESP_OK) return rc;
        if ((rc = matrix_upload(H.w2.format, H.w2.bytes.data(), d, hd, &L.w2)) != ESP_OK) return rc;
        weight_bytes_ += L.wqkv.bytes() + L.wo.bytes() + L.w13.bytes() + L.w2.bytes();
        resident_weight_bytes_ += L.wqkv.resident_bytes() + L.wo.resident_bytes() + L.w13.resident_bytes() + L.w2.resident_bytes();
        uint8_t *kc = nullptr, *vc = nullptr;
        if ((rc = device_alloc(&kc, cache_bytes)) != ESP_OK) return rc;
        L.k_cache = kc;
        if ((rc = device_alloc(&vc, cache_bytes)) != ESP_OK) return rc;
        L.v_cache = vc;
        H = HostLayer{};  // drop the host copy
    }
    h_embedding_ = HostTensor{}; h_lm_head_ = HostTensor{};
    fused.clear(); fused.shrink_to_fit();

    // ---- RoPE table, computed on the host with the reference's float expressions (:6759-6762) ----
    {
        std::vector<float> cs((size_t)c_.max_seq * half), sn((size_t)c_.max_seq * half);
        for (int p = 0; p < c_.max_seq; p++)
            for (int j = 0; j < half; j++) {
                const float frequency = 1.0f / powf(c_.rope_theta, (float)(2 * j) / (float)c_.head_dim);
                const float angle = (float)p * frequency;
                cs[(size_t)p * half + j] = cosf(angle);
                sn[(size_t)p * half + j] = sinf(angle);
            }
        if ((rc = device_alloc(&rope_cos_, cs.size())) != ESP_OK) return rc;
        if ((rc = device_alloc(&rope_sin_, sn.size())) != ESP_OK) return rc;
        ESP_HIP_TRY(hipMemcpy(rope_cos_, cs.data(), cs.size() * 4, hipMemcpyHostToDevice));
        ESP_HIP_TRY(hipMemcpy(rope_sin_, sn.data(), sn.size() * 4, hipMemcpyHostToDevice));
    }
    // ---- activations ----
    {
        const char *pa = getenv("ESPRESSO_HIP_PROMPT_ATTENTION");   // "0": prompt blocks keep the single-query attention kernel
        const bool block_attention = !(pa && pa[0] == '0');
        prompt_attention_ = block_attention && attention_prompt_supported(c_.n_head, c_.n_kv_head, c_.head_dim);
        short_span_attention_ = block_attention && span_attention_supported(c_.n_head, c_.n_kv_head, c_.head_dim);
        span_attention_ = block_attention && !prompt_attention_ && span_attention_supported(c_.n_head, c_.n_kv_head, c_.head_dim);
    }
    // the single-query attention kernel leaves its slices of every row of a block in scratch memory: those models keep short blocks
    const bool rows_attend_alone = !prompt_attention_ && !span_attention_;
    // (prompts of several sequences share blocks: room for up to 1024 rows of them)
    const long shared_rows = std::min<long>(1024, (long)c_.max_seq * c_.max_sequences);
    const size_t R = rows_attend_alone ? kMinPrefillBlockRows : prefill_block_rows(std::max(c_.max_seq, (int)shared_rows));
    if (c_.max_sequences > 1 && (rc = device_alloc(&d_tiles_, R / 32 + (size_t)c_.max_sequences)) != ESP_OK) return rc;
    if ((rc = allocate_common((int)R, d)) != ESP_OK) return rc;
    if ((rc = device_alloc(&qkv_, R * (ad + 2 * kd))) != ESP_OK) return rc;
    if ((rc = device_alloc(&q_, R * ad)) != ESP_OK) return rc;
    if ((rc = device_alloc(&gu_, R * 2 * hd)) != ESP_OK) return rc;
    if ((rc = device_alloc(&xn_, R * (size_t)(d > hd ? d : hd))) != ESP_OK) return rc;
    if ((rc = device_alloc(&ctx_, R * ad)) != ESP_OK) return rc;
    if ((rc = device_alloc(&act_, R * hd)) != ESP_OK) return rc;
    if (d % 256 == 0 && ad % 256 == 0 && hd % 256 == 0) {   // split rows for prompt blocks (Q4_K models)
        if ((rc = device_alloc(&xn_lo_, R * (size_t)d)) != ESP_OK) return rc;
        if ((rc = device_alloc(&ctx_lo_, R * (size_t)ad)) != ESP_OK) return rc;
        if ((rc = device_alloc(&act_lo_, R * (size_t)hd)) != ESP_OK) return rc;
        if ((rc = device_alloc(&xn_sums_, R * (size_t)(d / 16))) != ESP_OK) return rc;
        if ((rc = device_alloc(&ctx_sums_, R * (size_t)(ad / 16))) != ESP_OK) return rc;
        if ((rc = device_alloc(&act_sums_, R * (size_t)(hd / 16))) != ESP_OK) return rc;
    }
    {
        const size_t per_row = (size_t)c_.n_kv_head * kAttentionMaxSplits * (c_.n_head / c_.n_kv_head) * (c_.head_dim + 2);
        if ((rc = device_alloc(&attn_scratch_, (rows_attend_alone ? R : (size_t)kMaxStepRows) * per_row)) != ESP_OK) return rc;
    }
    gemm_workspace_floats_ = R * kGemmWorkspaceFloatsPerRow;
    if ((rc = device_alloc(&gemm_workspace_, gemm_workspace_floats_)) != ESP_OK) return rc;
    if (gemm_split_shared_k_pool(&gemm_shared_k_) != hipSuccess) {   // without the pool the prompt GEMM keeps its plain grid
        (void)hipGetLastError();
        gemm_shared_k_ = GemmSplitSharedK{};
    }
    {
        const char *fh = getenv("ESPRESSO_HIP_FUSED_HEAD_ARGMAX");   // "0": the head stores logits and separate launches pick the token
        fused_head_argmax_ = !(fh && fh[0] == '0');
        const char *sa = getenv("ESPRESSO_HIP_SPLIT_ACTIVATIONS");   // "0": activations rounded to fp16 once
        if (sa && sa[0] == '0') split_activations_ = false;
    }
    return finish_finalize();
}

int LlamaRuntime::clear_state() {
    const size_t cache_bytes = (size_t)c_.max_sequences * c_.kv_dim() * c_.max_seq * (c_.kv_format == FMT_F16 ? 2 : 4);
    for (Layer &L : layers_) {
        ESP_HIP_TRY(hipMemsetAsync(L.k_cache, 0, cache_bytes, context().stream));
        ESP_HIP_TRY(hipMemsetAsync(L.v_cache, 0, cache_bytes, context().stream));
    }
    return ESP_OK;
}

// The trunk over `M` rows whose (token, position, sequence) already sit in d_tokens_/d_pos_/d_seq_.
int LlamaRuntime::enqueue_trunk(int M, bool embedded, float *final_out) {
    hipStream_t s = context().stream;
    const int d = c_.d_model, ad = c_.attention_dim(), kd = c_.kv_dim();
    const bool kv16 = c_.kv_format == FMT_F16;
    int rc = ESP_OK;
    if (!embedded) ESP_HIP_TRY(launch_embed(embedding_, embedding_f16_, d_tokens_, M, d, hidden_, s));
    if (timing_enabled_) {   // an empty event pair: the overhead the pairs around real kernels carry
        if ((rc = time_begin(K_EVENT_PAIR)) != ESP_OK) return rc;
        if ((rc = time_end()) != ESP_OK) return rc;
    }
    // more than two rows (batched sequences, batched verify): one pass over the weights on the matrix cores
    if (M > 2 && matrix_prefill_ && matrix_prefill_supported()) return sixteen_rows_supported(M) ? enqueue_layers_sixteen(M) : enqueue_layers_matrix(M);
    for (Layer &L : layers_) {
        // both RMSNorms of the layer run inside the staging of the GEMV that consumes them
        GemvParams g;
        g.w = L.wqkv; g.norm_x = hidden_; g.norm_w = L.rms_att; g.norm_eps = c_.norm_eps; g.batch = M;
        // Activations reach the matrix cores as hi / lo fp16 pairs wherever the GEMV has that form (GemvParams::split_x)
        g.split_x = split_activations_ && gemv_splits_activations(L.wqkv, M);
        const size_t cache_seq_stride = (size_t)kd * c_.max_seq;
        if (L.q_norm) {
            // per-head q/k norm needs whole heads before RoPE: plain GEMV, then the post kernel
            g.y = qkv_; g.epilogue = EPI_STORE_F32;
            if ((rc = time_begin(K_QKV)) != ESP_OK) return rc;
            ESP_HIP_TRY(launch_gemv(g, s));
            if ((rc = time_end()) != ESP_OK) return rc;
            QkvPostArgs qa{};
            qa.qkv = qkv_; qa.q_norm = L.q_norm; qa.k_norm = L.k_norm; qa.norm_eps = c_.norm_eps;
            qa.n_head = c_.n_head; qa.n_kv_head = c_.n_kv_head; qa.head_dim = c_.head_dim; qa.max_seq = c_.max_seq;
            qa.rope_cos = rope_cos_; qa.rope_sin = rope_sin_; qa.pos = d_pos_; qa.seq = d_seq_;
            qa.q_out = q_; qa.k_cache = L.k_cache; qa.v_cache = L.v_cache; qa.cache_seq_stride = cache_seq_stride;
            ESP_HIP_TRY(launch_qkv_post(qa, M, kv16, s));
        } else {
            g.epilogue = EPI_QKV_ROPE;
            g.qkv.n_head = c_.n_head; g.qkv.n_kv_head = c_.n_kv_head; g.qkv.head_dim = c_.head_dim; g.qkv.max_seq = c_.max_seq;
            g.qkv.rope_cos = rope_cos_; g.qkv.rope_sin = rope_sin_; g.qkv.pos = d_pos_; g.qkv.seq = d_seq_;
            g.qkv.q_out = q_; g.qkv.k_cache = L.k_cache; g.qkv.v_cache = L.v_cache;
            g.qkv.cache_seq_stride = cache_seq_stride; g.qkv.kv_f16 = kv16 ? 1 : 0;
            if ((rc = time_begin(K_QKV)) != ESP_OK) return rc;
            ESP_HIP_TRY(launch_gemv(g, s));
            if ((rc = time_end()) != ESP_OK) return rc;
        }
        AttentionArgs aa{};
        aa.q = q_; aa.k_cache = L.k_cache; aa.v_cache = L.v_cache; aa.cache_seq_stride = cache_seq_stride;
        aa.n_head = c_.n_head; aa.n_kv_head = c_.n_kv_head; aa.head_dim = c_.head_dim; aa.max_seq = c_.max_seq;
        aa.pos = d_pos_; aa.seq = d_seq_; aa.ctx_f16 = ctx_;
        aa.split_scratch = attn_scratch_;
        aa.head_partials = attn_scratch_;
        // one attention launch instead of two where the wo GEMV can merge the partial states in its staging
        const bool project = projects_attention(L, M);   // one launch for attention and wo, whose planes the gate|up GEMV adds
        float *const planes = gemm_workspace_, *const joined = gemm_workspace_ + (size_t)M * c_.n_head * d;
        const bool merge_in_wo = !project && wo_merges_attention(L, M);
        if ((rc = time_begin(K_ATTENTION)) != ESP_OK) return rc;
        if (project) ESP_HIP_TRY(launch_attention_project(aa, L.wo, M, hidden_, planes, kv16, s));
        else if (merge_in_wo) ESP_HIP_TRY(launch_attention_partials(aa, M, kv16, s));
        else ESP_HIP_TRY(launch_attention(aa, M, kv16, s));
        if ((rc = time_end()) != ESP_OK) return rc;
        g = GemvParams{};
        g.batch = M;
        g.w = L.wo; g.x = ctx_; g.y = hidden_; g.residual = hidden_; g.epilogue = EPI_ADD_RESIDUAL;
        if (!project) {
            if (merge_in_wo) {
                g.x = nullptr; g.merge_partials = attn_scratch_; g.merge_head_dim = c_.head_dim;
                g.split_x = split_activations_ && gemv_splits_activations(L.wo, M);   // the merge leaves fp32 values to split
            }
            if ((rc = time_begin(K_WO)) != ESP_OK) return rc;
            ESP_HIP_TRY(launch_gemv(g, s));
            if ((rc = time_end()) != ESP_OK) return rc;
        }
        g.w = L.w13; g.x = nullptr; g.merge_partials = nullptr; g.norm_w = L.rms_ffn; g.norm_eps = c_.norm_eps;
        if (project) { g.norm_planes = planes; g.norm_plane_count = c_.n_head; g.norm_sum = joined; }
        else g.norm_x = hidden_;
        g.y = nullptr; g.residual = nullptr; g.out_f16 = act_; g.epilogue = EPI_SWIGLU_F16;
        const bool split_down = split_activations_ && gemv_splits_activations(L.w2, M);   // act_ then holds hi / lo row pairs
        g.split_x = split_activations_ && gemv_splits_activations(L.w13, M);
        g.split_out = split_down;
        if ((rc = time_begin(K_GATE_UP)) != ESP_OK) return rc;
        ESP_HIP_TRY(launch_gemv(g, s));
        if ((rc = time_end()) != ESP_OK) return rc;
        g.w = L.w2; g.x = act_; g.norm_x = nullptr; g.norm_planes = nullptr; g.norm_w = nullptr; g.split_x = split_down; g.split_out = false;
        g.y = final_out && &L == &layers_.back() ? final_out : hidden_;   // the last layer's output may go straight to its keeper
        g.residual = project ? joined : hidden_; g.out_f16 = nullptr; g.epilogue = EPI_ADD_RESIDUAL;
        if ((rc = time_begin(K_DOWN)) != ESP_OK) return rc;
        ESP_HIP_TRY(launch_gemv(g, s));
        if ((rc = time_end()) != ESP_OK) return rc;
    }
    (void)ad;
    return ESP_OK;
}

void LlamaRuntime::set_split_activations(bool enabled) {
    if (enabled == split_activations_) return;
    split_activations_ = enabled;
    drop_captured_graphs();   // captured with the other kernels
}

void LlamaRuntime::set_merged_attention(bool enabled) {
    if (enabled == merged_attention_) return;
    merged_attention_ = enabled;
    drop_captured_graphs();   // captured with the other path
}

void LlamaRuntime::release_loop_session() {
    DeviceLoopSession &ss = loop_session_;
    if (ss.one) (void)hipGraphExecDestroy(ss.one);
    if (ss.many) (void)hipGraphExecDestroy(ss.many);
    if (ss.state) (void)hipFree(ss.state);
    if (ss.log) (void)hipFree(ss.log);
    ss = DeviceLoopSession{};
}

bool LlamaRuntime::matrix_prefill_supported() const {
    auto ok = [](const DeviceMatrix &m) { return m.format != FMT_F32 && m.cols % 64 == 0; };
    for (const Layer &L : layers_)
        if (!ok(L.wqkv) || !ok(L.wo) || !ok(L.w13) || !ok(L.w2)) return false;
    return true;
}

bool LlamaRuntime::steps_hold_two_rows() const {
    for (const Layer &L : layers_)
        if (!gemv_holds_two_rows(L.wqkv) || !gemv_holds_two_rows(L.wo) || !gemv_holds_two_rows(L.w13) || !gemv_holds_two_rows(L.w2)) return false;
    return true;
}

// `rows` prompt tokens at positions base.. of one sequence: the layer loop of forwardToken (:6221-6347) over
// a block of rows, every projection as one dequant-fused MFMA GEMM.  Rows of the block see each other's
// keys and values causally because the whole block's K/V is written before its attention runs.
int LlamaRuntime::prefill_block(int seq, const uint32_t *tokens, int rows, int base, int last) {
    const PromptSpan span{seq, tokens, rows};
    const int rc = upload_block_rows(&span, 1, base);
    if (rc != ESP_OK) return rc;
    ESP_HIP_TRY(launch_embed(embedding_, embedding_f16_, d_tokens_, rows, c_.d_model, hidden_, context().stream));
    return enqueue_layers_matrix(rows, base + rows, last < rows ? last : 0);
}

// The rows beyond the last multiple of kMinPrefillBlockRows: a block of them alone is more exact where it takes 32-bit attention (fewer than 32 rows) or keeps weights that a long one rounds.  They are
// the rows whose logits the caller reads, so they stay as exact whatever is in front of them.
LastRows LlamaRuntime::last_rows(int count) const {
    const int rows = count % kMinPrefillBlockRows;
    if (count < kMinPrefillBlockRows || rows == 0) return {};
    const bool few = rows < kMatrixPrefillMinTokens;
    if (few && short_split_blocks_supported() && !split_blocks_supported()) return {rows, 0};   // activations are pairs there, which a long block has no place for
    if (few && finer_short_attention()) return {0, rows};
    if (split_blocks_supported()) return {};
    for (const Layer &L : layers_)
        for (const DeviceMatrix *m : {&L.wqkv, &L.wo, &L.w13, &L.w2})
            if (rounds_but_for_last(*m, rows, m == &L.w13)) return {0, rows};
    return {};
}
bool LlamaRuntime::rounds_but_for_last(const DeviceMatrix &m, int last, bool gate_up) const {
    return keeps_weights(m, last, gate_up) && !keeps_weights(m, kMinPrefillBlockRows, gate_up);
}

// Does a block of `rows` rows multiply with a layer's matrix as it is, no weight rounded to fp16?  (enqueue_layers_matrix asks launch_gemm)
bool LlamaRuntime::keeps_weights(const DeviceMatrix &m, int rows, bool gate_up) const {
    GemmParams p;
    int splits = 1;
    p.w = m; p.rows = rows; p.unrounded = true;
    if (gate_up) p.swiglu_out = act_;
    else p.deferred_splits = &splits;
    return gemm_keeps_weights(p);
}

// Products whose arithmetic does not hang on the block's rows: split rows (class 1); fp16 matrices, and packed ones that round their weights at the prompt's own rows already (class 2).  Attention
// is by prompt, with the kernel that the prompt's own length asks for.
int LlamaRuntime::shared_block_class(int count) const {
    const bool few = count < kMatrixPrefillMinTokens;
    if (const LastRows last = last_rows(count); last.own_block || last.in_block) return 0;
    if (few ? short_split_blocks_supported() : split_blocks_supported()) return 1;
    for (const Layer &L : layers_)
        for (const DeviceMatrix *m : {&L.wqkv, &L.wo, &L.w13, &L.w2})
            if (m->format != FMT_F16 && (m->format == FMT_F32 || count <= 128 || keeps_weights(*m, count, m == &L.w13))) return 0;
    return few && !short_span_attention_ ? 0 : 2;
}

// One pass over the weights for all of the prompts: 16 prompts of 15 to 60 tokens (600 rows) and 24 steps, eight 8B layers of Q4_K, 33.6 -> 23.3 ms (a pass for each prompt was bound by the weights'
// way from memory, 1.5 ms a layer for the sixteen; together 0.77).
int LlamaRuntime::prefill_shared_block(const PromptSpan *spans, int count) {
    int rc = upload_block_rows(spans, count, 0);
    if (rc != ESP_OK) return rc;
    hipStream_t s = context().stream;
    std::vector<int2> long_tiles, short_tiles;
    SharedBlock shared;
    int rows = 0;
    for (int k = 0; k < count; k++) {
        const bool few = spans[k].count < kMatrixPrefillMinTokens;
        (few ? shared.longest_short : shared.longest) = std::max(few ? shared.longest_short : shared.longest, spans[k].count);
        for (int r = 0; r < spans[k].count; r += 32) (few ? short_tiles : long_tiles).push_back(int2{rows + r, std::min(31, spans[k].count - 1 - r)});
        rows += spans[k].count;
    }
    shared.long_tiles = (int)long_tiles.size(); shared.short_tiles = (int)short_tiles.size();
    long_tiles.insert(long_tiles.end(), short_tiles.begin(), short_tiles.end());
    ESP_HIP_TRY(hipMemcpyAsync(d_tiles_, long_tiles.data(), sizeof(int2) * long_tiles.size(), hipMemcpyHostToDevice, s));
    ESP_HIP_TRY(hipStreamSynchronize(s));   // the vectors go out of scope
    ESP_HIP_TRY(launch_embed(embedding_, embedding_f16_, d_tokens_, rows, c_.d_model, hidden_, s));
    shared_ = shared;
    rc = shared_block_class(spans[0].count) == 1 ? enqueue_layers_split(rows, 0) : enqueue_layers_matrix(rows, 0);
    shared_ = SharedBlock{};
    return rc;
}

// Attention of a block: one prompt's rows (block_keys: the keys that the last of them sees), prompts that share it, or (neither) rows that attend alone.  Fewer than 32 rows of a prompt take 32-bit
// attention, as the steps they stand for, and so do all rows of models with fp16 caches (behind more than 2048 keys as far as their fp16 contexts show it: launch_span_attention).
int LlamaRuntime::enqueue_block_attention(AttentionArgs aa, int rows, int block_keys, int last) {
    hipStream_t s = context().stream;
    const bool kv16 = c_.kv_format == FMT_F16;
    if (last > 0 && last < kMatrixPrefillMinTokens && finer_short_attention() && !kv16) {
        const int ahead = rows - last;
        const size_t at = (size_t)ahead * c_.attention_dim();
        ESP_HIP_TRY(launch_prompt_attention(aa, ahead, block_keys - last, kv16, s));
        aa.q += at; aa.pos += ahead; aa.seq += ahead;
        aa.ctx_f16 += at;   // (split rows of so many belong to fp16 caches)
        ESP_HIP_TRY(launch_span_attention(aa, last, block_keys, kv16, s));
        return ESP_OK;
    }
    if (shared_.long_tiles + shared_.short_tiles > 0 && (prompt_attention_ || span_attention_)) {
        aa.tiles = d_tiles_; aa.tile_count = shared_.long_tiles;
        if (shared_.long_tiles && prompt_attention_) ESP_HIP_TRY(launch_prompt_attention(aa, shared_.longest, shared_.longest, kv16, s));
        else if (shared_.long_tiles) ESP_HIP_TRY(launch_span_attention(aa, shared_.longest, shared_.longest, kv16, s));
        aa.tiles = d_tiles_ + shared_.long_tiles; aa.tile_count = shared_.short_tiles;
        if (shared_.short_tiles) ESP_HIP_TRY(launch_span_attention(aa, shared_.longest_short, shared_.longest_short, kv16, s));
        return ESP_OK;
    }
    const bool few = rows < kMatrixPrefillMinTokens && short_span_attention_;
    if (block_keys && prompt_attention_ && !few) ESP_HIP_TRY(launch_prompt_attention(aa, rows, block_keys, kv16, s));
    else if (block_keys && (span_attention_ || few)) ESP_HIP_TRY(launch_span_attention(aa, rows, block_keys, kv16, s));
    else ESP_HIP_TRY(launch_attention(aa, rows, kv16, s));
    return ESP_OK;
}

// The layer loop over `rows` rows whose embeddings sit in hidden_ and whose (position, sequence) sit in
// d_pos_/d_seq_, every projection as one dequant-fused MFMA GEMM.  Rows that are one sequence at consecutive positions
// (a prompt block) take a matrix-core attention kernel, others the single-query one.
// Prompt blocks of Q4_K models: every projection with exact weights and split activations (launch_gemm_split), 32-bit attention: the block then stays as close to the fp32 CPU walk as the decode
// steps do.
bool LlamaRuntime::split_blocks_supported() const {
    return prompt_attention_ && c_.kv_format == FMT_F16 && splits_every_product();
}
// Blocks of fewer than 32 rows take the 32-bit attention kernel, whatever the head groups and the caches' format.
bool LlamaRuntime::short_split_blocks_supported() const { return short_span_attention_ && splits_every_product(); }
bool LlamaRuntime::splits_every_product() const {
    if (!split_activations_ || !xn_lo_ || c_.d_model > 8192) return false;
    for (const Layer &L : layers_)
        if (L.q_norm || !gemm_split_supported(L.wqkv) || !gemm_split_supported(L.wo) || !gemm_split_supported(L.w13) || !gemm_split_supported(L.w2)) return false;
    return true;
}

// Short blocks that carry activations, weights and attention as exactly as the single-row steps do pay from the fourth token on (8B: a block of 4..32
// tokens costs 3 steps per layer, 1B: 2.5).  Distance of the last hidden
// row from 64 bits, 5 / 13 / 24 / 31 tokens, 1B: blocks 8.3 / 5.8 / 4.6 / 4.0e-5, steps 8.4 / 6.2 / 4.9 / 4.9e-5; four layers of 8B: 2.37 / 2.16 / 2.01 / 1.85e-4 and
// 2.40 / 2.22 / 2.03 / 1.88e-4 (fp16 caches and contexts).
bool LlamaRuntime::block_prefill_pays(int count, int base) const {
    if (count >= kMatrixPrefillMinTokens) return true;
    if (count < 4 || !short_blocks_enabled()) return false;
    if (split_blocks_supported()) return true;   // whatever is behind them
    return count >= 5 && (short_split_blocks_supported() || short_blocks_exact()) && short_block_pays(count, base);
}

// A short block against the steps it replaces, microseconds per layer.  Its products take as long as two steps; its attention, one workgroup per query head and all keys in
// that workgroup's eight wavefronts, 0.135 (fp16 caches) or 0.36 ns (fp32) a key and dim.  A step takes its launches and its weights' way from memory, and its attention, whose
// workgroups share the keys, 0.8 ns a key and the keys' bytes at 2.9 TB/s.  So few tokens behind many keys stay steps: behind 8000 / 16000 keys, 5 tokens, steps -> block, four layers
// of 8B Q4_K with fp32 caches 1010 / 1340 -> 1930 / 3400 us, of 1B Q4_0 467 / 597 -> 525 / 785, where 31 tokens take 5200 / 7000 -> 1960 / 3460 and 2360 / 3000 -> 540 / 800.  Over 5 to 31
// tokens behind 16 to 16000 keys of fifteen models (six shapes, the four formats, both caches) the choice is 0.02 % off the faster one on average, 5.3 % at worst.
bool LlamaRuntime::short_block_pays(int count, int base) const {
    const Layer &L = layers_[0];
    const bool kv16 = c_.kv_format == FMT_F16;
    const float passes = (float)(steps_hold_two_rows() ? (count + 1) / 2 : count), keys = (float)(base + count);
    const float step = 22.0f + (float)(L.wqkv.bytes() + L.wo.bytes() + L.w13.bytes() + L.w2.bytes()) / 4.5e6f;
    const float step_key = 0.8e-3f + (float)(2 * c_.kv_dim() * (kv16 ? 2 : 4)) / 2.9e6f, block_key = (float)c_.head_dim * (kv16 ? 0.135e-3f : 0.36e-3f);
    return passes * (step + keys * step_key) >= 2.0f * step + keys * block_key;
}

// Q4_K models whose long blocks round (three query heads to a key/value head, fp32 caches): from the fifth token on; behind 100 tokens, 4 / 5 / 8 / 31 tokens, 3B 2225 / 3095 /
// 4272 / 16423 -> 2492 / 2474 / 2467 / 2319 us, four layers of 8B with fp32 caches 567 / 739 / 974 / 3327 -> 696 / 690 / 647 / 629.
// Blocks whose products keep every weight and whose attention is 32-bit round nothing that the single-row steps of these formats do not: activations and contexts are fp16 in
// both.  From the fifth token on they are also faster (behind 100 tokens, 4 / 5 / 16 / 31 tokens, steps -> block, us: 6 layers Q8_0 352 / 470 / 1316 / 2583 -> 337 / 324 / 350 / 366;
// 1.1B Q8_0 1430 / 2131 / 5436 / 11032 -> 1278 / 1259 / 1260 / 1358; 3B Q4_0 1966 / 2782 / 7341 / 14484 -> 2091 / 2061 / 2100 / 2159; two layers of 256 columns,
// 7 tokens 167 -> 93).
bool LlamaRuntime::short_blocks_exact() const {
    if (!short_span_attention_) return false;
    auto ok = [](const DeviceMatrix &m) {
        GemmParams p;
        p.w = m; p.rows = kMatrixPrefillMinTokens - 1; p.unrounded = true;
        return (m.format == FMT_Q8_0 || m.format == FMT_Q4_0 || m.format == FMT_F16) && (block_gemm_exact(m, p.rows) || rows_gemm_takes(p));
    };
    for (const Layer &L : layers_)
        if (!ok(L.wqkv) || !ok(L.wo) || !ok(L.w13) || !ok(L.w2)) return false;
    return true;
}

int LlamaRuntime::enqueue_layers_split(int rows, int block_keys, int last) {
    hipStream_t s = context().stream;
    const bool kv16 = c_.kv_format == FMT_F16;
    const int d = c_.d_model, ad = c_.attention_dim(), kd = c_.kv_dim();
    const size_t cache_seq_stride = (size_t)kd * c_.max_seq;
    SplitRowsView xn{xn_, xn_lo_, xn_sums_}, ctx{ctx_, ctx_lo_, ctx_sums_}, act{act_, act_lo_, act_sums_};
    // RMSNorm of hidden_ (or of the split-K planes a projection left, added to hidden_ first) into split rows
    auto norm = [&](const float *w, int splits) -> hipError_t {
        SplitRowsParams p;
        p.rows = rows; p.cols = d; p.norm_w = w; p.norm_eps = c_.norm_eps; p.out = xn;
        if (splits > 1) { p.x = gemm_workspace_; p.splits = splits; p.plane = (size_t)rows * d; p.residual = hidden_; p.y = hidden_; }
        else p.x = hidden_;
        return launch_split_rows(p, s);
    };
    ESP_HIP_TRY(norm(layers_.front().rms_att, 1));
    for (size_t li = 0; li < layers_.size(); li++) {
        Layer &L = layers_[li];
        GemmSplitParams g;
        g.rows = rows; g.workspace = gemm_workspace_; g.workspace_floats = gemm_workspace_floats_;
        int splits = 1;
        g.w = L.wqkv; g.x = xn; g.y = qkv_; g.deferred_splits = &splits;
        ESP_HIP_TRY(launch_gemm_split(g, s));
        QkvPostArgs qa{};
        qa.qkv = splits > 1 ? gemm_workspace_ : qkv_; qa.splits = splits; qa.plane = (size_t)rows * (ad + 2 * kd);
        qa.q_norm = nullptr; qa.k_norm = nullptr; qa.norm_eps = c_.norm_eps;
        qa.n_head = c_.n_head; qa.n_kv_head = c_.n_kv_head; qa.head_dim = c_.head_dim; qa.max_seq = c_.max_seq;
        qa.rope_cos = rope_cos_; qa.rope_sin = rope_sin_; qa.pos = d_pos_; qa.seq = d_seq_;
        qa.q_out = q_; qa.k_cache = L.k_cache; qa.v_cache = L.v_cache; qa.cache_seq_stride = cache_seq_stride;
        ESP_HIP_TRY(launch_qkv_post(qa, rows, kv16, s));
        AttentionArgs aa{};
        aa.q = q_; aa.k_cache = L.k_cache; aa.v_cache = L.v_cache; aa.cache_seq_stride = cache_seq_stride;
        aa.n_head = c_.n_head; aa.n_kv_head = c_.n_kv_head; aa.head_dim = c_.head_dim; aa.max_seq = c_.max_seq;
        aa.pos = d_pos_; aa.seq = d_seq_; aa.ctx_hi = ctx.hi; aa.ctx_lo = ctx.lo; aa.ctx_sums = ctx.sums;
        { int rc = enqueue_block_attention(aa, rows, block_keys, last); if (rc != ESP_OK) return rc; }
        g.w = L.wo; g.x = ctx; g.y = hidden_; g.residual = hidden_; splits = 1;
        ESP_HIP_TRY(launch_gemm_split(g, s));
        ESP_HIP_TRY(norm(L.rms_ffn, splits));
        g.w = L.w13; g.x = xn; g.y = nullptr; g.residual = nullptr; g.swiglu = act; g.deferred_splits = nullptr;
        g.shared_k = &gemm_shared_k_;
        ESP_HIP_TRY(launch_gemm_split(g, s));
        g.swiglu = SplitRowsView{}; g.shared_k = nullptr;
        const bool last = li + 1 == layers_.size();
        g.w = L.w2; g.x = act; g.y = hidden_; g.residual = hidden_; splits = 1; g.deferred_splits = last ? nullptr : &splits;
        ESP_HIP_TRY(launch_gemm_split(g, s));
        if (!last) ESP_HIP_TRY(norm(layers_[li + 1].rms_att, splits));
    }
    return ESP_OK;
}

// block_keys: the keys that the last row of a prompt block sees; 0 for rows that are not one sequence at consecutive positions.  last: rows at the end that are as in a block of their own (last_rows).
int LlamaRuntime::enqueue_layers_matrix(int rows, int block_keys, int last) {
    if (block_keys && (rows < kMatrixPrefillMinTokens ? short_split_blocks_supported() : split_blocks_supported())) return enqueue_layers_split(rows, block_keys, last);
    hipStream_t s = context().stream;
    const int d = c_.d_model, ad = c_.attention_dim(), kd = c_.kv_dim();
    const bool kv16 = c_.kv_format == FMT_F16;
    const size_t cache_seq_stride = (size_t)kd * c_.max_seq;
    GemmParams g;
    g.rows = rows; g.unrounded = true; g.workspace = gemm_workspace_; g.workspace_floats = gemm_workspace_floats_;
    // A product, in two launches where its last rows keep the weights and the others do not (each complete: no shares of K are left).  Prompts of 22 layers of
    // 1.1B Q8_0 and 30 of 576 columns in it, rounded like the others / in two launches / in a block of their own, us: 600 tokens 2990 / 3300 / 4250 and 2040 / 2260 / 3360, 520 2820 / 3550 / 3990 and
    // 1970 / 2070 / 3210.
    auto product = [&](bool gate_up) -> hipError_t {
        if (last == 0 || !rounds_but_for_last(g.w, last, gate_up)) return launch_gemm(g, s);
        GemmParams part = g;
        part.rows = rows - last;
        part.deferred_splits = nullptr;
        const hipError_t e = launch_gemm(part, s);
        if (e != hipSuccess) return e;
        const size_t at = (size_t)part.rows * g.w.rows;
        part.x += (size_t)part.rows * g.w.cols;
        part.y += at;
        if (part.residual) part.residual += at;
        if (part.swiglu_out) part.swiglu_out += at / 2;
        part.rows = last;
        return launch_gemm(part, s);
    };
    // The RMSNorm that follows a projection with a residual reads that projection's result; when the GEMM ran split-K the
    // norm kernel adds the partial sums itself (one launch instead of reduce + norm).
    const bool fuse_norm = rmsnorm_reduce_supported(d);
    auto project_and_norm = [&](const float *norm_w) -> int {   // g is set up for a GEMM into hidden_ with hidden_ as residual
        int splits = 1;
        g.deferred_splits = norm_w && fuse_norm ? &splits : nullptr;
        ESP_HIP_TRY(product(false));
        g.deferred_splits = nullptr;
        if (!norm_w) return ESP_OK;
        if (splits > 1) ESP_HIP_TRY(launch_rmsnorm_reduce(gemm_workspace_, splits, (size_t)rows * d, hidden_, hidden_, norm_w, c_.norm_eps, rows, d, xn_, s));
        else ESP_HIP_TRY(launch_rmsnorm(hidden_, norm_w, c_.norm_eps, rows, d, xn_, nullptr, s));
        return ESP_OK;
    };
    ESP_HIP_TRY(launch_rmsnorm(hidden_, layers_.front().rms_att, c_.norm_eps, rows, d, xn_, nullptr, s));
    for (size_t li = 0; li < layers_.size(); li++) {
        Layer &L = layers_[li];
        int qkv_splits = 1;   // split-K partial sums of q|k|v are added by the kernel that applies norm / RoPE and writes the caches
        g.w = L.wqkv; g.x = xn_; g.y = qkv_; g.residual = nullptr; g.deferred_splits = &qkv_splits;
        ESP_HIP_TRY(product(false));
        g.deferred_splits = nullptr;
        QkvPostArgs qa{};
        qa.qkv = qkv_splits > 1 ? gemm_workspace_ : qkv_; qa.splits = qkv_splits; qa.plane = (size_t)rows * (ad + 2 * kd);
        qa.q_norm = L.q_norm; qa.k_norm = L.k_norm; qa.norm_eps = c_.norm_eps;
        qa.n_head = c_.n_head; qa.n_kv_head = c_.n_kv_head; qa.head_dim = c_.head_dim; qa.max_seq = c_.max_seq;
        qa.rope_cos = rope_cos_; qa.rope_sin = rope_sin_; qa.pos = d_pos_; qa.seq = d_seq_;
        qa.q_out = q_; qa.k_cache = L.k_cache; qa.v_cache = L.v_cache; qa.cache_seq_stride = cache_seq_stride;
        ESP_HIP_TRY(launch_qkv_post(qa, rows, kv16, s));
        AttentionArgs aa{};
        aa.q = q_; aa.k_cache = L.k_cache; aa.v_cache = L.v_cache; aa.cache_seq_stride = cache_seq_stride;
        aa.n_head = c_.n_head; aa.n_kv_head = c_.n_kv_head; aa.head_dim = c_.head_dim; aa.max_seq = c_.max_seq;
        aa.pos = d_pos_; aa.seq = d_seq_; aa.ctx_f16 = ctx_; aa.split_scratch = attn_scratch_; aa.head_partials = attn_scratch_;
        { int rc = enqueue_block_attention(aa, rows, block_keys, last); if (rc != ESP_OK) return rc; }
        g.w = L.wo; g.x = ctx_; g.y = hidden_; g.residual = hidden_;
        { int rc = project_and_norm(L.rms_ffn); if (rc != ESP_OK) return rc; }
        g.w = L.w13; g.x = xn_; g.y = gu_; g.residual = nullptr; g.swiglu_out = act_;   // SwiGLU in the GEMM's epilogue where it can be
        ESP_HIP_TRY(product(true));
        g.swiglu_out = nullptr;
        g.w = L.w2; g.x = act_; g.y = hidden_; g.residual = hidden_;
        { int rc = project_and_norm(li + 1 < layers_.size() ? layers_[li + 1].rms_att : nullptr); if (rc != ESP_OK) return rc; }
    }
    (void)ad;
    return ESP_OK;
}

// Up to sixteen rows (a batch of sequences): every projection as one launch with its epilogue (launch_gemv, sixteen_rows).
bool LlamaRuntime::sixteen_rows_supported(int rows) const {
    for (const Layer &L : layers_)
        if (L.q_norm || !gemv_takes_sixteen_rows(L.wqkv, rows) || !gemv_takes_sixteen_rows(L.wo, rows) || !gemv_takes_sixteen_rows(L.w13, rows) || !gemv_takes_sixteen_rows(L.w2, rows))
            return false;
    return true;
}

int LlamaRuntime::enqueue_layers_sixteen(int rows) {
    hipStream_t s = context().stream;
    const int d = c_.d_model, kd = c_.kv_dim();
    const bool kv16 = c_.kv_format == FMT_F16;
    // the norm behind a projection with a residual, which may have left shares of K as planes
    auto norm = [&](const float *w, int splits) -> hipError_t {
        if (splits > 1) return launch_rmsnorm_reduce(gemm_workspace_, splits, (size_t)rows * d, hidden_, hidden_, w, c_.norm_eps, rows, d, xn_, s);
        return launch_rmsnorm(hidden_, w, c_.norm_eps, rows, d, xn_, nullptr, s);
    };
    const bool planes = rmsnorm_reduce_supported(d);
    ESP_HIP_TRY(norm(layers_.front().rms_att, 1));
    for (size_t li = 0; li < layers_.size(); li++) {
        Layer &L = layers_[li];
        int splits = 1;
        GemvParams g;
        g.batch = rows; g.sixteen_rows = true;
        g.w = L.wqkv; g.x = xn_; g.epilogue = EPI_QKV_ROPE;
        g.qkv.n_head = c_.n_head; g.qkv.n_kv_head = c_.n_kv_head; g.qkv.head_dim = c_.head_dim; g.qkv.max_seq = c_.max_seq;
        g.qkv.rope_cos = rope_cos_; g.qkv.rope_sin = rope_sin_; g.qkv.pos = d_pos_; g.qkv.seq = d_seq_;
        g.qkv.q_out = q_; g.qkv.k_cache = L.k_cache; g.qkv.v_cache = L.v_cache;
        g.qkv.cache_seq_stride = (size_t)kd * c_.max_seq; g.qkv.kv_f16 = kv16 ? 1 : 0;
        ESP_HIP_TRY(launch_gemv(g, s));
        AttentionArgs aa{};
        aa.q = q_; aa.k_cache = L.k_cache; aa.v_cache = L.v_cache; aa.cache_seq_stride = (size_t)kd * c_.max_seq;
        aa.n_head = c_.n_head; aa.n_kv_head = c_.n_kv_head; aa.head_dim = c_.head_dim; aa.max_seq = c_.max_seq;
        aa.pos = d_pos_; aa.seq = d_seq_; aa.ctx_f16 = ctx_; aa.split_scratch = attn_scratch_; aa.head_partials = attn_scratch_;
        ESP_HIP_TRY(launch_attention(aa, rows, kv16, s));
        g.w = L.wo; g.x = ctx_; g.y = hidden_; g.residual = hidden_; g.epilogue = EPI_ADD_RESIDUAL;
        g.workspace = planes ? gemm_workspace_ : nullptr; g.workspace_floats = gemm_workspace_floats_; g.deferred_splits = planes ? &splits : nullptr;
        ESP_HIP_TRY(launch_gemv(g, s));
        ESP_HIP_TRY(norm(L.rms_ffn, splits));
        g.w = L.w13; g.x = xn_; g.y = nullptr; g.residual = nullptr; g.out_f16 = act_; g.epilogue = EPI_SWIGLU_F16;
        ESP_HIP_TRY(launch_gemv(g, s));
        g.w = L.w2; g.x = act_; g.out_f16 = nullptr; g.y = hidden_; g.residual = hidden_; g.epilogue = EPI_ADD_RESIDUAL;
        splits = 1;
        ESP_HIP_TRY(launch_gemv(g, s));
        const bool last = li + 1 == layers_.size();   // (behind the last layer only for the sum: the head norms its rows itself)
        if (!last || splits > 1) ESP_HIP_TRY(norm(last ? final_norm_ : layers_[li + 1].rms_att, splits));
    }
    return ESP_OK;
}

// The head of one or two rows with its arg-max inside: final RMSNorm in the staging, one candidate per row and workgroup, no logits are written (:8219-8275).
int LlamaRuntime::run_head_candidates(const float *hidden_rows, int count, int *blocks) {
    hipStream_t s = context().stream;
    GemvParams g;
    g.w = lm_head_; g.norm_x = hidden_rows; g.norm_w = final_norm_; g.norm_eps = c_.norm_eps; g.batch = count; g.epilogue = EPI_ARGMAX;
    g.argmax_value = argmax_scratch_.part_value; g.argmax_index = argmax_scratch_.part_index; g.argmax_capacity = head_partial_capacity_;
    g.argmax_blocks = blocks;
    int rc;
    if ((rc = time_begin(K_HEAD)) != ESP_OK) return rc;
    ESP_HIP_TRY(launch_gemv(g, s));
    return time_end();
}

int LlamaRuntime::enqueue_device_head_candidates(HeadTokens *head) {
    *head = HeadTokens{};
    head->tokens = d_out_tokens_;
    if (!head_fuses_argmax()) return run_head(hidden_, 2);
    head->part_value = argmax_scratch_.part_value;
    head->part_index = argmax_scratch_.part_index;
    return run_head_candidates(hidden_, 2, &head->blocks);
}

// More than two rows: one product, unless the weights are 32-bit or the caller keeps prompts from blocks.
bool LlamaRuntime::head_in_one_product(int count) const { return count > 2 && matrix_prefill_ && lm_head_.format != FMT_F32 && lm_head_.cols % 64 == 0; }

GemmParams LlamaRuntime::head_product(int count) const {
    GemmParams m;
    m.w = lm_head_; m.x = xn_; m.y = logits_; m.rows = count; m.unrounded = true; m.workspace = gemm_workspace_; m.workspace_floats = gemm_workspace_floats_;
    return m;
}

// Normed rows are fp16 and sums 32-bit either way, and so are weights as they are, but for products that round them to fp16: heads of 49152 x 576 (Q8_0, Q4_0) from three rows on, Q4_K ones from nine rows on
// where neither launch for sixteen rows knows their width.
bool LlamaRuntime::head_is_as_exact_for_rows(int count) const {
    return !head_in_one_product(count) || gemv_takes_sixteen_rows(lm_head_, count) || gemm_keeps_weights(head_product(count));
}

int LlamaRuntime::run_head(const float *hidden_rows, int count, bool want_logits) {
    hipStream_t s = context().stream;
    if (count <= 2 && !want_logits && head_fuses_argmax()) {
        int blocks = 0, rc;
        if ((rc = run_head_candidates(hidden_rows, count, &blocks)) != ESP_OK) return rc;
        ESP_HIP_TRY(launch_argmax_final(argmax_scratch_, blocks, count, d_out_tokens_, s));
        return ESP_OK;
    }
    if (head_in_one_product(count)) {
        // batched rows: final RMSNorm, then the head as one MFMA GEMM
        ESP_HIP_TRY(launch_rmsnorm(hidden_rows, final_norm_, c_.norm_eps, count, c_.d_model, xn_, nullptr, s));
        if (gemv_takes_sixteen_rows(lm_head_, count)) {
            GemvParams g;
            g.w = lm_head_; g.x = xn_; g.y = logits_; g.batch = count; g.sixteen_rows = true; g.epilogue = EPI_STORE_F32;
            ESP_HIP_TRY(launch_gemv(g, s));
            ESP_HIP_TRY(launch_argmax(logits_, count, c_.vocab, d_out_tokens_, nullptr, argmax_scratch_, s));
            return ESP_OK;
        }
        ESP_HIP_TRY(launch_gemm(head_product(count), s));
        ESP_HIP_TRY(launch_argmax(logits_, count, c_.vocab, d_out_tokens_, nullptr, argmax_scratch_, s));
        return ESP_OK;
    }
    GemvParams g;   // final RMSNorm fused into the head GEMV's staging
    g.w = lm_head_; g.norm_x = hidden_rows; g.norm_w = final_norm_; g.norm_eps = c_.norm_eps;
    g.y = logits_; g.batch = count; g.epilogue = EPI_STORE_F32;
    int rc;
    if ((rc = time_begin(K_HEAD)) != ESP_OK) return rc;
    ESP_HIP_TRY(launch_gemv(g, s));
    if ((rc = time_end()) != ESP_OK) return rc;
    ESP_HIP_TRY(launch_argmax(logits_, count, c_.vocab, d_out_tokens_, nullptr, argmax_scratch_, s));
    return ESP_OK;
}

// Head GEMV with the arg-max in its epilogue, then one launch that picks the token among the workgroups' candidates, feeds it and
// fetches its embedding; the last layer writes the new hidden state where the next step's head reads it: 2 + 5 per layer launches
// (3 + 5 per layer when the head has to store its logits).
int LlamaRuntime::enqueue_greedy_token(int seq) {
    hipStream_t s = context().stream;
    GemvParams g;
    g.w = lm_head_; g.norm_x = device_last_hidden(seq); g.norm_w = final_norm_; g.norm_eps = c_.norm_eps; g.batch = 1;
    hipError_t e;
    if (head_fuses_argmax()) {
        int blocks = 0;
        g.epilogue = EPI_ARGMAX;
        g.argmax_value = argmax_scratch_.part_value; g.argmax_index = argmax_scratch_.part_index; g.argmax_capacity = head_partial_capacity_;
        g.argmax_blocks = &blocks;
        e = launch_gemv(g, s);
        if (e == hipSuccess)
            e = launch_greedy_tail(argmax_scratch_, blocks, d_out_tokens_, seq, d_visible_, d_tokens_, d_pos_, d_seq_, d_log_, d_log_count_,
                                   c_.max_seq, embedding_, embedding_f16_, c_.d_model, hidden_, c_.eos_token, s);
    } else {
        g.y = logits_; g.epilogue = EPI_STORE_F32;
        e = launch_gemv(g, s);
        if (e == hipSuccess)
            e = launch_greedy_step_tail(logits_, c_.vocab, d_out_tokens_, argmax_scratch_, seq, d_visible_, d_tokens_, d_pos_, d_seq_, d_log_,
                                        d_log_count_, c_.max_seq, embedding_, embedding_f16_, c_.d_model, hidden_, c_.eos_token, s);
    }
    return e == hipSuccess ? ESP_OK : fail_hip(e, "greedy step head");
}

}  // namespace esp
