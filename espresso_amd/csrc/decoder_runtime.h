// What every device-resident decoder shares, whatever its layers are: sequence slots and their visible lengths, the rows of a
// step, kept hidden states, the output head's token selection, prompts in blocks and portions, greedy steps as captured graphs.
// LlamaRuntime (llama_runtime.h) and LayeredRuntime (layered_runtime.h) supply the layers; the generation loops (generation.h),
// the engine (host/engine.h) and the C ABI drive this class.
#pragma once

#include <string>
#include <vector>

#include "context.h"
#include "kernels/decode_ops.h"

namespace esp {

class LlamaRuntime;
class LayeredRuntime;

// Rows of a prompt block: a whole prompt of up to 2048 tokens, so that its products have several rounds of workgroups (blocks of 512 -> one block, us: 1777 tokens of 3B Q4_K 20960 ->
// 16200, 1500 of eight layers of 8B 12580 -> 12150, 1100 of 1B Q8_0 6510 -> 4440, 1777 of 1.1B Q8_0 10930 -> 7160, 1700 of 30 layers of 576 columns in Q4_0 7250 -> 3570, 1700 of six Ranavik layers of
// 4096 columns 8150 -> 6230; as exact as blocks of 512: LlamaRuntime::last_rows, kExactRows); contexts that hold fewer take what they hold, and no runtime's blocks are shorter than 512.
constexpr int kMinPrefillBlockRows = 512, kMaxPrefillBlockRows = 2048;
inline int prefill_block_rows(int max_seq) {
    const int rows = max_seq > kMaxPrefillBlockRows ? kMaxPrefillBlockRows : (max_seq + 127) / 128 * 128;
    return rows < kMinPrefillBlockRows ? kMinPrefillBlockRows : rows;
}
constexpr int kStepsPerGraph = 8;             // greedy steps in the longer of the two captured step graphs
constexpr int kMatrixPrefillMinTokens = 32;   // shorter prompts take the steps' kernels, two tokens at a time where a step takes two rows, unless the runtime's short blocks are as exact
constexpr size_t kGemmWorkspaceFloatsPerRow = (size_t)16 << 10;   // planes of split-K products, per row of a block

struct DecoderShape {
    int d_model = 0, vocab = 0, max_seq = 0;
    int eos_token = -1;
    int max_sequences = 1;    // independent sequence slots (KV caches, recurrent states)
};

struct LastRows { int own_block = 0, in_block = 0; };
struct PromptSpan { int sequence; const uint32_t *tokens; int count; };   // a whole prompt of an empty sequence

class DecoderRuntime {
  public:
    virtual ~DecoderRuntime();
    virtual const DecoderShape &shape() const = 0;
    virtual LlamaRuntime *as_llama() { return nullptr; }
    virtual LayeredRuntime *as_layered() { return nullptr; }

    bool finalized() const { return finalized_; }
    int reset();                                  // all sequences (RealModelInferenceEngine.swift:616-635)
    int visible(int seq) const;
    // Rollback = lower the visible length.  Runtimes with recurrent state (can_roll_back() false) take only 0 and the length
    // the sequence has.
    int set_visible(int seq, int count);
    // A generation loop has run `count` more tokens of the sequence through its own rows (forward_rows, enqueue_device_rows), so the caches
    // and states hold them: recurrent runtimes included, whose visible length set_visible() does not raise.
    void add_consumed(int seq, int count) { visible_[seq] += count; }
    virtual bool can_roll_back() const { return true; }
    // whether one step may hold several rows of one sequence (draft verification)
    virtual bool takes_rows_of_one_sequence() const { return true; }
    // whether the step's kernels hold two rows of every matrix at once
    virtual bool steps_hold_two_rows() const { return true; }
    // Sequence slots for callers with requests that come and go: the lowest free slot, and its return.  A slot that is taken
    // again starts as an empty sequence.
    int acquire_sequence(int *seq);
    int release_sequence(int seq);

    // Runs the trunk over `rows` (token, position, sequence); positions are written into the caches.
    // Does not change the visible counts.
    int forward_rows(const StepRows &rows);
    // forward one token at the sequence's visible position and keep its hidden state (:672-680)
    int advance(int seq, uint32_t token);
    int prefill(int seq, const uint32_t *tokens, int count);   // from an empty sequence (:637-645)
    // Prompts of the sequences 0 .. count - 1, all empty; those that may share a block of rows do, so that the weights are read once for them.
    int prefill_batch(const uint32_t *const *prompts, const int *counts, int count);
    // The next `count` tokens of a sequence, from the caches and state that its earlier tokens left.  `want` lists (ascending)
    // the places among them whose logits go to `logits` ([want_count][vocab]).
    int append(int seq, const uint32_t *tokens, int count, const int *want = nullptr, int want_count = 0, float *logits = nullptr);
    // Final norm + LM head + first-max argmax of kept hidden states (:663-670, :825-849).
    int select_greedy(int seq, uint32_t *token);
    // The same for the sequences 0 .. count - 1, with the head read once for all of them where that is as exact.
    int select_greedy_rows(int count, uint32_t *tokens);
    // Head over rows of the most recent forward_rows(); tokens[i] for row i.
    int head_rows(int count, uint32_t *tokens);
    // Keep row `row` of the most recent forward_rows() as sequence `seq`'s last hidden state.
    int keep_row(int row, int seq);
    // `steps` greedy tokens from the sequence's current state (select, then advance, per token) as
    // replays of captured HIP graphs (eight steps per graph while that many are left, then one); the host synchronises once at the end.
    int continue_greedy(int seq, int steps, uint32_t *out_tokens);
    // The same, ending early at the configuration's stop token: the stop token is emitted (it is the last of *produced tokens) and not
    // consumed.  The step graph notices it on the device; the host looks once per 32 replays.
    int continue_greedy_until_stop(int seq, int steps, uint32_t *out_tokens, int *produced);
    void set_use_graph(bool enabled) { use_graph_ = enabled; }
    // Prompts for which block_prefill_pays() run in blocks through the MFMA kernels, others two tokens per step (default on;
    // off: one token per step, whatever the prompt's length).
    void set_matrix_prefill(bool enabled) { matrix_prefill_ = enabled; }
    int read_last_hidden(int seq, float *out);
    int read_logits(int seq, float *out);         // runs the head on the kept hidden state
    // the residual stream of rows of the most recent block or step (measurement and tests)
    int read_hidden_rows(int rows, float *out);

    virtual size_t weight_bytes_per_token() const = 0;
    // what the weights hold in HBM: the packed matrices, the tiled copies the matrix-core GEMVs read beside them, the embedding table
    virtual size_t resident_weight_bytes() const = 0;

    // Steps whose rows (token, position, sequence) already sit in the device arrays below: generation loops that keep
    // their decisions on the device enqueue these, also under stream capture.  Nothing here synchronises.
    int *device_row_tokens() { return d_tokens_; }
    int *device_row_positions() { return d_pos_; }
    int *device_row_sequences() { return d_seq_; }
    const int *device_head_tokens() const { return d_out_tokens_; }
    const float *device_hidden_rows() const { return hidden_; }
    float *device_last_hidden(int seq) { return last_hidden_ + (size_t)seq * hidden_stride_; }
    int enqueue_device_rows(int rows, bool embedded = false) { return enqueue_trunk(rows, embedded); }   // embedding (unless the rows hold it already), then every layer
    int enqueue_device_head(int rows) { return run_head(hidden_, rows); }         // final norm, head, first-max arg-max per row
    bool graph_replay_enabled() const { return use_graph_ && !timing_enabled_; }
    unsigned long long id() const { return id_; }
    // changes whenever the kernels a captured graph would hold have changed (switches of this runtime, esp_set_tuning): holders
    // of captured passes compare it before they replay
    unsigned long long graph_epoch() { sync_tuning(); return graph_epoch_; }

    // Per-kernel timing with HIP events on the library stream.  While enabled, every launch of the
    // kernels of a class is bracketed by an event pair; collect_kernel_times() synchronises and adds the
    // elapsed times to the totals.  The classes are the runtime's own.
    static constexpr int kMaxKernelClasses = 16;
    void set_kernel_timing(bool enabled) { timing_enabled_ = enabled; }
    int collect_kernel_times(double *total_us, long *launches, int classes, bool reset);

  protected:
    DecoderRuntime();
    // ---- what the layers supply ----
    // embedded: hidden_ already holds the rows' embeddings; final_out: where the last layer writes (default hidden_)
    virtual int enqueue_trunk(int rows, bool embedded = false, float *final_out = nullptr) = 0;
    // want_logits: the full-vocabulary logits are needed in logits_ (otherwise the head may store none)
    virtual int run_head(const float *hidden_rows, int count, bool want_logits = false) = 0;
    int select_rows(const float *hidden_rows, int count, uint32_t *tokens);   // run_head and its tokens
    // Does run_head round no more for `count` rows than for a single one?
    virtual bool head_is_as_exact_for_rows(int) const { return false; }
    // One greedy choice under capture: head over the sequence's kept state, the token into row 0 and the log, and what
    // enqueue_trunk(1, true) needs of its embedding.
    virtual int enqueue_greedy_token(int seq) = 0;
    // `rows` tokens at positions base.. of one sequence as one block, the last of them by last_rows; their rows end in hidden_.
    virtual int prefill_block(int seq, const uint32_t *tokens, int rows, int base, int last) = 0;
    virtual bool matrix_prefill_supported() const = 0;
    // Prompts of one class other than 0 may share a block and come out as in blocks of their own, but for the order of sums.
    virtual int shared_block_class(int count) const { (void)count; return 0; }
    // Prompts of a class, their rows behind each other (up to block_rows_), as one block; the rows end in hidden_.
    virtual int prefill_shared_block(const PromptSpan *spans, int count) { (void)spans; (void)count; return ESP_ERR_UNSUPPORTED; }
    // The last rows of `count` that a block of so few would compute more exactly than a long one: they go in such a block, or at the end of a long one whose kernels are others for them.  Fewer than
    // kMinPrefillBlockRows, and fewer than `count`.
    virtual LastRows last_rows(int count) const { (void)count; return {}; }
    // Whether `count` tokens behind `base` run in blocks rather than in steps (where the layers take blocks at all).
    virtual bool block_prefill_pays(int count, int base) const { (void)base; return count >= kMatrixPrefillMinTokens; }
    virtual int clear_state() = 0;                       // every cache and state of every sequence, enqueued on the stream
    virtual unsigned tuning_epoch() const { return 0; }

    // The buffers this class owns, for `block_rows` rows per block and hidden rows of `hidden_stride` floats.
    int allocate_common(int block_rows, int hidden_stride);
    int finish_finalize() { finalized_ = true; return reset(); }
    void drop_captured_graphs();
    void sync_tuning();
    int capture_step_graph(int seq);
    int capture_steps(int seq, int count, hipGraphExec_t *out);
    int replay_steps(int seq, int steps);
    int upload_block_rows(const PromptSpan *spans, int count, int base);
    int check_sequence(int seq) const;

    bool finalized_ = false;
    int hidden_stride_ = 0, block_rows_ = 0;
    float *hidden_ = nullptr, *logits_ = nullptr, *last_hidden_ = nullptr, *want_rows_ = nullptr;
    int *d_tokens_ = nullptr, *d_pos_ = nullptr, *d_seq_ = nullptr, *d_out_tokens_ = nullptr;
    std::vector<int> visible_;
    std::vector<char> taken_;
    // captured greedy step per sequence (head -> feed -> trunk -> keep), and its device-side state
    bool use_graph_ = true;
    std::vector<hipGraphExec_t> step_graphs_, multi_graphs_;   // one step, kStepsPerGraph steps
    unsigned long long id_ = 0, graph_epoch_ = 1;
    unsigned tuning_epoch_ = 0;   // the kernel-selection epoch this runtime's captured graphs were made under
    int *d_visible_ = nullptr, *d_log_ = nullptr, *d_log_count_ = nullptr;
    ArgmaxScratch argmax_scratch_;
    int head_partial_capacity_ = 0;      // (value, index) slots per row for the head's per-workgroup candidates
    bool matrix_prefill_ = true;
    bool capturing_ = false;             // enqueue_trunk is being captured into a sequence's step graph (replays may follow its stop token)

    struct TimedLaunch { int kernel_class; hipEvent_t start, stop; };
    bool timing_enabled_ = false;
    std::vector<TimedLaunch> timed_;        // pending pairs
    std::vector<hipEvent_t> event_pool_;
    double time_total_us_[kMaxKernelClasses] = {};
    long time_launches_[kMaxKernelClasses] = {};
    hipEvent_t take_event();
    int time_begin(int kernel_class);
    int time_end();
};

template <typename T>
void free_device(T *&p) {
    if (p) (void)hipFree(p);
    p = nullptr;
}

}  // namespace esp

// handle behind the runtime entry points of the C ABI, whatever the architecture
struct ESPLlamaRuntime {
    esp::DecoderRuntime *rt;
};
