// Causal attention of the rows of a prompt block for any number of query heads per key/value head (kernels/span_attention.hip).
#pragma once

#include "decode_ops.h"

namespace esp {

bool span_attention_supported(int n_head, int n_kv_head, int head_dim);
// `rows` rows that are one sequence at consecutive positions, the last of which sees `keys` keys; writes ctx_f16, or split rows where ctx_hi is given.
// pairs_do: fp16 caches may meet pairs of fp16 parts where that is faster and only ctx_f16 is written.
hipError_t launch_span_attention(const AttentionArgs &a, int rows, int keys, bool kv_f16, hipStream_t s, bool pairs_do = false);
// The same for head groups that attention_prompt_supported() knows, whose rows are a prompt's: 32-bit caches may round their operands to fp16 there.
inline hipError_t launch_prompt_attention(const AttentionArgs &a, int rows, int keys, bool kv_f16, hipStream_t s) {
    if (!attention_prompt_supported(a.n_head, a.n_kv_head, a.head_dim)) return hipErrorInvalidValue;
    return kv_f16 ? launch_span_attention(a, rows, keys, true, s, true) : launch_attention_prompt(a, rows, s);
}
void attention_prompt_set_key_sets(int sets);   // fp16 caches: 0 = wavefronts of a workgroup by size (default), 1 or 2 = always four or eight

}  // namespace esp
