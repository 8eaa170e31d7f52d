// Causal attention of the rows of a prompt block for any number of query heads per key/value head (kernels/span_attention.hip).
#pragma once

#include "decode_ops.h"

namespace esp {

bool span_attention_supported(int n_head, int n_kv_head, int head_dim);
// `rows` rows that are one sequence at consecutive positions, the last of which sees `keys` keys; writes ctx_f16, or split rows where ctx_hi is given.
hipError_t launch_span_attention(const AttentionArgs &a, int rows, int keys, bool kv_f16, hipStream_t s);

}  // namespace esp
