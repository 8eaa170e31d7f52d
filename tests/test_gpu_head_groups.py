"""Head groups other than one, two and four query heads per key/value head: prompt blocks through span_attention_kernel (tiles of 32 rows
and 32 keys, one to eight wavefronts per tile, a second block behind a full one) and batches of several rows through the single-row kernel
with a merge launch, against the oracle's walk token by token; fp16 and fp32 caches."""
import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_full_size import oracle_from_packed

pytestmark = pytest.mark.gpu


def build(head_dim, n_head, n_kv, kv_fp16, max_seq, sequences=1):
    import espresso_amd.llama as ll
    import espresso_amd.ops as ops
    import espresso_amd.synthetic as syn
    ops.init()
    cfg = ll.MultiModelConfig(n_layer=2, n_head=n_head, n_kv_head=n_kv, d_model=n_head * head_dim, head_dim=head_dim, hidden_dim=512, vocab=512, max_seq=max_seq)
    g, packed = syn.build_runtime(cfg, orc.FMT_F16, seed=head_dim + n_head, std=0.05, keep_packed=True, max_sequences=sequences,
                                  kv_format=orc.FMT_F16 if kv_fp16 else orc.FMT_F32)
    return cfg, g, lambda: oracle_from_packed(cfg, packed, orc.FMT_F16, 2, kv_fp16, max_seq)


@pytest.mark.parametrize("head_dim,n_head,n_kv,kv_fp16,prompt_len,max_seq", [
    (128, 3, 1, True, 32, 64), (128, 6, 2, False, 33, 64), (128, 6, 2, True, 97, 128), (128, 3, 1, False, 130, 256), (128, 6, 1, True, 300, 512),
    (64, 8, 1, True, 45, 256), (64, 9, 3, False, 77, 128), (64, 5, 1, True, 256, 300), (64, 8, 1, False, 289, 512), (64, 3, 1, True, 520, 600),
])
def test_prompt_block_matches_oracle(head_dim, n_head, n_kv, kv_fp16, prompt_len, max_seq):
    cfg, g, oracle = build(head_dim, n_head, n_kv, kv_fp16, max_seq)
    prompt = np.random.default_rng(prompt_len).integers(0, cfg.vocab, prompt_len)
    o = oracle()
    o.prefill([int(t) for t in prompt])
    g.prefill(prompt)
    # fp16 activations into every product on both sides; the attention's own error (fp32 sums) is far below their rounding
    for _ in range(2):
        ho, hg = o.last_hidden(), g.last_hidden()
        assert np.abs(ho - hg).max() <= 2e-3 * max(1.0, np.abs(ho).max())
        assert np.abs(o.logits() - g.logits()).max() <= 2e-2
        o.advance(5)
        g.advance(5)
    g.close()


@pytest.mark.parametrize("head_dim,n_head,n_kv,kv_fp16", [(64, 8, 1, True), (64, 9, 3, False), (128, 3, 1, True)])
def test_batch_of_sequences_matches_oracle(head_dim, n_head, n_kv, kv_fp16):
    import espresso_amd.llama as ll
    cfg, g, oracle = build(head_dim, n_head, n_kv, kv_fp16, 256, sequences=5)
    prompts = [np.random.default_rng(n).integers(0, cfg.vocab, n).astype(np.uint32) for n in (1, 7, 40, 90, 3)]
    got, _ = ll.generate_batch(g, prompts, 6)
    for s, p in enumerate(prompts):
        o = oracle()
        o.prefill([int(t) for t in p])
        for t in got[s]:   # a near tie may fall either way: the chosen token's logit is what has to match
            logits = o.logits()
            assert logits.max() - logits[t] <= 2e-2
            o.advance(t)
    g.close()
