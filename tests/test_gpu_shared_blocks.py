"""Prompts of several sequences that share blocks of rows, against the same prompts one after the other: models of split rows, of fp16 and of packed matrices, prompts below and above the 32 rows that
decide the attention kernel, prompts that take steps, more rows than one block holds."""
import numpy as np
import pytest

import espresso_amd._lib as lib

pytestmark = pytest.mark.gpu

SHAPES = {
    "split rows": (lib.FORMAT_Q4_K, lib.FORMAT_F16, dict(n_head=8, n_kv_head=2, d_model=512, head_dim=64, hidden_dim=768)),
    "split rows, short ones alone": (lib.FORMAT_Q4_K, lib.FORMAT_F16, dict(n_head=12, n_kv_head=4, d_model=1536, head_dim=128, hidden_dim=1024)),
    "fp16": (lib.FORMAT_F16, lib.FORMAT_F32, dict(n_head=9, n_kv_head=3, d_model=576, head_dim=64, hidden_dim=1536)),
    "fp16, heads of 32": (lib.FORMAT_F16, lib.FORMAT_F16, dict(n_head=8, n_kv_head=8, d_model=256, head_dim=32, hidden_dim=512)),
    "packed": (lib.FORMAT_Q8_0, lib.FORMAT_F16, dict(n_head=8, n_kv_head=4, d_model=1024, head_dim=128, hidden_dim=4096)),
    "packed, shared from 129 rows": (lib.FORMAT_Q8_0, lib.FORMAT_F16, dict(n_head=16, n_kv_head=16, d_model=2048, head_dim=128, hidden_dim=5632)),
}
LENGTHS = [(40, 37, 32, 31, 5, 3, 1), (200, 7, 129, 64, 6), (150, 300, 290, 280, 270, 33), (33, 34)]


@pytest.mark.parametrize("name", SHAPES)
@pytest.mark.parametrize("lengths", LENGTHS)
def test_shared_blocks_are_the_prompts_alone(name, lengths):
    import espresso_amd.llama as ll
    import espresso_amd.ops as o
    import espresso_amd.synthetic as syn
    o.init()
    fmt, kv, shape = SHAPES[name]
    cfg = ll.MultiModelConfig(n_layer=2, vocab=260, max_seq=320, **shape)
    alone, _ = syn.build_runtime(cfg, fmt, seed=3, std=0.05, kv_format=kv, max_sequences=len(lengths))
    both, _ = syn.build_runtime(cfg, fmt, seed=3, std=0.05, kv_format=kv, max_sequences=len(lengths))
    rng = np.random.default_rng(len(lengths))
    prompts = [rng.integers(0, 260, n).astype(np.uint32) for n in lengths]
    ll.generate_batch(both, prompts, 1)      # one token: chosen from the prompt's last row, none is walked
    for s, p in enumerate(prompts):
        alone.prefill(p, sequence=s)
    for s, p in enumerate(prompts):
        assert both.visible(sequence=s) == alone.visible(sequence=s) == len(p)
        a, b = alone.last_hidden(sequence=s), both.last_hidden(sequence=s)
        # the caches and contexts are fp16 where they are in both, and a last bit of them may fall either way
        assert np.sqrt(np.mean((a - b) ** 2)) <= 2.0 ** -10 * np.sqrt(np.mean(a ** 2)), (s, len(p))
        # what the caches hold: the next token's logits behind them
        x, y = alone.append(p[:1], want=[0], sequence=s)[0], both.append(p[:1], want=[0], sequence=s)[0]
        assert np.sqrt(np.mean((x - y) ** 2)) <= 2.0 ** -10 * np.sqrt(np.mean(x ** 2)), (s, len(p))
    alone.close()
    both.close()


def test_a_prompt_that_is_refused_is_refused():
    import espresso_amd.llama as ll
    import espresso_amd.ops as o
    import espresso_amd.synthetic as syn
    o.init()
    rt, _ = syn.build_runtime(ll.MultiModelConfig(n_layer=1, vocab=260, max_seq=64, n_head=8, n_kv_head=2, d_model=512, head_dim=64, hidden_dim=768), lib.FORMAT_Q4_K, seed=3, std=0.05,
                              kv_format=lib.FORMAT_F16, max_sequences=3)
    good = np.arange(40, dtype=np.uint32)
    with pytest.raises(Exception, match="outside vocab"):
        ll.generate_batch(rt, [good, np.array([1, 260], np.uint32), good], 4)
    assert rt.visible(sequence=0) == 40
    rt.close()


def test_a_block_that_fails_leaves_no_tokens():
    """A form whose shares of K do not fit the workspace is refused on the host, before any launch of the products: the sequences of that block are empty then, not as long as before."""
    import espresso_amd.llama as ll
    import espresso_amd.ops as o
    import espresso_amd.synthetic as syn
    o.init()
    fmt, kv, shape = SHAPES["packed, shared from 129 rows"]
    rt, _ = syn.build_runtime(ll.MultiModelConfig(n_layer=1, vocab=260, max_seq=320, **shape), fmt, seed=3, std=0.05, kv_format=kv, max_sequences=3)
    prompts = [np.arange(n, dtype=np.uint32) for n in (150, 160, 170)]
    ll.generate_batch(rt, prompts, 4)
    assert [rt.visible(sequence=s) > 149 for s in range(3)] == [True] * 3
    try:
        o.set_tuning("block_gemm_form", 148)   # eight shares of 320 x 6144 sums
        with pytest.raises(Exception, match="invalid argument"):
            ll.generate_batch(rt, prompts[:2], 4)
    finally:
        o.set_tuning("block_gemm_form", 0)
    assert [rt.visible(sequence=s) for s in (0, 1)] == [0, 0] and rt.visible(sequence=2) > 149
    ll.generate_batch(rt, prompts, 1)
    assert [rt.visible(sequence=s) for s in range(3)] == [150, 160, 170]
    rt.close()
