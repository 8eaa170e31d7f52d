"""batch_gemv_kernel (steps of a batch with Q4_K matrices): every number of row blocks and shares of K against the same sequences one at a time, rows that fill no block, widths of one to sixteen
super-blocks and more."""
import numpy as np
import pytest

import espresso_amd._lib as lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,kv", [
    (dict(n_head=16, n_kv_head=4, d_model=1024, head_dim=64, hidden_dim=2048, vocab=515), lib.FORMAT_F16),
    (dict(n_head=8, n_kv_head=8, d_model=1024, head_dim=128, hidden_dim=8192, vocab=260), lib.FORMAT_F32),
    (dict(n_head=24, n_kv_head=8, d_model=3072, head_dim=128, hidden_dim=3072, vocab=1001), lib.FORMAT_F16),
])
def test_batches_are_their_sequences(shape, kv):
    import espresso_amd.llama as ll
    import espresso_amd.ops as o
    import espresso_amd.synthetic as syn
    o.init()
    cfg = ll.MultiModelConfig(n_layer=2, max_seq=64, **shape)
    rng = np.random.default_rng(cfg.d_model)
    prompts = [rng.integers(0, cfg.vocab, n).astype(np.uint32) for n in (7, 40, 9, 33, 5, 12, 8, 6, 35, 11, 10, 7, 6, 5, 9, 8)]
    rt, _ = syn.build_runtime(cfg, lib.FORMAT_Q4_K, seed=5, std=0.05, kv_format=kv, max_sequences=16)
    one, _ = syn.build_runtime(cfg, lib.FORMAT_Q4_K, seed=5, std=0.05, kv_format=kv)
    try:
        for count, form in [(16, 0), (3, 0), (5, 0)] + [(16 if blocks % 2 else 11, 10 * blocks + shares) for blocks in range(1, 9) for shares in (1, 2, 4, 8)]:
            o.set_tuning("batch_gemv_form", form)
            rt.reset()
            out, _ = ll.generate_batch(rt, prompts[:count], 4)
            for s in (0, count - 1):      # the same tokens one sequence at a time
                one.reset()
                one.prefill(prompts[s])
                for t in out[s][:-1]:
                    one.advance(int(t))
                one_next = one.append(np.array(out[s][-1:], np.uint32), want=[0])[0]
                rt.set_visible(len(prompts[s]) + len(out[s]) - 1, sequence=s)
                b = rt.append(np.array(out[s][-1:], np.uint32), want=[0], sequence=s)[0]
                # activations are fp16 in the batch and pairs of fp16 in single steps: 2e-4 to 6e-4 of the logits' size, an order below what a wrong row or super-block makes
                assert np.sqrt(np.mean((one_next - b) ** 2)) <= 2e-3 * np.sqrt(np.mean(one_next ** 2)), (count, form, s)
    finally:
        o.set_tuning("batch_gemv_form", 0)
        rt.close()
        one.close()
