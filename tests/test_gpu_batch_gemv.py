"""batch_gemv_kernel (steps of a batch with Q4_K matrices): every number of row blocks and shares of K against the same sequences one at a time, rows that fill no block, widths of one to sixteen
super-blocks and more."""
import numpy as np
import pytest

import espresso_amd._lib as lib
from test_gpu_block_gemm import check_kept, rms_off

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


@pytest.mark.parametrize("rows,cols", [(515, 1024), (40, 2048), (272, 3072), (129, 4096), (96, 8192), (48, 14336)])
def test_step_products_keep_their_weights(rows, cols):
    """The product by itself against 64 bits, every number of row blocks and shares of K: no weight is rounded (fp16 ones would be 2e-4 off), rows that fill no block and no workgroup."""
    import espresso_amd.ops as o
    o.init()
    m = o.Matrix(lib.FORMAT_Q4_K, o.synth_weights(lib.FORMAT_Q4_K, rows + cols, 0.02, rows * cols), rows, cols)
    rng = np.random.default_rng(cols)
    try:
        for form in [0] + [10 * blocks + shares for blocks in range(1, 9) for shares in (1, 2, 4, 7)]:
            o.set_tuning("batch_gemv_form", form)
            check_kept(m, lambda x, r: m.step_product(x, r, shares=True), (3, 16) if form else (1, 3, 9, 15, 16), rng)
            if form in (0, 31):
                check_kept(m, lambda x, r: m.step_product(x, r), (3, 16), rng)
    finally:
        o.set_tuning("batch_gemv_form", 0)
    m.close()


@pytest.mark.parametrize("width", [1088, 4096, 4160, 8192])
def test_norms_of_few_rows(width):
    """Norms of up to 64 rows in 1024 threads, one and two fours of columns each, and of one row more: prompts, and steps of a batch, against the tokens one at a time, whose norms are in the products."""
    import espresso_amd.llama as ll
    import espresso_amd.ops as o
    import espresso_amd.synthetic as syn
    o.init()
    cfg = ll.MultiModelConfig(n_layer=2, n_head=4, n_kv_head=4, d_model=width, head_dim=64, hidden_dim=256, vocab=260, max_seq=128)
    rt, _ = syn.build_runtime(cfg, lib.FORMAT_F16, seed=3, std=width ** -0.5, max_sequences=3)   # products as large as their inputs: scores of a few units, which carry no rounding further
    tokens = np.random.default_rng(width).integers(0, 260, 65).astype(np.uint32)
    steps = []
    for t in tokens:
        rt.advance(int(t))
        steps.append(rt.logits())
    for count in (64, 65):
        rt.reset()
        got = rt.append(tokens[:count], want=range(count))
        # activations and contexts are fp16 in both, queries and softmax weights in blocks: 2^-12 of each at the root mean square, some ten of them in two layers, where a last bit may fall either way
        assert rms_off(got, np.stack(steps[:count])) <= 2.0 ** -9, count
    out, _ = ll.generate_batch(rt, [tokens[:40], tokens[:41], tokens[:42]], 4)
    for s in range(3):
        n = 40 + s + len(out[s])
        rt.set_visible(n - 1, sequence=s)
        b = rt.append(np.array(out[s][-1:], np.uint32), want=[0], sequence=s)[0]
        rt.set_visible(0)
        for t in list(tokens[:40 + s]) + out[s]:
            rt.advance(int(t))
        assert rms_off(b, rt.logits()) <= 2.0 ** -9, s
    rt.close()
