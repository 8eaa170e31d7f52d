"""Output heads of Q4_K models 1024 and 3072 columns wide (more than 32768 rows): the matrix-core form whose wavefronts own whole rows, against float64 and
against the arg-max of the stored logits."""
import numpy as np
import pytest

import espresso_amd._lib as lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import espresso_amd.ops as o
    o.init()
    return o


@pytest.mark.parametrize("rows,cols", [(32772, 1024), (32785, 3072), (49152, 1024)])
def test_products_match_float64(ops, rows, cols):
    m = ops.Matrix(lib.FORMAT_Q4_K, ops.synth_weights(lib.FORMAT_Q4_K, rows + cols, 0.02, rows * cols), rows, cols)
    w = m.dequantize().astype(np.float64)
    rng = np.random.default_rng(cols)
    for batch in (1, 2):
        x = rng.normal(0, 1, (batch, cols)).astype(np.float16)
        want = x.astype(np.float64) @ w.T
        # exact products and fp32 sums; scale * q and the minimum are summed apart, up to 63 * 15 steps of the super-block's scale each
        bound = 16 * (cols + cols / 16 + 16) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T + 1)
        assert (np.abs(m.gemv(x) - want) <= bound).all(), batch
    m.close()


@pytest.mark.parametrize("d", [1024, 3072])
def test_greedy_tokens_are_the_logits_maxima(ops, d):
    import espresso_amd.llama as ll
    import espresso_amd.synthetic as syn
    cfg = ll.MultiModelConfig(n_layer=1, n_head=d // 64, n_kv_head=d // 64, d_model=d, head_dim=64, hidden_dim=1024, vocab=32790, max_seq=32)
    rt, _ = syn.build_runtime(cfg, lib.FORMAT_Q4_K, seed=5, std=0.05)
    prompt = [1, 5, 32789, 7]
    tokens, _ = rt.generate(prompt, 6)
    rt.reset()
    rt.prefill(prompt)
    for t in tokens:
        logits = rt.logits()
        assert int(np.argmax(logits)) == t
        rt.advance(t)
    rt.close()
