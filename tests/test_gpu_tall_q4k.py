"""Tall output heads of Q4_K models 1024 and 3072 columns wide: the matrix-core form whose wavefronts own whole rows where the one that splits K declines, against float64 and
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


@pytest.mark.parametrize("rows,cols", [(32772, 1024), (32785, 3072), (49152, 1024), (131090, 1024)])
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


@pytest.mark.parametrize("batch", [1, 2])
def test_heights_that_fit_the_rounds_keep_the_form_that_splits_k(ops, batch):
    """40960 rows of 1024 columns are few enough for the form whose wavefronts split K (6.1 us, whole rows 7.4): each row then adds in the order it has in a matrix of 16384 rows."""
    blocks = ops.synth_weights(lib.FORMAT_Q4_K, 11, 0.02, 40960 * 1024)
    x = np.random.default_rng(3).normal(0, 1, (batch, 1024)).astype(np.float16)
    got = []
    for rows in (16384, 40960):
        m = ops.Matrix(lib.FORMAT_Q4_K, blocks[:rows * 1024 // 256 * 144], rows, 1024)
        got.append(m.gemv(x)[:, :16384])
        m.close()
    assert np.array_equal(*got)


@pytest.mark.parametrize("d,vocab", [(1024, 32790), (3072, 32790), (1024, 131090)])
def test_greedy_tokens_are_the_logits_maxima(ops, d, vocab):
    import espresso_amd.llama as ll
    import espresso_amd.synthetic as syn
    cfg = ll.MultiModelConfig(n_layer=1, n_head=d // 64, n_kv_head=d // 64, d_model=d, head_dim=64, hidden_dim=1024, vocab=vocab, max_seq=32)
    rt, _ = syn.build_runtime(cfg, lib.FORMAT_Q4_K, seed=5, std=0.05)
    prompt = [1, 5, vocab - 1, 7]
    tokens, _ = rt.generate(prompt, 6)
    rt.reset()
    rt.prefill(prompt)
    for t in tokens:
        logits = rt.logits()
        assert int(np.argmax(logits)) == t
        rt.advance(t)
    rt.close()
