"""Prompts of one block and of several long ones: what they leave agrees with short portions and with the walk token by token."""
import numpy as np
import pytest

import espresso_amd._lib as lib
import espresso_amd.layered as layered
import espresso_amd.llama as ll
import layered_util as lu
import model_util as mu
from oracle import oracle as orc
from test_gpu_block_gemm import check_kept

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,heads,kv_heads,kv_fp16,count", [
    (orc.FMT_Q8_0, 4, 2, True, 2049),    # two blocks of 1152 and 897 rows, both attention kernels of long blocks
    (orc.FMT_Q8_0, 3, 1, False, 1999), (orc.FMT_Q4_0, 3, 1, True, 2304), (orc.FMT_F16, 4, 4, True, 1025),
    (orc.FMT_Q4_K, 4, 1, True, 2111),    # exact products, queries and softmax weights as pairs
    (orc.FMT_Q4_K, 4, 2, False, 1537),
])
def test_long_blocks_match_portions_and_steps(fmt, heads, kv_heads, kv_fp16, count):
    d = 256 if fmt == orc.FMT_Q4_K or heads == 4 else 192
    cfg = dict(n_layer=2, n_head=heads, n_kv_head=kv_heads, d_model=d, head_dim=64, hidden_dim=512, vocab=256, max_seq=2560)
    w = mu.random_weights(orc.LlamaConfig(**cfg), 7 + fmt, std=0.08, norm_jitter=0.05)
    packed, _ = mu.pack_weights(w, fmt)
    rt = ll.LlamaRuntime(ll.MultiModelConfig(**cfg), kv_format=orc.FMT_F16 if kv_fp16 else orc.FMT_F32)
    ll.load_packed_weights(rt, packed, fmt)
    prompt = np.random.default_rng(count).integers(0, 256, count).astype(np.uint32)

    def last(run):
        rt.reset()
        run()
        assert rt.visible() == count
        return rt.last_hidden()

    whole = last(lambda: rt.prefill(prompt))
    assert np.array_equal(last(lambda: rt.prefill(prompt)), whole)
    scale = max(1.0, np.abs(whole).max())
    # blocks round weights, activations and softmax weights to fp16 (2^-11 each), whatever the block's length; what
    # differs with the length is the order of sums: 4e-3 is what blocks are held to against the walk elsewhere
    portions = last(lambda: [rt.append(prompt[i:i + 300]) for i in range(0, count, 300)])
    assert np.abs(portions - whole).max() <= 4e-3 * scale
    ll.set_matrix_prefill(rt, False)
    steps = last(lambda: rt.prefill(prompt))
    assert np.abs(steps - whole).max() <= 4e-3 * scale


@pytest.mark.parametrize("config", [
    lu.config([lu.latent(window=30), lu.retention(decay=[0.995, 1.0]), lu.latent(kv_from=0, window=9)]),
    lu.sequential([lu.mamba2(), lu.attention(window=70), lu.mamba2(heads=2, groups=1), lu.attention(kv_from=1, window=11, ff=0)]),
])
@pytest.mark.parametrize("precision", ["f32", "bf16"])
def test_layered_blocks_past_the_ring(tmp_path, precision, config):
    """More tokens than a block and than the cached ring holds (window - 1 + 2048 rows)."""
    m = lu.Model(tmp_path, config, seed=5, gain=1.5)
    t = lu.tokens(m.cfg, 2450, 2)
    want = m.logits(t)
    rt = m.runtime(precision, max_seq=2500)
    for s, portions in enumerate(([2400, 1], [2100, 3, 300, 1], [513, 1700, 2])):
        assert lu.error(lu.feed(rt, t, portions, s), want) < lu.limit(precision), portions


@pytest.mark.parametrize("fmt", ["q8_0", "q4_0", "q4_k"])
@pytest.mark.parametrize("rows,cols", [(576, 1536), (960, 576), (576, 576), (768, 768), (2048, 512)])   # smallest-model shapes, the most that is kept (2^20 weights)
def test_small_products_keep_their_weights_in_long_blocks(fmt, rows, cols):
    """What a block of 512 rows keeps exact, a longer one does: one row more, between, and the longest block."""
    import espresso_amd.ops as ops
    f = lib.FORMAT_NAMES[fmt]
    cols = (cols + 255) // 256 * 256 if fmt == "q4_k" else cols
    rows = min(rows, 2 ** 20 // cols // 32 * 32)
    ops.init()
    m = ops.Matrix(f, ops.synth_weights(f, rows + cols, 0.02, rows * cols), rows, cols)
    rng = np.random.default_rng(cols)
    for shares in (False, True):
        check_kept(m, lambda x, r: m.layer_product(x, r, shares=shares), (512, 513, 1055, 2048), rng)
    m.close()
