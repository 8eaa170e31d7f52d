"""Prompts of one block and of several long ones: what they leave agrees with short portions and with the walk token by token."""
import numpy as np
import pytest

import espresso_amd._lib as lib
import espresso_amd.layered as layered
import espresso_amd.llama as ll
import layered_util as lu
import model_util as mu
from oracle import oracle as orc
from test_gpu_block_gemm import check_kept, rms_off

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,heads,kv_heads,kv_fp16,count", [
    (orc.FMT_Q8_0, 4, 2, True, 2049),    # a block of 2048 rows and one row in a block of its own
    (orc.FMT_Q8_0, 3, 1, False, 1999), (orc.FMT_Q4_0, 3, 1, True, 2304), (orc.FMT_F16, 4, 4, True, 1025),
    (orc.FMT_Q4_K, 4, 1, True, 2111),    # exact products of split rows
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


# shape, format, caches; prompts and the rows beyond 512 k that are more exact in a block of their own: weights kept at 40 and at 200 rows but not at 512 (gate|up of 4608 x 768, down of
# 768 x 2304), 32-bit attention of fewer than 32 rows (three query heads to a key/value head have it in every block)
WIDE = dict(n_head=12, n_kv_head=4, d_model=768, head_dim=64, hidden_dim=2304)
PAIRS = dict(WIDE, n_kv_head=6)
CASES = [
    (PAIRS, lib.FORMAT_Q8_0, lib.FORMAT_F16, 552, 40), (WIDE, lib.FORMAT_Q8_0, lib.FORMAT_F32, 552, 40), (WIDE, lib.FORMAT_Q4_0, lib.FORMAT_F16, 2760, 200), (WIDE, lib.FORMAT_Q4_K, lib.FORMAT_F16, 1064, 40),
    (PAIRS, lib.FORMAT_Q8_0, lib.FORMAT_F16, 1034, 10), (PAIRS, lib.FORMAT_Q4_0, lib.FORMAT_F32, 513, 1),
    (WIDE, lib.FORMAT_Q4_K, lib.FORMAT_F16, 1031, 7),   # activations as pairs: a block of its own
    (PAIRS, lib.FORMAT_F16, lib.FORMAT_F16, 1031, 7), (dict(n_head=8, n_kv_head=2, d_model=512, head_dim=64, hidden_dim=768), lib.FORMAT_Q4_K, lib.FORMAT_F16, 543, 31),   # attention alone
]


@pytest.mark.parametrize("shape,fmt,kv,count,last", CASES)
def test_last_rows_are_as_exact_as_in_a_block_of_their_own(shape, fmt, kv, count, last):
    import espresso_amd.ops as ops
    import espresso_amd.synthetic as syn
    ops.init()
    cfg = ll.MultiModelConfig(n_layer=2, vocab=260, max_seq=2816, **shape)
    rt, _ = syn.build_runtime(cfg, fmt, seed=3, std=0.05, kv_format=kv, max_sequences=2)
    prompt = np.random.default_rng(count).integers(0, 260, count).astype(np.uint32)
    rt.prefill(prompt[:count - last])
    want = rt.append(prompt[count - last:], want=range(last))
    rt.reset()
    got = rt.append(prompt, want=range(count - last, count))
    hidden = rt.last_hidden()
    # the same roundings, sums in another order: a last bit of an fp16 activation falls either way, up to 5.3e-4 of the logits' size; in a long block like its other rows they are 1.0 to 1.7e-3 off
    # (512 wide: products of split rows, attention in 32 bits)
    assert rms_off(got, want) <= (2.0 ** -18 if shape["d_model"] == 512 else 3 * 2.0 ** -12)
    rt.reset()
    ll.generate_batch(rt, [prompt, prompt[:count - 3]], 1)
    assert np.array_equal(rt.last_hidden(), hidden)
    rt.close()


@pytest.mark.parametrize("fmt,kv,count", [(lib.FORMAT_F16, lib.FORMAT_F16, 600), (lib.FORMAT_Q8_0, lib.FORMAT_F16, 1008), (lib.FORMAT_Q4_K, lib.FORMAT_F32, 1012)])
def test_rows_that_gain_nothing_stay_in_the_long_block(fmt, kv, count):
    """A last stretch whose block would round the same way adds no pass over the weights: one launch of each product, whatever follows the last 512 rows."""
    import espresso_amd.ops as ops
    import espresso_amd.synthetic as syn
    ops.init()
    cfg = ll.MultiModelConfig(n_layer=1, vocab=260, max_seq=1024, n_head=16, n_kv_head=16, d_model=2048, head_dim=128, hidden_dim=5632)
    rt, _ = syn.build_runtime(cfg, fmt, seed=3, std=0.03, kv_format=kv)
    prompt = np.random.default_rng(count).integers(0, 260, count).astype(np.uint32)
    rt.prefill(prompt[:512])
    rt.append(prompt[512:])
    apart = rt.last_hidden()
    rt.reset()
    rt.prefill(prompt)
    # another order of sums somewhere
    assert not np.array_equal(rt.last_hidden(), apart) and np.abs(rt.last_hidden() - apart).max() <= 4e-3 * max(1.0, np.abs(apart).max())
    rt.close()
