"""Passes of the exact two-token loop on the device where their kernels branch: widths whose two rows of attention states are merged at once (768 and 2048 columns; 4096 row after row), heads that leave
candidates of one or many workgroups and heads that leave tokens, drafts that are right (the model itself) and wrong (another model)."""
import numpy as np
import pytest

import espresso_amd._lib as lib
import model_util as mu
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ll():
    import espresso_amd.llama as ll
    import espresso_amd.ops as ops
    ops.init()
    return ll


def model(ll, fmt, width, head_dim, vocab, seed):
    kw = dict(n_layer=2, n_head=width // head_dim, n_kv_head=max(1, width // head_dim // 2), d_model=width, head_dim=head_dim, hidden_dim=768, vocab=vocab, max_seq=96)
    packed, _ = mu.pack_weights(mu.random_weights(orc.LlamaConfig(**kw), seed, std=0.05), fmt)
    g = ll.LlamaRuntime(ll.MultiModelConfig(**kw))
    ll.load_packed_weights(g, packed, fmt)
    return g


@pytest.mark.parametrize("fused_argmax", [True, False])
@pytest.mark.parametrize("fmt,width,head_dim,vocab", [(orc.FMT_F16, 768, 64, 9000), (orc.FMT_Q8_0, 768, 128, 130), (orc.FMT_F16, 2048, 64, 500), (orc.FMT_Q8_0, 2048, 128, 20000),
                                                      (orc.FMT_Q8_0, 4096, 128, 300), (orc.FMT_Q4_K, 4096, 128, 300), (orc.FMT_Q4_0, 2048, 64, 500), (orc.FMT_F32, 256, 64, 77)])
def test_two_token_stream_is_the_greedy_stream(ll, monkeypatch, fmt, width, head_dim, vocab, fused_argmax):
    monkeypatch.setenv("ESPRESSO_HIP_FUSED_HEAD_ARGMAX", "1" if fused_argmax else "0")   # read when a model is finished
    g = model(ll, fmt, width, head_dim, vocab, 5)
    prompt = np.random.default_rng(2).integers(0, vocab, 9).tolist()
    want = g.generate(prompt, 41)[0]
    for draft in (model(ll, fmt, width, head_dim, vocab, 5), model(ll, orc.FMT_F16, 768, 64, vocab, 8), model(ll, orc.FMT_F32, 64, 16, vocab, 9)):
        for _ in range(2):   # the second call replays the passes that the first has captured
            got = ll.generate_two_token(g, draft, prompt, 41)[0]
            assert got == want
        draft.close()
    g.close()


@pytest.mark.parametrize("fmt", ["f16", "q8_0"])
@pytest.mark.parametrize("n_head,hidden", [(12, 2048), (1, 64), (5, 1056), (2, 4096)])
def test_two_rows_add_planes_on_the_matrix_cores(ll, fmt, n_head, hidden):
    """768 columns, where attention and wo leave up to twelve planes a row to gate|up: the matrix-core kernel against the dot-product one, whose sums and norms these are, and both against single steps."""
    import espresso_amd.ops as ops
    import espresso_amd.synthetic as syn
    cfg = ll.MultiModelConfig(n_layer=2, n_head=n_head, n_kv_head=n_head, d_model=768, head_dim=64, hidden_dim=hidden, vocab=512, max_seq=64)
    g, _ = syn.build_runtime(cfg, lib.FORMAT_NAMES[fmt], seed=hidden, std=0.05)
    tokens = np.random.default_rng(n_head).integers(0, cfg.vocab, 8)
    want = []
    for t in tokens:
        g.advance(int(t))
        want.append(np.concatenate([g.logits(), g.last_hidden()]))
    got = {}
    try:
        ops.set_tuning("short_blocks", 0)
        for mfma in (0, -1):
            ops.set_tuning("q80_mfma", mfma)
            g.reset()
            got[mfma] = []
            for i in range(0, 8, 2):
                logits = g.append(tokens[i:i + 2], want=(0, 1))
                got[mfma].append(np.concatenate([logits[1], g.last_hidden()]))
    finally:
        ops.set_tuning("short_blocks", 1)
        ops.set_tuning("q80_mfma", -1)
    g.close()
    for i in range(4):   # other orders of fp32 sums; activations are rounded to fp16 in between
        limit = 2.0 ** -9 * max(1.0, np.abs(want[2 * i + 1]).max())
        assert np.abs(got[-1][i] - got[0][i]).max() <= limit and np.abs(got[-1][i] - want[2 * i + 1]).max() <= limit, i


@pytest.mark.parametrize("fmt,d_model,kv", [("f16", 704, "f32"), ("q8_0", 704, "f16"), ("q4_0", 768, "f32"), ("f16", 768, "f16")])
def test_two_rows_of_many_heads_behind_long_prefixes(ll, fmt, d_model, kv):
    """Contexts of more than 256 tokens and 12 heads: blocks of 128 rows of wo for two rows (704: the last one is half), of 64 for one."""
    import espresso_amd.ops as ops
    import espresso_amd.synthetic as syn
    cfg = ll.MultiModelConfig(n_layer=2, n_head=12, n_kv_head=4, d_model=d_model, head_dim=64, hidden_dim=512, vocab=512, max_seq=300)
    g, _ = syn.build_runtime(cfg, lib.FORMAT_NAMES[fmt], seed=d_model, std=0.05, kv_format=lib.FORMAT_F16 if kv == "f16" else lib.FORMAT_F32)
    tokens = np.random.default_rng(d_model).integers(0, cfg.vocab, 280).astype(np.uint32)
    try:
        ops.set_tuning("short_blocks", 0)
        for first in (2, 127, 271):
            g.reset()
            g.prefill(tokens[:first])
            got = np.concatenate([g.append(tokens[i:i + 2], want=(0, 1)) for i in range(first, first + 8, 2)])
            g.set_visible(first)
            for i in range(8):
                g.advance(int(tokens[first + i]))
                want = g.logits()   # other orders of fp32 sums; activations are rounded to fp16 in between
                assert np.abs(got[i] - want).max() <= 2.0 ** -9 * max(1.0, np.abs(want).max()), (first, i)
    finally:
        ops.set_tuning("short_blocks", 1)
    g.close()
