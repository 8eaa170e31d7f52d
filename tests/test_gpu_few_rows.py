"""Steps and blocks of a few rows: the narrow forms of the exact Q4_K GEMM, batches of up to sixteen sequences in one launch per
projection, and short prompts two tokens per step."""
import numpy as np
import pytest

import espresso_amd._lib as lib
from oracle import oracle as orc
from test_gpu_full_size import oracle_from_packed

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mods():
    import espresso_amd.llama as ll
    import espresso_amd.ops as ops
    import espresso_amd.synthetic as syn
    ops.init()
    return ll, ops, syn


@pytest.mark.parametrize("form", [1, 2, 4])
@pytest.mark.parametrize("rows,cols", [(130, 1024), (384, 2048), (40, 3072)])
def test_narrow_split_gemm_matches_float64(mods, form, rows, cols):
    _, ops, _ = mods
    m = ops.Matrix(lib.FORMAT_Q4_K, ops.synth_weights(lib.FORMAT_Q4_K, rows, 0.02, rows * cols), rows, cols)
    w = m.dequantize().astype(np.float64)
    try:
        ops.set_tuning("split_gemm_narrow", form)
        for n in (3, 31, 32, 33, 64, 65, 129):
            x = np.random.default_rng(n).normal(0, 1, (n, cols)).astype(np.float32)
            res = np.random.default_rng(n + 1).normal(0, 1, (n, rows)).astype(np.float32)
            want = x.astype(np.float64) @ w.T + res
            # the bound test_gpu_split_gemm.py holds the whole form to: the split leaves 2^-22 per activation, the sums are fp32
            assert np.abs(m.matmul_f32(x, res) - want).max() <= 4e-6 * (want - res).std() + 1e-6, n
            if rows % 8:
                continue
            g = x.astype(np.float64) @ w.T
            gate, up = g[:, 0::2], g[:, 1::2]
            act = gate / (1 + np.exp(-gate)) * up
            assert (np.abs(m.matmul_f32_swiglu(x) - act) <= 5e-6 * g.std() * (np.abs(up) + np.abs(gate) + 1.0)).all(), n
    finally:
        ops.set_tuning("split_gemm_narrow", -1)
    m.close()


@pytest.mark.parametrize("cols", [256, 1024])   # weights staged through LDS, and read in the tiled order
@pytest.mark.parametrize("form", [0, 1, 2, 4])
def test_silu_is_exact_to_its_split_rows(mods, cols, form):
    """Gates and ups that the product holds exactly (weights 0 and 1), so that only SiLU and the 22 bits of the planes are left."""
    _, ops, _ = mods
    units, n = 64, 31
    block = np.zeros((2 * units, cols // 256, 144), np.uint8)
    block[:, :, 0:2] = np.frombuffer(np.float16(0.125).tobytes(), np.uint8)
    block[:, :, 4:8] = block[:, :, 12:16] = 1                      # every sub-block's scale 1, every minimum 0
    for u in range(units):
        block[2 * u, 0, 16 + u % 32] = 8 << 4 * (u // 32)          # gate = x[u]
        block[2 * u + 1, 0, 16 + 127] = 8 << 4                     # up = x[255]
    m = ops.Matrix(lib.FORMAT_Q4_K, block, 2 * units, cols)
    x = np.zeros((n, cols), np.float32)
    x[:, :units] = np.round(np.linspace(-16, 16, n * units) * 1024).reshape(n, units) / 1024
    x[:, 255] = 1024
    g = x[:, :units].astype(np.float64)
    want = 1024 * g / (1 + np.exp(-g))
    try:
        ops.set_tuning("split_gemm_narrow", form)
        got = m.matmul_f32_swiglu(x)
    finally:
        ops.set_tuning("split_gemm_narrow", -1)
    # expf 2^-23, sum, quotient and product 2^-24 each, planes 2^-23
    assert (np.abs(got - want) <= 3.5 * 2.0 ** -23 * np.abs(want) + 1e-12).all(), np.nanmax(np.abs(got - want) / np.maximum(np.abs(want), 1e-9))
    m.close()


# column counts of the sixteen-row kernel: d_model and attention width, hidden size
@pytest.mark.parametrize("fmt,d,hidden,kv_fp16", [(orc.FMT_Q4_K, 1024, 2048, True), (orc.FMT_Q4_K, 2048, 3072, False), (orc.FMT_Q4_K, 3072, 8192, True),
                                                  (orc.FMT_Q4_K, 4096, 14336, True), (orc.FMT_Q4_0, 4096, 14336, False),
                                                  (orc.FMT_Q4_0, 2048, 8192, True), (orc.FMT_Q4_0, 3072, 8192, False)])
def test_batches_match_oracle(mods, fmt, d, hidden, kv_fp16):
    ll, ops, syn = mods
    cfg = ll.MultiModelConfig(n_layer=1, n_head=d // 128, n_kv_head=d // 512, d_model=d, head_dim=128, hidden_dim=hidden, vocab=520 if fmt != orc.FMT_Q4_K else 512, max_seq=64)
    g, packed = syn.build_runtime(cfg, fmt, seed=d, keep_packed=True, max_sequences=16, kv_format=orc.FMT_F16 if kv_fp16 else orc.FMT_F32)
    o = oracle_from_packed(cfg, packed, fmt, 1, kv_fp16, 64)
    prompts = [np.random.default_rng(s).integers(0, cfg.vocab, 1 + s % 5).astype(np.uint32) for s in range(16)]
    for n in (3, 8, 9, 16):
        g.reset()
        got, _ = ll.generate_batch(g, prompts[:n], 5)
        for s in (0, n // 2, n - 1):
            o.reset()
            o.prefill([int(t) for t in prompts[s]])
            for t in got[s]:   # a near tie may fall either way: the chosen token's logit is what has to match
                logits = o.logits()
                assert logits.max() - logits[t] <= 2e-2, (n, s)
                o.advance(int(t))
        # the caches hold what the steps wrote
        logits = g.append([int(got[n - 1][-1])], want=[0], sequence=n - 1)[0]
        assert np.abs(logits - o.logits()).max() <= 2e-2
    g.close()


@pytest.mark.parametrize("fmt,d,hidden", [("q8_0", 256, 512), ("f16", 576, 1536), ("q4_0", 768, 2048), ("q4_k", 1024, 3072)])
def test_short_prompts_in_pairs_match_single_steps(mods, fmt, d, hidden):
    ll, ops, syn = mods
    cfg = ll.MultiModelConfig(n_layer=2, n_head=d // 64, n_kv_head=d // 64, d_model=d, head_dim=64, hidden_dim=hidden, vocab=512, max_seq=64)
    g, _ = syn.build_runtime(cfg, lib.FORMAT_NAMES[fmt], seed=5, std=0.05)   # fp32 caches: no block form takes prompts this short
    tokens = np.random.default_rng(d).integers(0, cfg.vocab, 12)
    want = []
    for t in tokens:
        g.advance(int(t))
        want.append(g.logits())
    want = np.array(want)
    for portions in ([12], [2, 3, 7], [1, 11], [5, 2, 2, 3]):
        g.reset()
        got = []
        for n in portions:
            at = g.visible()
            got.append(g.append(tokens[at:at + n], want=range(n)))
        # one and two rows take the same products in another order of their fp32 sums; activations are rounded to fp16 in between
        assert np.abs(np.concatenate(got) - want).max() <= 2.0 ** -9 * max(1.0, np.abs(want).max()), portions
        assert np.abs(g.logits() - want[-1]).max() <= 2.0 ** -9 * max(1.0, np.abs(want).max())
    g.close()


@pytest.mark.parametrize("fmt,hidden", [("q8_0", 53248), ("f16", 40960), ("f16", 40448), ("q4_0", 53248), ("q4_k", 53248)])
def test_short_prompts_of_feed_forwards_too_wide_for_pairs(mods, fmt, hidden):
    """Two rows of 40960 columns and more do not fit the LDS of a workgroup: such prompts walk one token per step."""
    ll, ops, syn = mods
    cfg = ll.MultiModelConfig(n_layer=1, n_head=4, n_kv_head=4, d_model=256, head_dim=64, hidden_dim=hidden, vocab=512, max_seq=16)
    g, _ = syn.build_runtime(cfg, lib.FORMAT_NAMES[fmt], seed=5, std=0.05)
    tokens = np.random.default_rng(hidden).integers(0, cfg.vocab, 5).astype(np.uint32)
    for t in tokens:
        g.advance(int(t))
    want = g.logits()
    try:
        for blocks in (0, 1):   # such steps, then what such prompts take by themselves
            ops.set_tuning("short_blocks", blocks)
            g.prefill(tokens)
            assert np.abs(g.logits() - want).max() <= 2.0 ** -9 * max(1.0, np.abs(want).max())   # as above
    finally:
        ops.set_tuning("short_blocks", 1)
    g.close()


def test_short_exact_blocks_keep_32_bit_attention(mods):
    """Turns of 4 to 31 tokens, which single steps could walk as well, match the steps behind the same prefix, whether four or eight wavefronts deal their keys (which shows in the last bits)."""
    ll, ops, syn = mods
    cfg = ll.MultiModelConfig(n_layer=2, n_head=8, n_kv_head=2, d_model=1024, head_dim=128, hidden_dim=3072, vocab=512, max_seq=256)
    g, _ = syn.build_runtime(cfg, lib.FORMAT_Q4_K, seed=9, std=0.05, kv_format=lib.FORMAT_F16)
    tokens = np.random.default_rng(4).integers(0, cfg.vocab, 200).astype(np.uint32)
    def turn(n, sets=0):
        ops.set_tuning("prompt_attention_key_sets", sets)
        g.set_visible(150)
        return g.append(tokens[150:150 + n], want=range(n))
    try:
        g.prefill(tokens[:150])
        assert not np.array_equal(turn(40, 1), turn(40, 2))
        for n in (4, 9, 31):
            ll.set_matrix_prefill(g, False)
            want = turn(n)
            ll.set_matrix_prefill(g, True)
            for sets in (0, 1, 2):   # contexts and caches are fp16 on both ways, sums in another order
                assert np.abs(turn(n, sets) - want).max() <= 2.0 ** -9 * max(1.0, np.abs(want).max()), (n, sets)
        assert not np.array_equal(turn(31, 1), turn(31, 2))
    finally:
        ops.set_tuning("prompt_attention_key_sets", 0)
    g.close()


def test_without_matrix_prefill_every_token_is_a_step(mods):
    ll, ops, syn = mods
    cfg = ll.MultiModelConfig(n_layer=2, n_head=4, n_kv_head=4, d_model=256, head_dim=64, hidden_dim=512, vocab=512, max_seq=64)
    g, _ = syn.build_runtime(cfg, lib.FORMAT_Q8_0, seed=5, std=0.05)
    tokens = np.random.default_rng(1).integers(0, cfg.vocab, 43).astype(np.uint32)
    ll.set_kernel_timing(g, True)
    try:
        for enabled, blocks, count, steps in [(False, 1, 43, 43), (False, 1, 7, 7), (True, 0, 7, 4), (True, 1, 7, 0)]:   # (a block's products are not among the counted launches)
            ops.set_tuning("short_blocks", blocks)
            ll.set_matrix_prefill(g, enabled)
            g.reset()
            ll.kernel_times(g)
            g.prefill(tokens[:count])
            assert ll.kernel_times(g)["qkv"]["launches"] == cfg.n_layer * steps, (enabled, blocks, count)
    finally:
        ops.set_tuning("short_blocks", 1)
    g.close()


@pytest.mark.parametrize("cols", [2048, 3072, 8192])
@pytest.mark.parametrize("rows", [16, 130, 4097, 16400, 33000])
def test_q4_0_matrix_core_widths_match_float64(mods, rows, cols):
    _, ops, _ = mods
    m = ops.Matrix(lib.FORMAT_Q4_0, ops.synth_weights(lib.FORMAT_Q4_0, rows, 0.02, rows * cols), rows, cols)
    w = m.dequantize().astype(np.float64).reshape(rows, cols)
    try:
        ops.set_tuning("q40_mfma", 1)
        for batch in (1, 2):
            x = np.random.default_rng(batch).normal(0, 1, (batch, cols)).astype(np.float16)
            res = np.random.default_rng(rows).normal(0, 1, (batch, rows)).astype(np.float32)
            want = x.astype(np.float64) @ w.T
            # exact products, fp32 sums: the bound test_gpu_q40_mfma.py holds the other widths to
            tol = 2e-5 * np.abs(w).max() * np.sqrt(cols) + 1e-6
            assert np.abs(m.gemv(x) - want).max() <= tol, batch
            assert np.abs(m.gemv(x, res) - (want + res)).max() <= tol + 1e-5, batch
    finally:
        ops.set_tuning("q40_mfma", -1)
    m.close()


@pytest.mark.parametrize("d,heads,kv,hidden", [(2048, 32, 8, 8192), (3072, 24, 8, 8192)])
def test_q4_0_decode_matches_oracle(mods, d, heads, kv, hidden):
    """Norm, RoPE / cache, merged attention, SwiGLU, residual and arg-max forms, then the two-row steps of a short prompt."""
    ll, ops, syn = mods
    cfg = ll.MultiModelConfig(n_layer=1, n_head=heads, n_kv_head=kv, d_model=d, head_dim=d // heads, hidden_dim=hidden, vocab=9000, max_seq=48)
    g, packed = syn.build_runtime(cfg, orc.FMT_Q4_0, seed=d, kv_format=orc.FMT_F16, keep_packed=True)
    o = oracle_from_packed(cfg, packed, orc.FMT_Q4_0, 1, True, 48)
    prompt = [1, 8999, 777, 16, 5]
    o.prefill(prompt)
    ops.set_tuning("short_blocks", 0)
    try:
        g.prefill(np.asarray(prompt, np.uint32))
    finally:
        ops.set_tuning("short_blocks", 1)
    for _ in range(5):
        want = o.logits()
        assert np.abs(want - g.logits()).max() <= 2e-2
        tok = o.select_greedy()
        if o.top2_margin() > 1e-3:
            assert g.select_greedy() == tok
        o.advance(tok)
        g.advance(tok)
    g.close()


# rows of one, two, four and eight float4 (groups of eight) per thread, whole and ragged; partial sums of split products behind them
@pytest.mark.parametrize("fmt,d,heads,hidden", [(orc.FMT_F16, 64, 1, 4096), (orc.FMT_Q8_0, 1088, 17, 640), (orc.FMT_Q8_0, 2304, 18, 640),
                                                (orc.FMT_F16, 4352, 34, 640), (orc.FMT_Q4_K, 2304, 18, 768), (orc.FMT_Q4_K, 4352, 34, 512)])
def test_block_rows_match_oracle(mods, fmt, d, heads, hidden):
    ll, ops, syn = mods
    cfg = ll.MultiModelConfig(n_layer=2, n_head=heads, n_kv_head=heads, d_model=d, head_dim=d // heads, hidden_dim=hidden, vocab=512, max_seq=48)
    g, packed = syn.build_runtime(cfg, fmt, seed=d, kv_format=orc.FMT_F16, keep_packed=True)
    o = oracle_from_packed(cfg, packed, fmt, 2, True, 48)
    prompt = np.random.default_rng(d).integers(0, cfg.vocab, 37).astype(np.uint32)
    o.prefill([int(t) for t in prompt])
    g.prefill(prompt)
    want = o.logits()
    # fp16 activations in front of every product (fp16 weights too where the block kernels round them)
    assert np.abs(g.logits() - want).max() <= 2.0 ** -8 * max(1.0, np.abs(want).max())
    g.close()
