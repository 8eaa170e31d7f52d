"""block_gemm_kernel against float64 at the edges of its tiles: activation rows around multiples of 32 and of the tile, weight rows that leave
wavefronts and workgroups partly or wholly without rows, columns that leave groups of wavefronts short of steps or without any, every format,
every form, with and without a residual."""
import numpy as np
import pytest

import espresso_amd._lib as lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import espresso_amd.ops as o
    o.init()
    yield o
    o.set_tuning("block_gemm_form", 0)


def rms_off(got, want):
    return np.sqrt(np.mean((got - want) ** 2)) / np.sqrt(np.mean(want ** 2))


FORMS = [181, 182, 141, 143, 121, 128, 281, 242, 221, 381, 341, 322, 481, 484, 441, 443]   # row tiles, wavefronts along the weights, shares of K


@pytest.mark.parametrize("fmt,rows,cols", [
    ("q4_k", 256, 256), ("q4_k", 33, 2304), ("q4_k", 290, 4096), ("q4_0", 4, 128), ("q4_0", 300, 1152), ("q4_0", 64, 2688),
    ("q8_0", 258, 128), ("q8_0", 30, 1408), ("q8_0", 520, 640),
])
def test_products_match_float64(ops, fmt, rows, cols):
    f = lib.FORMAT_NAMES[fmt]
    m = ops.Matrix(f, ops.synth_weights(f, rows + cols, 0.02, rows * cols), rows, cols)
    w = m.dequantize().astype(np.float16).astype(np.float64)   # what reaches the matrix cores: each weight rounded to fp16 once
    rng = np.random.default_rng(cols)
    for form in FORMS:
        ops.set_tuning("block_gemm_form", form)
        for batch in (9, 32, 33, 97, 128, 161):
            x = rng.normal(0, 1, (batch, cols)).astype(np.float16)
            residual = rng.normal(0, 1, (batch, rows)).astype(np.float32) if batch % 2 else None
            want = x.astype(np.float64) @ w.T + (0 if residual is None else residual)
            # exact products, fp32 sums in some order: one rounding per addition, relative to the sum of the magnitudes
            bound = (cols + 16) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T + 1)
            if fmt == "q4_k":   # a weight that fp32 rounding leaves within its last bit of a tie may round to fp16 the other way: one in 2^12, four in a row allowed
                bound = bound + 4 * 2.0 ** -11 * np.abs(x).max(1).astype(np.float64)[:, None] * np.abs(w).max()
            assert (np.abs(m.gemv(x, residual) - want) <= bound).all(), (form, batch)
    ops.set_tuning("block_gemm_form", 0)
    m.close()


def check_kept(m, product, batches, rng):
    """Products that keep every weight: within the rounding of fp32 sums, and far below what weights rounded to fp16 would be off."""
    w = m.dequantize().astype(np.float64)
    rounded = m.dequantize().astype(np.float16).astype(np.float64)
    off, off_rounded = [], []
    for batch in batches:
        x = rng.normal(0, 1, (batch, m.cols)).astype(np.float16)
        residual = rng.normal(0, 1e-3, (batch, m.rows)).astype(np.float32) if batch % 2 else None
        x64 = x.astype(np.float64)
        want = x64 @ w.T + (0 if residual is None else residual)
        got = product(x, residual)
        # exact products (integers below 2^8 against 11-bit numbers), one rounding per addition and per scale, relative to the sum of the magnitudes
        bound = (m.cols + m.cols / 16 + 16) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w).T + 1)
        assert (np.abs(got - want) <= bound).all(), batch
        spread = np.sqrt((x64 ** 2) @ (w ** 2).T) + 1e-30
        off.append(((got - want) / spread).ravel())
        off_rounded.append(((x64 @ rounded.T - x64 @ w.T) / spread).ravel())
        # fp32 sums cost 2^-24 an addition; fp16-rounded weights are off by 2^-12 / sqrt(3) each
        rms = lambda v: np.sqrt(np.mean(v ** 2))  # noqa: E731
        assert batch < 9 or rms(off[-1]) <= 2.0 ** -21 < rms(off_rounded[-1]) / 8, (batch, rms(off[-1]), rms(off_rounded[-1]))
    off, off_rounded = rms(np.concatenate(off)), rms(np.concatenate(off_rounded))
    assert off <= 2.0 ** -21 < off_rounded / 8, (off, off_rounded)


@pytest.mark.parametrize("fmt,rows,cols", [("q8_0", 256, 128), ("q8_0", 40, 2304), ("q8_0", 290, 1408), ("q4_0", 4, 128), ("q4_0", 300, 1152), ("q4_0", 72, 8320)])
def test_few_rows_keep_their_weights(ops, fmt, rows, cols):
    """Up to 32 rows, every exact form."""
    f = lib.FORMAT_NAMES[fmt]
    m = ops.Matrix(f, ops.synth_weights(f, rows + cols, 0.02, rows * cols), rows, cols)
    rng = np.random.default_rng(cols)
    ops.set_tuning("rows_gemm", 0)
    try:
        for form in (181, 182, 141, 143, 121, 128):
            ops.set_tuning("block_gemm_form", form)
            check_kept(m, lambda x, r: m.layer_product(x, r, shares=form % 4 != 0), (3, 5, 8, 9, 31, 32), rng)
    finally:
        ops.set_tuning("block_gemm_form", 0)
        ops.set_tuning("rows_gemm", 1)
    m.close()


@pytest.mark.parametrize("fmt", ["q8_0", "q4_0"])
@pytest.mark.parametrize("rows,cols,batches", [(2048, 2048, (9, 31, 33, 64, 65, 97, 128)), (2090, 2048, (33, 64, 65, 96)), (2075, 2304, (32, 33, 61)), (2048, 3072, (9, 33, 64)),
                                               (768, 2048, (9, 32, 33, 128)), (300, 768, (9, 33, 128)), (2090, 5632, (3, 9, 31, 32))])
def test_rules_keep_weights_of_small_products(ops, fmt, rows, cols, batches):
    """What the layers' products take by size: here (one to four row tiles, with and without shares of K, ragged weight rows) or in rows_gemm.hip."""
    f = lib.FORMAT_NAMES[fmt]
    m = ops.Matrix(f, ops.synth_weights(f, rows + cols, 0.02, rows * cols), rows, cols)
    rng = np.random.default_rng(cols)
    check_kept(m, lambda x, r: m.layer_product(x, r, shares=True), batches, rng)
    check_kept(m, lambda x, r: m.layer_product(x, r), batches, rng)
    if cols >= 2048 and cols % 512 == 0 and rows >= 2048:
        ops.set_tuning("rows_gemm", 0)
        try:
            for form in (181, 143, 121, 124):   # the same products here whatever the rule
                ops.set_tuning("block_gemm_form", form)
                check_kept(m, lambda x, r: m.layer_product(x, r, shares=True), batches, rng)
        finally:
            ops.set_tuning("block_gemm_form", 0)
            ops.set_tuning("rows_gemm", 1)
    m.close()


@pytest.mark.parametrize("cols,batch,here", [(2304, 12, False), (2304, 31, True), (2304, 48, False), (2816, 48, False), (2048, 48, True), (2560, 12, True)])
def test_shares_of_k_by_columns(ops, cols, batch, here):
    """Rows of a multiple of 512 columns are shared where a layer adds the shares; others, which the kernel of one launch reads faster, at 17 to 32 rows only."""
    m = ops.Matrix(lib.FORMAT_Q8_0, ops.synth_weights(lib.FORMAT_Q8_0, cols, 0.02, 2048 * cols), 2048, cols)
    x = np.random.default_rng(cols).normal(0, 1, (batch, cols)).astype(np.float16)
    default = m.layer_product(x, shares=True)
    try:
        ops.set_tuning("rows_gemm", 2)   # always that kernel, which adds in another order
        assert np.array_equal(default, m.layer_product(x, shares=True)) != here
    finally:
        ops.set_tuning("rows_gemm", 1)
    m.close()


@pytest.mark.parametrize("fmt", ["q8_0", "q4_k"])
def test_forms_do_not_change_how_weights_are_rounded(ops, fmt):
    """A chosen form is the same product: a handle's five rows of Q8_0 round their weights as they do by size."""
    f = lib.FORMAT_NAMES[fmt]
    m = ops.Matrix(f, ops.synth_weights(f, 7, 0.02, 300 * 1024), 300, 1024)
    w = m.dequantize()
    x = np.random.default_rng(2).normal(0, 1, (9 if fmt == "q4_k" else 5, 1024)).astype(np.float16)
    x64 = x.astype(np.float64)
    spread = np.sqrt((x64 ** 2) @ (w.astype(np.float64) ** 2).T)
    rms = lambda v: np.sqrt(np.mean((v / spread) ** 2))  # noqa: E731
    try:
        for form in (0, 181, 143, 121):
            ops.set_tuning("block_gemm_form", form)
            got = m.gemv(x)
            assert rms(got - x64 @ w.astype(np.float16).astype(np.float64).T) <= 2.0 ** -21 < rms(got - x64 @ w.astype(np.float64).T) / 8, form
    finally:
        ops.set_tuning("block_gemm_form", 0)
    m.close()


@pytest.mark.parametrize("fmt,kv", [("q8_0", lib.FORMAT_F32), ("q4_0", lib.FORMAT_F16), ("f16", lib.FORMAT_F16)])
@pytest.mark.parametrize("heads,kv_heads", [(12, 12), (12, 4)])
def test_short_blocks_are_the_steps(ops, fmt, kv, heads, kv_heads):
    """Prompts of 5 to 31 tokens as one block, behind a prefix and without one, against the same tokens one at a time."""
    import espresso_amd.llama as ll
    import espresso_amd.synthetic as syn
    cfg = ll.MultiModelConfig(n_layer=2, n_head=heads, n_kv_head=kv_heads, d_model=768, head_dim=64, hidden_dim=2304, vocab=260, max_seq=128)
    rt, _ = syn.build_runtime(cfg, lib.FORMAT_NAMES[fmt], seed=3, std=0.05, kv_format=kv)
    tokens = np.random.default_rng(1).integers(0, 260, 80).astype(np.uint32)
    for prefix, count in ((0, 5), (0, 31), (40, 9), (33, 17)):
        rt.reset()
        if prefix:
            rt.prefill(tokens[:prefix])
        block = rt.append(tokens[prefix:prefix + count], want=range(count))
        rt.set_visible(prefix)
        steps = []
        for t in tokens[prefix:prefix + count]:
            rt.advance(int(t))
            steps.append(rt.logits())
        want = np.stack(steps)
        # the same roundings in both: activations and contexts to fp16, where a last bit may fall either way: 3.5 to 5.5e-4 of the logits' size over two layers ...
        assert rms_off(block, want) <= 3 * 2.0 ** -12 and np.abs(block - want).max() <= 2.0 ** -9 * max(1.0, np.abs(want).max()), (prefix, count)
        if fmt != "f16":   # ... where a form that rounds the weights is 1.1 to 1.4e-3 off
            try:
                ops.set_tuning("rows_gemm", 0)
                ops.set_tuning("block_gemm_form", 241)
                rt.set_visible(prefix)
                assert rms_off(rt.append(tokens[prefix:prefix + count], want=range(count)), want) > 3 * 2.0 ** -12, (prefix, count)
            finally:
                ops.set_tuning("rows_gemm", 1)
                ops.set_tuning("block_gemm_form", 0)
    rt.close()


@pytest.mark.parametrize("fmt", ["q8_0", "q4_k"])
def test_gate_up_epilogue_matches_planes(ops, fmt):
    """Prompts through a two-layer model: SiLU(gate) * up in the product's epilogue, and by the launch that adds planes."""
    import espresso_amd.llama as ll
    import espresso_amd.synthetic as syn
    cfg = ll.MultiModelConfig(n_layer=2, n_head=12, n_kv_head=4, d_model=768, head_dim=64, hidden_dim=2304, vocab=260, max_seq=256)
    logits = {}
    ops.set_tuning("rows_gemm", 0)
    try:
        for form in (241, 243, 481, 0):
            ops.set_tuning("block_gemm_form", form)
            rt, _ = syn.build_runtime(cfg, lib.FORMAT_NAMES[fmt], seed=3, std=0.05)
            ll.set_split_activations(rt, False)
            logits[form] = rt.append(np.arange(161, dtype=np.uint32), want=[0, 7, 160])
            rt.close()
    finally:
        ops.set_tuning("block_gemm_form", 0)
        ops.set_tuning("rows_gemm", 1)
    # activations are rounded to fp16 between the products, where a last bit may fall either way
    for form in (243, 481, 0):
        assert np.abs(logits[241] - logits[form]).max() <= 2.0 ** -9 * max(1.0, np.abs(logits[241]).max()), form


@pytest.mark.parametrize("fmt", ["q8_0", "q4_0"])
def test_small_products_of_more_rows_keep_their_weights(ops, fmt):
    """33 to 96 rows of 2048 columns whose weights a step keeps, in shares of K, against one launch without shares (rows_gemm = 2: always that kernel).  Of 128 rows the
    2560 weight rows of q|k|v are too many for the rule and rounded."""
    import espresso_amd.llama as ll
    import espresso_amd.synthetic as syn
    cfg = ll.MultiModelConfig(n_layer=1, n_head=32, n_kv_head=4, d_model=2048, head_dim=64, hidden_dim=256, vocab=260, max_seq=192)
    rt, _ = syn.build_runtime(cfg, lib.FORMAT_NAMES[fmt], seed=3, std=0.05, kv_format=lib.FORMAT_F16)
    tokens = np.random.default_rng(1).integers(0, 260, 129).astype(np.uint32)
    try:
        for count in (34, 64, 65, 96, 128):
            logits = {}
            for mode, form in ((1, 0), (2, 0), (0, 241)):
                ops.set_tuning("rows_gemm", mode)
                ops.set_tuning("block_gemm_form", form)
                rt.reset()
                logits[mode] = rt.append(tokens[:count], want=[0, 31, 32, count - 1])
            # fp32 sums in another order; activations are rounded to fp16 between the products, where a last bit may fall either way: 1.6 to 2.8e-4 of the logits'
            # size, with rounded weights (mode 0) 8.8e-4 to 1.06e-3
            assert np.abs(logits[1] - logits[2]).max() <= 2.0 ** -9 * max(1.0, np.abs(logits[2]).max()), count
            assert (rms_off(logits[1], logits[2]) <= 2.0 ** -11) == (count <= 96) and rms_off(logits[0], logits[2]) > 2.0 ** -11, count
    finally:
        ops.set_tuning("rows_gemm", 1)
        ops.set_tuning("block_gemm_form", 0)
        rt.close()


@pytest.mark.parametrize("fmt,rows,cols,batch,key,value", [
    ("q4_0", 256, 256, 3, "rows_gemm", 2), ("q4_0", 768, 768, 8, "rows_gemm", 2), ("q4_0", 2048, 2048, 5, "rows_gemm", 2), ("q4_0", 5632, 2048, 8, "rows_gemm", 2), ("q4_0", 8192, 3072, 3, "rows_gemm", 2),
    ("q4_0", 11264, 2048, 8, "rows_gemm", 0), ("q4_0", 2048, 5632, 8, "rows_gemm", 0),   # more workgroups than compute units, long rows: here
    ("q8_0", 768, 768, 16, "block_gemm_form", 121), ("q4_k", 2048, 2048, 16, "block_gemm_form", 122),   # no shares of K whose sum is a launch
])
def test_single_products_pay_for_no_launch_that_adds_shares(ops, fmt, rows, cols, batch, key, value):
    """A matrix handle's product has no next kernel that could add shares of K: where those and their launch cost more than they give, another form is taken.
    Forms that split K differently add in another order, so equal bits are the same split."""
    f = lib.FORMAT_NAMES[fmt]
    m = ops.Matrix(f, ops.synth_weights(f, rows + cols, 0.02, rows * cols), rows, cols)
    x = np.random.default_rng(cols).normal(0, 1, (batch, cols)).astype(np.float16)
    default = m.gemv(x)
    try:
        ops.set_tuning(key, value)
        assert np.array_equal(default, m.gemv(x))
    finally:
        ops.set_tuning("rows_gemm", 1)
        ops.set_tuning("block_gemm_form", 0)
    w = m.dequantize()
    w = (w if fmt == "q4_0" else w.astype(np.float16)).astype(np.float64)
    bound = (cols + cols / 16 + 16) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T + 1)   # as above
    if fmt == "q4_k":
        bound = bound + 4 * 2.0 ** -11 * np.abs(x).max(1).astype(np.float64)[:, None] * np.abs(w).max()
    assert (np.abs(default - x.astype(np.float64) @ w.T) <= bound).all()
    m.close()


@pytest.mark.parametrize("fmt,rows,cols", [("q8_0", 300, 640), ("q4_0", 256, 1152), ("q4_k", 290, 1280)])
@pytest.mark.parametrize("heights", [1481, 2481, 1381, 3381])
def test_two_heights_of_tiles_are_the_same_product(ops, fmt, rows, cols, heights):
    """Tiles of 64 rows behind long ones, at the edges of both: every sum in the order that tiles of one height have."""
    f = lib.FORMAT_NAMES[fmt]
    m = ops.Matrix(f, ops.synth_weights(f, rows + cols, 0.02, rows * cols), rows, cols)
    rng = np.random.default_rng(cols)
    first = heights // 1000 * 32 * (heights // 100 % 10)
    try:
        for batch in (first, first + 1, first + 64, first + 65, first + 190):
            x = rng.normal(0, 1, (batch, cols)).astype(np.float16)
            residual = rng.normal(0, 1, (batch, rows)).astype(np.float32)
            ops.set_tuning("block_gemm_form", heights % 1000)
            want = m.gemv(x, residual), m.layer_gate_up(x)
            ops.set_tuning("block_gemm_form", heights)
            assert np.array_equal(want[0], m.gemv(x, residual)) and np.array_equal(want[1], m.layer_gate_up(x)), batch
    finally:
        ops.set_tuning("block_gemm_form", 0)
    m.close()
