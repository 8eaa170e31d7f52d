"""wide_split_kernel (exact Q4_K weights, split activations, tiles of 128 x 256) against float64 at the edges of its tiles: rows of activations and of weights that leave wavefronts or
workgroups partly or wholly without work, one to many super-blocks, shares of K of unequal length, with and without a residual, behind a SiLU and without."""
import numpy as np
import pytest

import espresso_amd._lib as lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import espresso_amd.ops as o
    o.init()
    yield o
    o.set_tuning("wide_split_shares", 0)


def matrix(ops, rows, cols):
    m = ops.Matrix(lib.FORMAT_Q4_K, ops.synth_weights(lib.FORMAT_Q4_K, rows + cols, 0.02, rows * cols), rows, cols)
    return m, m.dequantize().astype(np.float64)


@pytest.mark.parametrize("rows,cols,batches", [(4, 256, (1, 129)), (256, 512, (128, 200)), (290, 1792, (33, 257)), (520, 4096, (65, 300))])
def test_products_match_float64(ops, rows, cols, batches):
    m, w = matrix(ops, rows, cols)
    rng = np.random.default_rng(cols)
    for batch in batches:
        x = rng.normal(0, 1, (batch, cols)).astype(np.float32)
        residual = rng.normal(0, 1, (batch, rows)).astype(np.float32) if batch % 2 else None
        want = x.astype(np.float64) @ w.T + (0 if residual is None else residual)
        # the activations carry 22 bits; exact products, one rounding per addition relative to the sum of the magnitudes, which scale * q and the minimum, summed apart, reach up to
        # sixteen times over
        bound = (16 * (cols + 64) * 2.0 ** -24 + 2.0 ** -21) * (np.abs(x).astype(np.float64) @ np.abs(w).T + 1)
        for shares in (1, 2, 3, 8):
            ops.set_tuning("wide_split_shares", shares)
            got = m.matmul_f32(x, residual)
            assert (np.abs(got - want) <= bound).all(), (shares, batch)
            assert np.array_equal(m.matmul_f32(x, residual), got)
    ops.set_tuning("wide_split_shares", 0)
    m.close()


@pytest.mark.parametrize("rows,cols,batch", [(64, 256, 5), (576, 768, 130), (1088, 2048, 257)])
def test_swiglu_matches_float64(ops, rows, cols, batch):
    m, w = matrix(ops, rows, cols)
    x = np.random.default_rng(batch).normal(0, 1, (batch, cols)).astype(np.float32)
    y = x.astype(np.float64) @ w.T
    gate, up = y[:, 0::2], y[:, 1::2]
    ops.set_tuning("wide_split_shares", 1)
    err = np.abs(m.matmul_f32_swiglu(x) - gate / (1 + np.exp(-gate)) * up)
    ops.set_tuning("wide_split_shares", 0)
    # gate and up carry the product's few 1e-6 (relative to its spread); d(SiLU(g) u) = SiLU'(g) u dg + SiLU(g) du
    assert (err <= 5e-6 * y.std() * (np.abs(up) + np.abs(gate) + 1)).all()
    m.close()


@pytest.mark.parametrize("planted", [np.inf, -np.inf, np.nan])
def test_what_is_not_finite_stays_in_its_row(ops, planted):
    """Rows past the end of a tile repeat the last one, steps past the end of a share its last: neither may reach another row's sum."""
    m, _ = matrix(ops, 300, 1280)
    x = np.random.default_rng(1).normal(0, 1, (131, 1280)).astype(np.float32)
    for shares in (1, 3):
        ops.set_tuning("wide_split_shares", shares)
        clean = m.matmul_f32(x)
        y = x.copy()
        y[-1, -1] = planted
        got = m.matmul_f32(y)
        assert np.array_equal(got[:-1], clean[:-1]) and not np.isfinite(got[-1]).any(), shares
    ops.set_tuning("wide_split_shares", 0)
    m.close()


def test_blocks_by_rule_are_the_blocks_without(ops):
    """A model's prompt block, whose gate | up and down take the tiles by size, against the kernels it has without them."""
    import espresso_amd.llama as ll
    import espresso_amd.synthetic as syn
    cfg = ll.MultiModelConfig(n_layer=2, n_head=16, n_kv_head=4, d_model=1024, head_dim=64, hidden_dim=8192, vocab=260, max_seq=704)
    rt, _ = syn.build_runtime(cfg, lib.FORMAT_Q4_K, seed=4, std=0.05, kv_format=lib.FORMAT_F16)
    tokens = np.random.default_rng(2).integers(0, 260, 700).astype(np.uint32)
    logits = {}
    for shares in (-1, 0, 1):
        ops.set_tuning("wide_split_shares", shares)
        rt.reset()
        logits[shares] = rt.append(tokens, want=[0, 300, 699])
    ops.set_tuning("wide_split_shares", 0)
    rt.close()
    # fp16 caches, whose last bit may fall either way
    for got in logits.values():
        assert np.abs(got - logits[-1]).max() <= 2.0 ** -9 * max(1.0, np.abs(logits[-1]).max())


@pytest.mark.parametrize("rows,cols", [(288, 1280), (512, 512)])
def test_two_heights_of_tiles_are_the_same_product(ops, rows, cols):
    """Tiles of 64 rows behind tiles of 128, at the edges of both: every sum in the order that tiles of one height have."""
    m, _ = matrix(ops, rows, cols)
    rng = np.random.default_rng(cols)
    try:
        for tiles in (1, 2):
            for batch in (128 * tiles + 1, 128 * tiles + 64, 128 * tiles + 65, 128 * tiles + 190):
                x = rng.normal(0, 1, (batch, cols)).astype(np.float32)
                residual = rng.normal(0, 1, (batch, rows)).astype(np.float32)
                ops.set_tuning("wide_split_shares", 1)
                want = m.matmul_f32(x, residual), m.matmul_f32_swiglu(x) if rows % 64 == 0 else None
                ops.set_tuning("wide_split_shares", 100 * tiles)
                assert np.array_equal(want[0], m.matmul_f32(x, residual)), (tiles, batch)
                assert want[1] is None or np.array_equal(want[1], m.matmul_f32_swiglu(x)), (tiles, batch)
    finally:
        ops.set_tuning("wide_split_shares", 0)
    m.close()
