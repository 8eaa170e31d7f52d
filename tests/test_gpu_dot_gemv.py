"""The dot-product GEMV: what it requests before the arithmetic, at the edges of its rounds (64 items per lane round), of the
groups a thread keeps in registers, and of its row pairs."""
import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_full_size import oracle_from_packed

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mods():
    import espresso_amd.llama as ll
    import espresso_amd.ops as ops
    import espresso_amd.synthetic as syn
    ops.init()
    yield ll, ops, syn
    for key in ("q40_mfma", "q80_mfma"):
        ops.set_tuning(key, -1)


ITEM = {orc.FMT_Q4_0: 32, orc.FMT_Q8_0: 16, orc.FMT_F16: 8, orc.FMT_F32: 4}


@pytest.mark.parametrize("fmt", list(ITEM))
@pytest.mark.parametrize("items", [2, 64, 66, 128, 130, 256, 258, 520])
def test_rounds_of_items(mods, fmt, items):
    _, ops, _ = mods
    cols = items * ITEM[fmt]
    if cols % 32:
        cols += 32 - cols % 32
    ops.set_tuning("q40_mfma", 0)
    ops.set_tuning("q80_mfma", 0)
    rng = np.random.default_rng(items)
    for rows in (1, 7, 9):
        w = rng.normal(0, 0.02, (rows, cols)).astype(np.float32)
        packed = orc.quantize(fmt, w) if fmt in (orc.FMT_Q4_0, orc.FMT_Q8_0) else (w.astype(np.float16) if fmt == orc.FMT_F16 else w).view(np.uint8)
        m = ops.Matrix(fmt, packed, rows, cols)
        deq = m.dequantize().astype(np.float64).reshape(rows, cols)
        for batch in (1, 2):
            x = rng.normal(0, 1, (batch, cols)).astype(np.float16)
            res = rng.normal(0, 1, (batch, rows)).astype(np.float32)
            want = x.astype(np.float64) @ deq.T
            # exact products; a lane adds at most 4 x 32 x items / 64 of them and six partial sums, every addition within 2^-24
            bound = 2.0 ** -23 * (np.abs(x.astype(np.float64)) @ np.abs(deq).T) * (8 + cols / 64) + 1e-6
            if fmt == orc.FMT_Q4_0:   # nibble - 8 is exact, its sums of 32 are scaled once
                bound = bound * 2
            assert (np.abs(m.gemv(x) - want) <= bound).all(), (rows, batch)
            assert (np.abs(m.gemv(x, res) - (want + res)) <= bound + 2.0 ** -22 * np.abs(want + res)).all(), (rows, batch)
        m.close()


def test_a_refused_product_leaves_nothing_to_the_next(mods):
    """Two rows of 40960 columns do not fit a workgroup's LDS; the call that follows the refusal is not blamed for it."""
    _, ops, _ = mods
    from espresso_amd._lib import EspressoError
    wide = ops.Matrix(orc.FMT_F16, np.zeros((2, 40960), np.float16).view(np.uint8), 2, 40960)
    w = np.random.default_rng(0).normal(0, 1, (8, 64)).astype(np.float16)
    m = ops.Matrix(orc.FMT_F16, w.view(np.uint8), 8, 64)
    x = np.random.default_rng(1).normal(0, 1, (1, 64)).astype(np.float16)
    for _ in range(2):
        with pytest.raises(EspressoError):
            wide.gemv(np.zeros((2, 40960), np.float16))
        assert np.abs(m.gemv(x) - x.astype(np.float64) @ w.astype(np.float64).T).max() <= 1e-4
    assert (wide.gemv(np.zeros((1, 40960), np.float16)) == 0).all()
    m.close()
    wide.close()


@pytest.mark.parametrize("cols", [4, 8, 12, 252, 260, 1028, 4092, 5124])
def test_fp32_rows_of_whole_fours(mods, cols):
    """Every multiple of four columns is taken: rows of the activations start at any multiple of eight bytes, and the last four columns count."""
    _, ops, _ = mods
    rng = np.random.default_rng(cols)
    for rows in (1, 6, 9):
        w = rng.normal(0, 0.02, (rows, cols)).astype(np.float32)
        w[:, -4:] *= 50
        m = ops.Matrix(orc.FMT_F32, w.view(np.uint8), rows, cols)
        for batch in (1, 2, 3):
            x = rng.normal(0, 1, (batch, cols)).astype(np.float16)
            res = rng.normal(0, 1, (batch, rows)).astype(np.float32)
            want = x.astype(np.float64) @ w.astype(np.float64).T
            bound = 2.0 ** -23 * (np.abs(x.astype(np.float64)) @ np.abs(w.astype(np.float64)).T) * (8 + cols / 64) + 1e-6   # as above
            assert (np.abs(m.gemv(x) - want) <= bound).all(), (rows, batch)
            assert (np.abs(m.gemv(x, res) - (want + res)) <= bound + 2.0 ** -22 * np.abs(want + res)).all(), (rows, batch)
        m.close()


# norm rows of up to 512 groups of eight stay in registers; attention states beyond one group per thread; odd pair counts
@pytest.mark.parametrize("fmt,d,heads,kv,hidden", [(orc.FMT_F16, 576, 9, 3, 1536), (orc.FMT_Q8_0, 4352, 34, 2, 608), (orc.FMT_Q4_0, 2304, 18, 2, 4224),
                                                   (orc.FMT_F16, 64, 1, 1, 72)])
def test_decode_matches_oracle(mods, fmt, d, heads, kv, hidden):
    ll, ops, syn = mods
    ops.set_tuning("q40_mfma", -1)
    ops.set_tuning("q80_mfma", -1)
    cfg = ll.MultiModelConfig(n_layer=1, n_head=heads, n_kv_head=kv, d_model=d, head_dim=d // heads, hidden_dim=hidden, vocab=520, max_seq=32)
    g, packed = syn.build_runtime(cfg, fmt, seed=d, keep_packed=True)
    o = oracle_from_packed(cfg, packed, fmt, 1, False, 32)
    for i, t in enumerate((3, 500, 44, 17, 9)):
        g.advance(t)
        o.advance(t)
        want = o.logits()
        # activations are rounded to fp16 in front of every product
        assert np.abs(g.logits() - want).max() <= 2.0 ** -8 * max(1.0, np.abs(want).max()), i
    g.close()
