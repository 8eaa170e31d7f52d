"""Products with fp16 matrices against float64 at the edges of the tiles: every form, rows of activations and of weights that leave wavefronts or workgroups partly or wholly without
work, shares of K of unequal length, one to many steps of 64 columns, with and without a residual."""
import numpy as np
import pytest

import espresso_amd._lib as lib

pytestmark = pytest.mark.gpu

TILES = [(64, 128), (64, 256), (128, 128), (128, 256), (192, 128), (192, 256), (256, 128), (256, 256)]


@pytest.fixture(scope="module")
def ops():
    import espresso_amd.ops as o
    o.init()
    yield o
    o.set_tuning("wide_gemm_form", 0)


def matrix(ops, rng, rows, cols):
    w = rng.normal(0, 0.02, (rows, cols)).astype(np.float16)
    return ops.Matrix(lib.FORMAT_NAMES["f16"], w.view(np.uint8), rows, cols), w.astype(np.float64)


@pytest.mark.parametrize("rows,cols,batches", [(4, 64, (3, 65)), (129, 192, (64, 193)), (300, 704, (9, 257)), (256, 1088, (256, 300)), (515, 2112, (31, 130)), (96, 1472, (1100,))])
def test_products_match_float64(ops, rows, cols, batches):
    rng = np.random.default_rng(cols)
    m, w = matrix(ops, rng, rows, cols)
    for batch in batches:
        x = rng.normal(0, 1, (batch, cols)).astype(np.float16)
        residual = rng.normal(0, 1, (batch, rows)).astype(np.float32) if batch % 2 else None
        want = x.astype(np.float64) @ w.T + (0 if residual is None else residual)
        # exact products, fp32 sums in some order: one rounding per addition, relative to the sum of the magnitudes
        bound = (cols + 16) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T + 1)
        for form in [0] + [10000 * bm + 10 * bn + shares for bm, bn in TILES for shares in (1, 2, 3, 8)]:
            ops.set_tuning("wide_gemm_form", form)
            got = m.gemv(x, residual)
            assert (np.abs(got - want) <= bound).all(), (form, batch)
            assert np.array_equal(m.gemv(x, residual), got)
    ops.set_tuning("wide_gemm_form", 0)
    m.close()


# weight rows that end inside a tile, between two wavefronts and at a tile's end; fewer rows of activations than a tile, ragged ones, whole tiles
@pytest.mark.parametrize("rows,cols,batches", [(134, 192, (3, 65, 193)), (522, 448, (64, 130, 257)), (256, 64, (9, 300))])
def test_gate_up_matches_float64(ops, rows, cols, batches):
    """SiLU(gate) * up in the product's epilogue (one share of K) and by the launch that adds planes (more), every tile."""
    rng = np.random.default_rng(rows)
    w = rng.normal(0, 2.0 / np.sqrt(cols), (rows, cols)).astype(np.float16)   # gates of both signs, up to six or so
    m = ops.Matrix(lib.FORMAT_NAMES["f16"], w.view(np.uint8), rows, cols)
    w = w.astype(np.float64)
    for batch in batches:
        x = rng.normal(0, 1, (batch, cols)).astype(np.float16)
        y = x.astype(np.float64) @ w.T
        gate, up = y[:, 0::2], y[:, 1::2]
        silu = gate / (1 + np.exp(-gate))
        want = silu * up
        # products as above; SiLU's slope is at most 1.1; its fp32 forms are off by 2^-22 of the gate, and the result is rounded to fp16 once
        off = (cols + 16) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T + 1)
        bound = (1.1 * off[:, 0::2] + 2.0 ** -22 * np.abs(gate)) * (np.abs(up) + off[:, 1::2]) + np.abs(silu) * off[:, 1::2] + 2.0 ** -11 * np.abs(want) + 2.0 ** -25
        for form in [0] + [10000 * bm + 10 * bn + shares for bm, bn in TILES for shares in (1, 2, 3)]:
            ops.set_tuning("wide_gemm_form", form)
            got = m.layer_gate_up(x).astype(np.float64)
            assert (np.abs(got - want) <= bound).all(), (form, batch)
    ops.set_tuning("wide_gemm_form", 0)
    m.close()


@pytest.mark.parametrize("planted", [np.inf, -np.inf, np.nan])
def test_what_is_not_finite_stays_in_its_row(ops, planted):
    """Rows past the end of a tile repeat the last one, steps past the end of a share its last: neither may reach another row's sum."""
    rows, cols, batch = 70, 320, 67
    rng = np.random.default_rng(1)
    m, _ = matrix(ops, rng, rows, cols)
    x = rng.normal(0, 1, (batch, cols)).astype(np.float16)
    for form in (0, 641283, 641281, 2562561):
        ops.set_tuning("wide_gemm_form", form)
        clean = m.gemv(x)
        y = x.copy()
        y[-1, -1] = planted
        got = m.gemv(y)
        assert np.array_equal(got[:-1], clean[:-1]) and not np.isfinite(got[-1]).any(), form
    ops.set_tuning("wide_gemm_form", 0)
    m.close()


def test_a_form_without_room_for_its_planes_is_by_size(ops):
    """Eight shares of 512 x 1100 sums are more than a product's workspace."""
    rng = np.random.default_rng(3)
    m, _ = matrix(ops, rng, 1100, 1024)
    x = rng.normal(0, 1, (512, 1024)).astype(np.float16)
    by_size = m.layer_product(x)
    for form in (641288, 2562568):
        ops.set_tuning("wide_gemm_form", form)
        assert np.array_equal(m.layer_product(x), by_size), form
    ops.set_tuning("wide_gemm_form", 0)
    m.close()
