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
