"""stream_gemm_kernel at the edges of its tiles: activation rows up to 32, weight rows that end within a tile, columns that leave wavefronts short of units or without any."""
import numpy as np
import pytest

import espresso_amd._lib as lib
from test_gpu_block_gemm import check_kept

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import espresso_amd.ops as o
    o.init()
    yield o


@pytest.fixture(autouse=True)
def by_size_again(ops):
    yield
    for key in ("rows_gemm", "stream_gemm"):
        ops.set_tuning(key, 1)


@pytest.mark.parametrize("fmt,rows,cols", [("q8_0", 4, 64), ("q8_0", 36, 192), ("q8_0", 290, 1408), ("q8_0", 40, 2304), ("q4_0", 4, 128), ("q4_0", 300, 1152), ("q4_0", 72, 8320)])
def test_products_keep_their_weights(ops, fmt, rows, cols):
    """In one launch at any size, and in shares of K up to 32 rows."""
    f = lib.FORMAT_NAMES[fmt]
    m = ops.Matrix(f, ops.synth_weights(f, rows + cols, 0.02, rows * cols), rows, cols)
    rng = np.random.default_rng(cols)
    ops.set_tuning("stream_gemm", 2)
    ops.set_tuning("rows_gemm", 2)
    check_kept(m, lambda x, r: m.layer_product(x, r), (3, 8, 17, 31, 32), rng)
    if cols % 128 == 0:
        ops.set_tuning("rows_gemm", 0)
        check_kept(m, lambda x, r: m.layer_product(x, r, shares=True), (3, 9, 31, 32), rng)
    m.close()


@pytest.mark.parametrize("fmt,rows,cols,batches", [
    ("q8_0", 2304, 768, (12, 32)), ("q8_0", 576, 1024, (5, 31)), ("q8_0", 4090, 1024, (3,)), ("q4_0", 4096, 768, (9, 31)), ("q4_0", 2048, 1024, (3, 32)),
])
def test_one_launch_adds_as_before(ops, fmt, rows, cols, batches):
    """Products that were one launch of rows_gemm.hip: the same shares of K in the same order, so the same bits, with the SiLU of gate and up too."""
    f = lib.FORMAT_NAMES[fmt]
    m = ops.Matrix(f, ops.synth_weights(f, rows + cols, 0.02, rows * cols), rows, cols)
    rng = np.random.default_rng(cols)
    for batch in batches:
        x = rng.normal(0, 1, (batch, cols)).astype(np.float16)
        residual = rng.normal(0, 1, (batch, rows)).astype(np.float32)
        got = m.layer_product(x, residual, shares=True), m.layer_gate_up(x)
        ops.set_tuning("stream_gemm", 0)
        assert np.array_equal(got[0], m.layer_product(x, residual, shares=True)) and np.array_equal(got[1], m.layer_gate_up(x)), batch
        ops.set_tuning("stream_gemm", 1)
    m.close()


@pytest.mark.parametrize("fmt", ["q8_0", "q4_0"])
@pytest.mark.parametrize("rows,cols,batches", [(2048, 2048, (5, 17, 32)), (2570, 2048, (31,)), (3072, 3072, (9, 32)), (2048, 5632, (9, 32))])
def test_shares_of_small_products(ops, fmt, rows, cols, batches):
    """What the layers' products take by size, in shares of K that the next kernel adds: not block_gemm.hip's, which adds in another order, and as exact."""
    f = lib.FORMAT_NAMES[fmt]
    m = ops.Matrix(f, ops.synth_weights(f, rows + cols, 0.02, rows * cols), rows, cols)
    check_kept(m, lambda x, r: m.layer_product(x, r, shares=True), batches, np.random.default_rng(cols))
    m.close()
