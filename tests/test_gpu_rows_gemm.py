"""rows_gemm_kernel against float64 at the edges of its tiles: columns that leave wavefronts without work, weight rows and activation rows
around multiples of 32 and of the eight-row loads, every format, with and without a residual."""
import numpy as np
import pytest

import espresso_amd._lib as lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import espresso_amd.ops as o
    o.init()
    o.set_tuning("rows_gemm", 2)   # wherever the kernel can run
    yield o
    o.set_tuning("rows_gemm", 1)


@pytest.mark.parametrize("fmt,rows,cols", [
    ("q4_k", 33, 256), ("q4_k", 64, 2048), ("q4_k", 31, 2304), ("q4_0", 4, 64), ("q4_0", 96, 576), ("q4_0", 40, 1600), ("q8_0", 32, 128),
    ("q8_0", 68, 576), ("q8_0", 16, 4160), ("f16", 36, 64), ("f16", 60, 704), ("f16", 2, 1536),
])
def test_products_match_float64(ops, fmt, rows, cols):
    f = lib.FORMAT_NAMES[fmt]
    m = ops.Matrix(f, ops.synth_weights(f, rows + cols, 0.02, rows * cols), rows, cols)
    w = m.dequantize().astype(np.float64)
    rounded = m.dequantize().astype(np.float16).astype(np.float64)
    rng = np.random.default_rng(cols)
    off, off_rounded = [], []
    for batch in (3, 8, 9, 16, 17, 32, 33, 65):
        x = rng.normal(0, 1, (batch, cols)).astype(np.float16)
        residual = rng.normal(0, 1, (batch, rows)).astype(np.float32) if batch % 2 else None
        want = x.astype(np.float64) @ w.T + (0 if residual is None else residual)
        # products are exact (integers below 2^10 against 11-bit numbers, scales applied in fp32), sums are fp32 in some order: at most
        # one rounding per product and one per scale, each relative to the sum of the magnitudes
        bound = (cols + cols / 16 + 16) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T + 1)
        if fmt == "q4_k":   # scale * q and the minimum are summed apart: up to twice 63 * 15 steps of the super-block's scale each
            bound = bound * 16
        assert (np.abs(m.gemv(x, residual) - want) <= bound).all(), batch
        # relative to the products' root of squares, which is what rounding each of them adds up to
        spread = np.sqrt((x.astype(np.float64) ** 2) @ (w ** 2).T) + 1e-30
        x64 = x.astype(np.float64)
        off.append(((m.gemv(x) - x64 @ w.T) / spread).ravel())
        off_rounded.append(((x64 @ rounded.T - x64 @ w.T) / spread).ravel())
    # No weight is rounded: what is left is the fp32 sums' 2^-24 per addition (a lane's chain is an eighth of the row and one sum per block), eight times
    # that in Q4_K's two opposite sums.  fp16-rounded weights are off by 2^-12 / sqrt(3) each, 2^8 times the bound, wherever a weight has more than fp16's bits.
    rms = lambda parts: np.sqrt(np.mean(np.concatenate(parts) ** 2))  # noqa: E731
    limit = 2.0 ** -20 if fmt == "q4_k" else 2.0 ** -22
    assert rms(off) <= limit, rms(off)
    if fmt != "f16":
        assert rms(off_rounded) > 8 * limit, rms(off_rounded)
    m.close()


def test_gate_up_epilogue_matches_the_separate_launch(ops):
    """A two-layer model's batch step: SiLU(gate) * up in the product's epilogue and, with the kernel off, in a launch of its own."""
    import espresso_amd.llama as ll
    import espresso_amd.synthetic as syn
    cfg = ll.MultiModelConfig(n_layer=2, n_head=3, n_kv_head=3, d_model=192, head_dim=64, hidden_dim=320, vocab=260, max_seq=64)
    logits = {}
    for mode in (0, 2):
        ops.set_tuning("rows_gemm", mode)
        rt, _ = syn.build_runtime(cfg, lib.FORMAT_F16, seed=3, std=0.05, max_sequences=3)
        logits[mode] = rt.append(np.arange(45, dtype=np.uint32), want=[0, 7, 44])
        rt.close()
    ops.set_tuning("rows_gemm", 2)
    # fp16 weights are exact in both; activations are rounded to fp16 between the products, where a last bit may fall either way
    assert np.abs(logits[0] - logits[2]).max() <= 2.0 ** -10 * max(1.0, np.abs(logits[0]).max())
