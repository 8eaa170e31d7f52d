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


FORMS = [181, 182, 141, 143, 121, 128, 281, 242, 221, 381, 341, 322, 481, 484, 441, 443]   # row tiles, wavefronts along the weights, shares of K


@pytest.mark.parametrize("fmt,rows,cols", [
    ("q4_k", 256, 256), ("q4_k", 33, 2304), ("q4_k", 290, 4096), ("q4_0", 4, 128), ("q4_0", 300, 1152), ("q4_0", 64, 2688),
    ("q8_0", 258, 128), ("q8_0", 30, 1408), ("q8_0", 520, 640), ("f16", 70, 384), ("f16", 272, 1664),
])
def test_products_match_float64(ops, fmt, rows, cols):
    f = lib.FORMAT_NAMES[fmt]
    m = ops.Matrix(f, ops.synth_weights(f, rows + cols, 0.02, rows * cols), rows, cols)
    w = m.dequantize().astype(np.float16).astype(np.float64)   # what reaches the matrix cores: each weight rounded to fp16 once
    rng = np.random.default_rng(cols)
    for form in FORMS if fmt != "f16" else FORMS[::2]:
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
