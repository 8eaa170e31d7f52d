"""block_split_kernel (exact Q4_K weights, split activations) against float64 at the edges of its tiles, every form, and short blocks of models whose long blocks
take other kernels against single steps."""
import numpy as np
import pytest

import espresso_amd._lib as lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import espresso_amd.ops as o
    o.init()
    yield o
    o.set_tuning("block_split_form", 0)


@pytest.mark.parametrize("rows,cols", [(256, 256), (4, 2304), (290, 1536), (520, 4096)])
def test_matmul_f32_rounds_no_operand(ops, rows, cols):
    m = ops.Matrix(lib.FORMAT_Q4_K, ops.synth_weights(lib.FORMAT_Q4_K, rows + cols, 0.02, rows * cols), rows, cols)
    w = m.dequantize().astype(np.float64)
    rng = np.random.default_rng(cols)
    for form in (121, 122, 141, 143, 181, 188, 241, 242, 281, 284, 381, 383):
        ops.set_tuning("block_split_form", form)
        for batch in (3, 31, 33, 64, 97, 161):
            x = rng.normal(0, 1, (batch, cols)).astype(np.float32)
            residual = rng.normal(0, 1, (batch, rows)).astype(np.float32) if batch % 2 else None
            want = x.astype(np.float64) @ w.T + (0 if residual is None else residual)
            # the activations carry 22 bits; exact products, one rounding per addition relative to the sum of the magnitudes, which scale * q and the minimum,
            # summed apart, reach up to sixteen times over
            bound = (16 * (cols + 64) * 2.0 ** -24 + 2.0 ** -21) * (np.abs(x).astype(np.float64) @ np.abs(w).T + 1)
            assert (np.abs(m.matmul_f32(x, residual) - want) <= bound).all(), (form, batch)
    ops.set_tuning("block_split_form", 0)
    m.close()


@pytest.mark.parametrize("heads,kv_heads,head_dim,kv", [(24, 8, 128, lib.FORMAT_F16), (16, 16, 64, lib.FORMAT_F32), (16, 2, 64, lib.FORMAT_F32)])
def test_short_blocks_are_the_steps(ops, heads, kv_heads, head_dim, kv):
    """Q4_K models whose long blocks round their operands: turns of 5 to 31 tokens keep activations, weights and attention as the steps do (of widths whose steps carry
    activations in two parts)."""
    import espresso_amd.llama as ll
    import espresso_amd.synthetic as syn
    cfg = ll.MultiModelConfig(n_layer=2, n_head=heads, n_kv_head=kv_heads, d_model=1024, head_dim=head_dim, hidden_dim=3072, vocab=260, max_seq=128)
    rt, _ = syn.build_runtime(cfg, lib.FORMAT_Q4_K, seed=3, std=0.05, kv_format=kv)
    tokens = np.random.default_rng(1).integers(0, 260, 80).astype(np.uint32)
    for form in (0, 121, 181, -1):
        ops.set_tuning("block_split_form", form)
        for prefix, count in ((0, 5), (0, 31), (37, 9), (44, 17)):
            rt.reset()
            if prefix:
                rt.prefill(tokens[:prefix])
            block = rt.append(tokens[prefix:prefix + count], want=range(count))
            rt.set_visible(prefix)
            steps = []
            for t in tokens[prefix:prefix + count]:
                rt.advance(int(t))
                steps.append(rt.logits())
            # contexts, and caches where they are fp16, round the same way in both, where a last bit may fall either way: 1.5 to 4.2e-4 of the logits' size; rounded weights
            # would be some 1e-3 off (test_gpu_block_gemm.py)
            want = np.stack(steps)
            assert np.sqrt(np.mean((block - want) ** 2)) <= 2.0 ** -11 * np.sqrt(np.mean(want ** 2)), (form, prefix, count)
            assert np.abs(block - want).max() <= 2.0 ** -9 * max(1.0, np.abs(want).max()), (form, prefix, count)
    ops.set_tuning("block_split_form", 0)
    rt.close()


def test_gate_up_forms_agree(ops):
    """SiLU(gate) * up as split rows with their sums, ragged rows: every form against the whole-tile kernel."""
    import espresso_amd.llama as ll
    import espresso_amd.synthetic as syn
    cfg = ll.MultiModelConfig(n_layer=2, n_head=16, n_kv_head=4, d_model=1024, head_dim=64, hidden_dim=3072, vocab=260, max_seq=256)
    rt, _ = syn.build_runtime(cfg, lib.FORMAT_Q4_K, seed=4, std=0.05, kv_format=lib.FORMAT_F16)
    tokens = np.random.default_rng(2).integers(0, 260, 161).astype(np.uint32)
    logits = {}
    for form in (-1, 0, 121, 141, 181, 241, 281, 381):
        ops.set_tuning("block_split_form", form)
        rt.reset()
        logits[form] = rt.append(tokens, want=[0, 40, 160])
    ops.set_tuning("block_split_form", 0)
    rt.close()
    # fp16 caches, whose last bit may fall either way
    for form, got in logits.items():
        assert np.abs(got - logits[-1]).max() <= 2.0 ** -9 * max(1.0, np.abs(logits[-1]).max()), form
