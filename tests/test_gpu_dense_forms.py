"""bf16 products of layered models in every tile: rows of activations around the tiles' edges, feed-forwards and mixers whose columns end inside a tile of 256."""
import numpy as np
import pytest

import espresso_amd.layered as layered
import layered_util as lu

pytestmark = pytest.mark.gpu

TILES = [(64, 128), (64, 256), (128, 128), (128, 256), (192, 128), (192, 256), (256, 128), (256, 256)]


@pytest.mark.parametrize("config", [
    lu.config([lu.latent(heads=5, dim=40, ff=100), lu.retention(heads=3, dim=48, vdim=72, ff=333)], width=200, vocab=300),
    lu.sequential([lu.mamba2(heads=6, vdim=40, state=40, ff=260), lu.attention(heads=8, dim=32, vdim=40, dims=16, ff=90)], width=130, vocab=140),
])
def test_blocks_in_every_tile(tmp_path, config):
    import espresso_amd.ops as ops
    m = lu.Model(tmp_path, config, seed=11, gain=1.5)
    t = lu.tokens(m.cfg, 321, 3)
    want = m.logits(t)
    rt = m.runtime("bf16", max_seq=330)
    layered.set_min_block_rows(rt, 1)
    try:
        for bm, bn in TILES:
            ops.set_tuning("dense_gemm_form", 10000 * bm + 10 * bn + 1)
            for portions in ([321], [65, 256], [1, 63, 129, 128]):
                rt.reset()
                assert lu.error(lu.feed(rt, t, portions), want) < lu.limit("bf16"), (bm, bn, portions)
    finally:
        ops.set_tuning("dense_gemm_form", 0)
        layered.set_min_block_rows(rt, 3)
