"""Turns of 5 to 31 tokens: one block or the steps it stands for, whichever is faster behind what is cached."""
import numpy as np
import pytest

import espresso_amd._lib as lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mods():
    import espresso_amd.llama as ll
    import espresso_amd.ops as ops
    import espresso_amd.synthetic as syn
    ops.init()
    return ll, ops, syn


@pytest.mark.parametrize("fmt,kv,kv_heads", [("q8_0", lib.FORMAT_F32, 12), ("f16", lib.FORMAT_F16, 4), ("q4_k", lib.FORMAT_F16, 4)])
def test_few_tokens_behind_many_keys_are_steps(mods, fmt, kv, kv_heads):
    """A block's attention has one workgroup for all keys of a query head, a step's shares them: five tokens behind 12000 keys took twice as long as a block (fp32 caches)."""
    ll, ops, syn = mods
    cfg = ll.MultiModelConfig(n_layer=2, n_head=12, n_kv_head=kv_heads, d_model=768, head_dim=64, hidden_dim=2304, vocab=260, max_seq=12288)
    rt, _ = syn.build_runtime(cfg, lib.FORMAT_NAMES[fmt], seed=3, std=0.05, kv_format=kv)
    tokens = np.random.default_rng(1).integers(0, 260, 12000 + 31).astype(np.uint32)
    rt.prefill(tokens[:12000])
    ll.set_kernel_timing(rt, True)
    for prefix, count, passes in [(40, 5, 0), (12000, 5, 3), (12000, 6, 3), (12000, 31, 0), (500, 31, 0), (12000, 4, 2)]:
        rt.set_visible(prefix)
        ll.kernel_times(rt)
        rt.append(tokens[prefix:prefix + count])
        assert rt.visible() == prefix + count
        assert ll.kernel_times(rt)["qkv"]["launches"] == cfg.n_layer * passes, (prefix, count)   # a block's products are not among them
    rt.close()
