"""Single steps of the layered models at widths around the ring of steps in flight (512 columns each, four or two), vocabularies of more than one round of the head's workgroups, and chains of captured
greedy steps, against the plain statement."""
import numpy as np
import pytest

import espresso_amd.layered as layered
import layered_util as lu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,ff,vocab", [(512, 300, 97), (1024, 1500, 9000), (1030, 2100, 333), (2048, 1030, 97), (2050, 4100, 97)])
@pytest.mark.parametrize("parallel", [True, False])
def test_steps_at_the_rings_edges(tmp_path, width, ff, vocab, parallel):
    if parallel:
        cfg = lu.config([lu.retention(heads=3, dim=48, vdim=72, ff=ff), lu.latent(heads=5, dim=40, ff=ff)], width=width, vocab=vocab)
    else:
        cfg = lu.sequential([lu.mamba2(heads=6, vdim=40, state=40, ff=ff), lu.attention(heads=8, dim=32, vdim=40, dims=16, ff=ff)], width=width, vocab=vocab)
    m = lu.Model(tmp_path, cfg, seed=3, gain=1.5)
    t = lu.tokens(m.cfg, 6, 3)
    want = m.logits(t)
    rt = m.runtime("bf16", max_seq=32)
    got = lu.feed(rt, t, [1] * 6)
    assert lu.error(got, want) < lu.limit("bf16")
    # captured steps: the same tokens as one step at a time
    rt.reset()
    rt.prefill(t)
    chain = [int(x) for x in rt.generate(t, 9)[0]]
    rt.reset()
    rt.prefill(t)
    alone = []
    for _ in range(9):
        alone.append(int(np.argmax(rt.logits())))
        rt.advance(alone[-1])
    assert chain == alone


# Rows of 36865 to 38400 columns: whole steps of 512 within 150 KB, whole turns of four beyond it
@pytest.mark.parametrize("ff", [36700, 37300, 37500])
@pytest.mark.parametrize("parallel", [True, False])
def test_the_longest_rows(tmp_path, ff, parallel):
    if parallel:
        cfg = lu.config([lu.retention(heads=3, dim=48, vdim=72, ff=ff), lu.latent(heads=5, dim=40, ff=ff)], width=64, vocab=97)
    else:
        cfg = lu.sequential([lu.mamba2(heads=6, vdim=40, state=40, ff=ff), lu.attention(heads=8, dim=32, vdim=40, dims=16, ff=ff)], width=64, vocab=97)
    m = lu.Model(tmp_path, cfg, seed=3, gain=1.5)
    t = lu.tokens(m.cfg, 5, 3)
    want = m.logits(t)
    rt = m.runtime("bf16", max_seq=32)
    assert lu.error(lu.feed(rt, t, [1] * 5), want) < lu.limit("bf16")


# Slices of latent attention merged in one request (32 and fewer of a rank of up to 512) and in several
@pytest.mark.parametrize("rank,keys", [(64, 1), (64, 33), (512, 65), (576, 40), (960, 1100), (128, 2100)])
def test_slices_of_latents_merged(tmp_path, rank, keys):
    m = lu.Model(tmp_path, lu.config([lu.latent(heads=3, dim=40, kv_rank=rank, window=4096, ff=64)], width=96, vocab=61), seed=5, gain=1.5)
    t = lu.tokens(m.cfg, keys + 2, 7)
    want = m.logits(t)
    rt = m.runtime("bf16", max_seq=4096)
    got = lu.feed(rt, t, [200] * (keys // 200) + ([keys % 200] if keys % 200 else []) + [1])
    assert lu.error(got[-2:], want[-2:]) < lu.limit("bf16")


# Groups of query heads whose sums meet together, fewer than a full set of them too, long heads beside eight queries; slices in one request and in several
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,keys", [(4, 4, 16, 24, 1), (6, 3, 32, 40, 33), (3, 1, 64, 128, 300), (10, 2, 40, 72, 70), (7, 1, 136, 16, 290), (8, 1, 480, 320, 40), (16, 2, 1024, 1024, 36)])
def test_heads_of_a_group_together(tmp_path, heads, kv_heads, dim, vdim, keys):
    m = lu.Model(tmp_path, lu.sequential([lu.attention(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, dims=16, window=512, ff=64)], width=96, vocab=61), seed=5, gain=1.5)
    t = lu.tokens(m.cfg, keys + 2, 7)
    want = m.logits(t)
    rt = m.runtime("bf16", max_seq=512)
    got = lu.feed(rt, t, [200] * (keys // 200) + ([keys % 200] if keys % 200 else []) + [1])
    assert lu.error(got[-2:], want[-2:]) < lu.limit("bf16")
