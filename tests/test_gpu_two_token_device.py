"""The exact two-token loop with its passes on the device (one captured graph per pass, no host decision in between)
against the same loop driven from the host (graph replay switched off on the target): the same tokens, the same six
counters of the reference loop (RealModelInferenceEngine.swift:6109-6186) and the same state left in both models,
for drafts that never, sometimes and always agree, with stop tokens, odd and even budgets and the end of the context."""
import numpy as np
import pytest

import model_util as mu
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

BASE = dict(n_head=4, n_kv_head=2, d_model=256, head_dim=64, hidden_dim=512, vocab=512)
COUNTERS = ("passes", "committed_total", "accepted_total", "reference_passes", "reference_committed_total", "reference_accepted_total")


@pytest.fixture(scope="module")
def llama():
    import espresso_amd.llama as ll
    import espresso_amd.ops as o
    o.init()
    return ll


def build(ll, packed, fmt, n_layer, max_seq, eos=-1):
    cfg = ll.MultiModelConfig(n_layer=n_layer, max_seq=max_seq, eos_token=eos, **BASE)
    rt = ll.LlamaRuntime(cfg)
    ll.load_packed_weights(rt, dict(packed, layers=packed["layers"][:n_layer]), fmt)
    return rt


def weights(fmt, seed, n_layer, upper_scale=1.0):
    """Random model whose layers above the first are scaled by `upper_scale` in their output projections: 0 makes the first layer
    alone an exact draft of the whole model, small values a draft that agrees most of the time."""
    ocfg = orc.LlamaConfig(gemv_inputs_fp16=True, n_layer=n_layer, max_seq=64, **BASE)
    w = mu.random_weights(ocfg, seed, std=0.08)
    for L in w["layers"][1:]:
        L["wo"] *= upper_scale
        L["w2"] *= upper_scale
    return mu.pack_weights(w, fmt)[0]


def both_ways(ll, target, draft, prompt, budget, reference_accounting=True):
    results = []
    for on_device in (True, False):
        ll.set_graph_replay(target, on_device)
        target.reset(); draft.reset()
        tokens, st = ll.generate_two_token(target, draft, prompt, budget, reference_accounting)
        results.append((tokens, {k: st[k] for k in COUNTERS}, target.visible(), draft.visible(), target.last_hidden(), draft.last_hidden(),
                        target.select_greedy(), draft.select_greedy()))
    ll.set_graph_replay(target, True)
    dev, host = results
    assert dev[0] == host[0]
    assert dev[1] == host[1], (dev[1], host[1])
    assert dev[2:4] == host[2:4]                                     # visible token counts of target and draft
    assert np.array_equal(dev[4], host[4]) and np.array_equal(dev[5], host[5])   # kept hidden states, bit for bit
    assert dev[6:] == host[6:]
    return dev[0], dev[1]


@pytest.mark.parametrize("fmt", [orc.FMT_Q8_0, orc.FMT_Q4_K])
def test_device_passes_equal_the_host_loop(llama, fmt):
    prompt = [7, 8, 9, 10, 11]
    seen = set()
    for label, upper in (("never agrees", None), ("sometimes", 0.15), ("always", 0.0)):
        if upper is None:
            target = build(llama, weights(fmt, 21, 3), fmt, 3, 64)
            draft = build(llama, weights(fmt, 22, 1), fmt, 1, 64)
        else:
            packed = weights(fmt, 23, 3, upper)
            target, draft = build(llama, packed, fmt, 3, 64), build(llama, packed, fmt, 1, 64)
        plain = target.generate(prompt, 50)[0]
        for budget in (1, 2, 3, 4, 5, 8, 21, 50):
            for ref in (True, False):
                tokens, st = both_ways(llama, target, draft, prompt, budget, ref)
                assert tokens == plain[:budget], (label, budget)
                if budget == 50 and ref:
                    rate = st["accepted_total"] / st["passes"]
                    seen.add(label)
                    if label == "never agrees": assert rate < 0.2
                    if label == "always":      # 49 tokens after the first: 24 accepted passes and a last pass with one token of budget
                        assert (st["passes"], st["accepted_total"], st["committed_total"]) == (25, 24, 49)
                    if label == "sometimes": assert 0.1 < rate < 1.0, rate
        target.close(); draft.close()
    assert seen == {"never agrees", "sometimes", "always"}


def test_stop_token_and_context_end_on_the_device(llama):
    fmt = orc.FMT_Q8_0
    packed = weights(fmt, 23, 3, 0.15)
    prompt = [7, 8, 9, 10, 11]
    probe = build(llama, packed, fmt, 3, 64)
    plain = probe.generate(prompt, 40)[0]
    probe.close()
    # every position of the stream once as the stop token: the stop may fall on the first or the second token of a pass
    for stop_at in range(0, 12):
        eos = plain[stop_at]
        first = plain.index(eos)
        target, draft = build(llama, packed, fmt, 3, 64, eos=eos), build(llama, packed, fmt, 1, 64, eos=eos)
        tokens, _ = both_ways(llama, target, draft, prompt, 40)
        assert tokens == plain[:first + 1]
        target.close(); draft.close()
    # the context ends before the budget does (prompt 5 + generated tokens fill max_seq)
    for max_seq in (12, 13, 20):
        target, draft = build(llama, packed, fmt, 3, max_seq), build(llama, packed, fmt, 1, max_seq)
        tokens, _ = both_ways(llama, target, draft, prompt, 40)
        assert tokens == plain[:max_seq - len(prompt)]
        target.close(); draft.close()
    # a draft with a shorter context than the target bounds the loop as well (:6040-6047)
    target, draft = build(llama, packed, fmt, 3, 64), build(llama, packed, fmt, 1, 17)
    tokens, _ = both_ways(llama, target, draft, prompt, 40)
    assert tokens == plain[:17 - len(prompt)]
    target.close(); draft.close()


def build_batch(ll, packed, fmt, n_layer, max_seq, n_seq):
    cfg = ll.MultiModelConfig(n_layer=n_layer, max_seq=max_seq, **BASE)
    rt = ll.LlamaRuntime(cfg, max_sequences=n_seq)
    ll.load_packed_weights(rt, dict(packed, layers=packed["layers"][:n_layer]), fmt)
    return rt


@pytest.mark.parametrize("n_seq", [1, 3, 16])
def test_lock_step_loops_on_the_device_equal_the_host_loops(llama, n_seq):
    """generate_batch (plain greedy and the exact two-token loop over several sequences): passes replayed as graphs with the
    per-sequence variables on the device against the host-driven loops - the same streams, counters and visible counts."""
    fmt = orc.FMT_Q8_0
    rng = np.random.default_rng(n_seq)
    prompts = [rng.integers(0, BASE["vocab"], int(rng.integers(3, 9))).astype(np.uint32) for _ in range(n_seq)]
    for label, upper in (("never agrees", None), ("sometimes", 0.15), ("always", 0.0)):
        if upper is None:
            target = build_batch(llama, weights(fmt, 21, 3), fmt, 3, 64, n_seq)
            draft = build_batch(llama, weights(fmt, 22, 1), fmt, 1, 64, n_seq)
        else:
            packed = weights(fmt, 23, 3, upper)
            target, draft = build_batch(llama, packed, fmt, 3, 64, n_seq), build_batch(llama, packed, fmt, 1, 64, n_seq)
        for budget in (1, 2, 3, 4, 9, 30):
            runs = {}
            for on_device in (True, False):
                for d in (None, draft):
                    llama.set_graph_replay(target, on_device)
                    target.reset(); draft.reset()
                    toks, st = llama.generate_batch(target, prompts, budget, draft=d)
                    runs[(on_device, d is not None)] = (toks, (st["passes"], st["committed_total"], st["accepted_total"]),
                                                        [target.visible(s) for s in range(n_seq)], [draft.visible(s) for s in range(n_seq)])
            llama.set_graph_replay(target, True)
            assert runs[(True, False)] == runs[(False, False)], (label, budget, "plain greedy")
            assert runs[(True, True)] == runs[(False, True)], (label, budget, "two-token")
            assert runs[(True, True)][0] == runs[(True, False)][0]                  # the exact loop gives the greedy streams
            assert all(len(t) == budget for t in runs[(True, True)][0])
            if label == "always" and budget == 30:
                passes, committed, accepted = runs[(True, True)][1]
                assert accepted == 14 * n_seq and committed == 29 * n_seq and passes == 15
        target.close(); draft.close()


def test_device_loop_session_is_reused_and_rebuilt(llama):
    """The target keeps the loop's device state, log and captured passes between calls: the same pair again (other budgets, long
    enough for the four-pass graph and too short for it), another draft, the first draft again, and a pair whose kernels changed
    (merged attention switched off and on) all give the host-driven loop's result."""
    fmt = orc.FMT_F16
    packed = weights(fmt, 31, 3, upper_scale=0.05)
    other = weights(fmt, 32, 3, upper_scale=1.0)
    target = build(llama, packed, fmt, 3, 64)
    draft_a, draft_b = build(llama, packed, fmt, 1, 64), build(llama, other, fmt, 1, 64)
    prompt = [7, 8, 9, 10, 11]
    seen = []
    for draft, budget in ((draft_a, 40), (draft_a, 9), (draft_a, 33), (draft_b, 40), (draft_a, 40), (draft_b, 5)):
        tokens, _ = both_ways(llama, target, draft, prompt, budget)
        seen.append(tokens)
    assert seen[0] == seen[4] and seen[0][:9] == seen[1] and seen[3][:5] == seen[5] and seen[0] == seen[3]   # exact: the draft does not matter
    for enabled in (False, True):
        llama.set_merged_attention(draft_a, enabled)
        llama.set_merged_attention(target, enabled)
        tokens, _ = both_ways(llama, target, draft_a, prompt, 40)
        assert tokens == seen[0]
    for rt in (target, draft_a, draft_b):
        rt.close()


@pytest.mark.parametrize("fmt", [orc.FMT_Q8_0, orc.FMT_F16])
@pytest.mark.parametrize("n_seq", [1, 2, 3, 16])
def test_first_tokens_of_a_batch_are_those_of_its_sequences(llama, fmt, n_seq):
    """The head over the kept rows of all sequences at once against one sequence at a time (margins of 1e-3 and more)."""
    rt = build_batch(llama, weights(fmt, 31, 2), fmt, 2, 64, n_seq)
    rng = np.random.default_rng(n_seq)
    prompts = [rng.integers(0, BASE["vocab"], 3 + s % 5).astype(np.uint32) for s in range(n_seq)]
    got = llama.generate_batch(rt, prompts, 1)[0]
    for s in range(n_seq):
        top = np.sort(rt.logits(s))[-2:]
        if top[1] - top[0] > 1e-3:
            assert got[s] == [rt.select_greedy(s)]
    rt.close()


def near_head(fmt, rows, cols, seed):
    """Blocks of a head whose rows are one row of large weights and a little noise: their logits lie as close as rounding the weights to fp16 moves them (0.02 of a step where the rows differ by one
    or two), and sums of 32 bits do not."""
    rng = np.random.default_rng(seed)
    half = lambda x: np.asarray(x, np.float16).view(np.uint8).reshape(*np.shape(x), 2)  # noqa: E731
    if fmt in (orc.FMT_Q8_0, orc.FMT_Q4_0):
        n = cols // 32
        d = np.broadcast_to(half(rng.uniform(0.001, 0.002, n)), (rows, n, 2))
        if fmt == orc.FMT_Q8_0:
            q = (rng.integers(64, 126, cols) * rng.choice([-1, 1], cols))[None] + rng.integers(-2, 3, (rows, cols), dtype=np.int8)
            return np.concatenate([d, q.astype(np.int8).view(np.uint8).reshape(rows, n, 32)], -1).ravel()
        q = np.where(rng.random(cols) < 0.5, rng.integers(0, 3, (rows, cols)), rng.integers(13, 16, (rows, cols))).astype(np.uint8).reshape(rows, n, 32)
        return np.concatenate([d, q[..., :16] | q[..., 16:] << 4], -1).ravel()
    n = cols // 256
    sc, m = rng.integers(1, 64, (n, 8)).astype(np.uint8), rng.integers(32, 64, (n, 8)).astype(np.uint8)   # value sc d q - m dmin, the second part a hundred times the first one's step
    head = np.concatenate([half(rng.uniform(1e-5, 2e-5, n)), half(rng.uniform(1e-3, 2e-3, n)), sc[:, :4] | sc[:, 4:] >> 4 << 6, m[:, :4] | m[:, 4:] >> 4 << 6, sc[:, 4:] & 15 | (m[:, 4:] & 15) << 4], -1)
    return np.concatenate([np.broadcast_to(head, (rows, n, 16)), rng.integers(0, 256, (rows, n, 128), dtype=np.uint8)], -1).ravel()


# a vocabulary and widths that no kernel with exact weights takes as a batch (Q4_K from nine rows on), and ones that one does
@pytest.mark.parametrize("fmt,d_model,vocab,n_seq", [(orc.FMT_Q8_0, 576, 49152, 3), (orc.FMT_Q8_0, 576, 49152, 16), (orc.FMT_Q4_0, 576, 49152, 16), (orc.FMT_Q4_K, 1536, 32000, 9), (orc.FMT_Q4_K, 1536, 32000, 8),
                                                     (orc.FMT_Q8_0, 768, 32000, 16), (orc.FMT_Q4_K, 1024, 32000, 16), (orc.FMT_Q4_0, 2048, 32000, 3)])
def test_first_tokens_of_a_batch_hang_on_exact_heads(llama, fmt, d_model, vocab, n_seq):
    kw = dict(n_layer=1, n_head=d_model // 64, n_kv_head=d_model // 64, d_model=d_model, head_dim=64, hidden_dim=512, max_seq=16)
    packed = mu.pack_weights(mu.random_weights(orc.LlamaConfig(gemv_inputs_fp16=True, vocab=256, **kw), 5, std=0.05), fmt)[0]
    packed["embedding"] = np.random.default_rng(6).normal(0, 1, (vocab, d_model)).astype(np.float16).view(np.uint8).ravel()
    packed["lm_head"] = near_head(fmt, vocab, d_model, 7)
    rt = llama.LlamaRuntime(llama.MultiModelConfig(vocab=vocab, **kw), max_sequences=n_seq)
    llama.load_packed_weights(rt, packed, fmt)
    rng = np.random.default_rng(n_seq)
    checked = 0
    for _ in range(max(2, 192 // n_seq)):
        rt.reset()
        got = llama.generate_batch(rt, [rng.integers(0, vocab, 3 + s % 4).astype(np.uint32) for s in range(n_seq)], 1)[0]
        for s in range(n_seq):
            logits = rt.logits(s)
            top = np.sort(logits)[-2:]
            if top[1] - top[0] > 1e-3 * logits.std():   # what a hidden row's own rounding to fp16 may move
                assert got[s] == [rt.select_greedy(s)], s
                checked += 1
    assert checked > 100
    rt.close()
