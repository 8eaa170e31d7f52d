"""The block attention kernels by themselves, against 64 bits: how exact they are, and that a row meets only the keys it sees."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import espresso_amd.ops as ops
    ops.init()
    yield ops
    ops.set_tuning("prompt_attention_key_sets", 0)


def inputs(rows, first, heads, kv_heads, size, dtype, seed, sharp=1.0):
    rng = np.random.default_rng(seed)
    q = rng.normal(0, sharp, (rows, heads, size)).astype(np.float32)
    return q, rng.normal(0, 1, (first + rows, kv_heads, size)).astype(dtype), rng.normal(0, 1, (first + rows, kv_heads, size)).astype(dtype)


def exact(q, k, v):
    rows, heads, size = q.shape
    first, share = k.shape[0] - rows, heads // k.shape[1]
    out = np.empty(q.shape)
    for h in range(heads):
        s = q[:, h].astype(np.float64) @ k[:, h // share].astype(np.float64).T / np.sqrt(size)
        s[np.arange(k.shape[0])[None, :] > first + np.arange(rows)[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = p / p.sum(1, keepdims=True) @ v[:, h // share].astype(np.float64)
    return out


# tiles of 32 rows and keys, prefixes that are whole tiles and not, one to eight wavefronts per tile
SHAPES = [(1, 0, 3, 1, 128), (4, 0, 8, 8, 64), (31, 1, 8, 1, 64), (32, 32, 9, 3, 64), (33, 31, 6, 2, 128), (93, 700, 8, 2, 64), (97, 33, 4, 1, 128), (300, 0, 6, 2, 128), (512, 45, 6, 2, 128),
          (256, 257, 32, 8, 64)]


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("rows,first,heads,kv_heads,size", SHAPES)
def test_span_attention_is_as_exact_as_fp32(ops, rows, first, heads, kv_heads, size, dtype):
    """Split rows carry 22 bits, so a context that fp32 sums are behind shows.  Scores of hundreds: rounding queries or keys to 22 bits moves a weight by
    2^-23 times the score's terms, rounding them to fp16 by 2^-11."""
    planes = heads * size % 256 == 0
    for sharp in (1.0, 60.0):
        q, k, v = inputs(rows, first, heads, kv_heads, size, dtype, rows + first, sharp)
        want = exact(q, k, v)
        got, _ = ops.block_attention("span", q, k, v, split_rows=planes)
        one, _ = ops.block_attention("single_row", q, k, v)
        # an fp32 sum of `size` products is off by about 2^-24 sqrt(size) of their root of squares, which is sharp after the scale 1 / sqrt(size); a weight by that much of
        # itself, and the context by that much of the values' spread; planes end at 2^-22, fp16 at 2^-11 of the result
        def off(c):
            return np.sqrt(np.mean((c - want) ** 2))
        assert off(got) <= 2.0 ** -24 * (np.sqrt(size) * sharp + 8) + 2.0 ** (-22 if planes else -11) * np.sqrt(np.mean(want ** 2)), sharp
        if not planes:   # the same fp16 rounding on both sides: no worse than the kernel that does every row by itself
            assert off(got) <= 1.02 * off(one) + 1e-9, sharp


# four and eight wavefronts (1, 2; 0: by size, eight from 24 tiles of keys on) where some have no tile of keys, one, or one more than the others; the shares of dims that they finish, and their sums of 32
@pytest.mark.parametrize("sets", [0, 1, 2])
@pytest.mark.parametrize("rows,first,heads,kv_heads,size", [(1, 0, 4, 4, 64), (1, 31, 2, 1, 128), (32, 1, 12, 4, 64), (33, 95, 2, 2, 128), (64, 193, 6, 2, 128), (31, 224, 4, 1, 64), (2, 255, 8, 2, 128), (31, 737, 4, 1, 64),
                                                             (5, 731, 8, 2, 128), (1, 800, 12, 4, 64)])
def test_span_attention_by_any_number_of_wavefronts(ops, rows, first, heads, kv_heads, size, sets):
    ops.set_tuning("prompt_attention_key_sets", sets)
    q, k, v = inputs(rows, first, heads, kv_heads, size, np.float16, rows + first, 4.0)
    want = exact(q, k, v)
    for planes in (True, False):
        got, _ = ops.block_attention("span", q, k, v, split_rows=planes)
        # as above: 2^-24 of scores and sums, planes end at 2^-22 and fp16 at 2^-11 of the result
        assert np.sqrt(np.mean((got - want) ** 2)) <= 2.0 ** -24 * (np.sqrt(size) * 4.0 + 8) + 2.0 ** (-22 if planes else -11) * np.sqrt(np.mean(want ** 2)), planes
    ops.set_tuning("prompt_attention_key_sets", 0)


# prompts of more rows than one workgroup a compute unit (32 heads by 16 tiles of rows) up to 2048 keys, and behind them
@pytest.mark.parametrize("rows,first", [(512, 1536), (512, 1537), (490, 1650), (481, 3000)])
def test_prompts_behind_long_prefixes_are_as_exact_as_rows_alone(ops, rows, first):
    for sharp in (1.0, 30.0):
        q, k, v = inputs(rows, first, 32, 8, 128, np.float16, rows, sharp)
        at = np.r_[0:3, 30:34, rows - 9:rows]
        want = np.concatenate([exact(q[i:i + 1], k[:first + i + 1], v[:first + i + 1]) for i in at])
        def off(c):
            return np.sqrt(np.mean((c - want) ** 2))
        one = ops.block_attention("single_row", q, k, v)[0][at]
        for kernel in ("prompt", "span"):   # the same fp16 rounding of the context on all sides
            assert off(ops.block_attention(kernel, q, k, v)[0][at]) <= 1.02 * off(one) + 1e-9, (kernel, sharp)
        assert off(ops.block_attention("prompt", q, k, v, split_rows=True)[0][at]) <= 2.0 ** -24 * (np.sqrt(128) * sharp + 8) + 2.0 ** -22 * np.sqrt(np.mean(want ** 2))


def in_steps(q, k, v):
    """As exact(), but for scores that are fp32 sums of exact products of sixteen dims each."""
    rows, heads, size = q.shape
    first, share = k.shape[0] - rows, heads // k.shape[1]
    out = np.empty(q.shape)
    for h in range(heads):
        s = np.zeros((rows, k.shape[0]), np.float32)
        for d in range(0, size, 16):
            s = (s + q[:, h, d:d + 16].astype(np.float64) @ k[:, h // share, d:d + 16].astype(np.float64).T).astype(np.float32)
        s = s.astype(np.float64) / np.sqrt(size)
        s[np.arange(k.shape[0])[None, :] > first + np.arange(rows)[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = p / p.sum(1, keepdims=True) @ v[:, h // share].astype(np.float64)
    return out


@pytest.mark.parametrize("rows,first,heads,kv_heads,size", [(40, 700, 6, 2, 128), (300, 200, 8, 2, 128), (93, 1500, 12, 4, 64), (200, 900, 8, 4, 64)])
def test_scores_round_as_sums_of_whole_products_do(ops, rows, first, heads, kv_heads, size):
    """Scores of sixteen, where what rounds them outweighs the rest.  The matrix cores round twice in a product of sixteen dims: sqrt(2) of in_steps(), and a tenth for weights and sums.  Three parts of a
    query one after the other into the same sum would be three times as many roundings."""
    got = want = steps = []
    for seed in (1, 2):
        q, k, v = inputs(rows, first, heads, kv_heads, size, np.float16, seed, 16.0)
        want = want + [exact(q, k, v)]
        steps = steps + [in_steps(q, k, v)]
        got = got + [ops.block_attention("span", q, k, v, split_rows=True)[0]]
    def off(c):
        return np.sqrt(np.mean((np.array(c) - np.array(want)) ** 2))
    assert off(got) <= 1.1 * np.sqrt(2) * off(steps), off(got) / off(steps)


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("scale", [2.0 ** -40, 2.0 ** -12, 2.0 ** 14, 2.0 ** 60])
def test_span_attention_takes_queries_of_any_size(ops, scale, dtype):
    q, k, v = inputs(40, 50, 6, 2, 128, dtype, 5)
    k = (k / 64).astype(dtype)
    if dtype == np.float32:
        k = (k / np.float32(scale)).astype(np.float32)   # products of the same size as before
        want = exact(q * np.float32(scale), k, v)
    else:
        want = exact(np.float32(q * np.float32(scale)), k, v)
    got, _ = ops.block_attention("span", q * np.float32(scale), k, v, split_rows=True)
    if dtype == np.float32 or scale < 1:
        assert np.abs(got - want).max() <= 2e-6 * np.abs(want).max()
    else:   # one key takes everything, and which one hangs on a score's last bits where two are near: as many rows as with fp32 sums
        one, _ = ops.block_attention("single_row", q * np.float32(scale), k, v)
        near = [(np.abs(c - want).max(-1) <= 2.0 ** -11 * np.abs(want).max(-1)).mean() for c in (got, one)]
        assert near[0] >= near[1] - 0.02 > 0.9


@pytest.mark.parametrize("kernel,heads,size", [("span", 6, 128), ("span", 6, 64), ("prompt", 8, 128)])
def test_the_largest_queries_meet_fp16_caches(ops, kernel, heads, size):
    """Queries of up to 2^120, whose scores are still floats: one key takes everything, as above."""
    q, k, v = inputs(40, 50, heads, 2, size, np.float16, 8)
    q, k = q * np.float32(2.0 ** 118), (k / 64).astype(np.float16)
    want = exact(q, k, v)
    got, _ = ops.block_attention(kernel, q, k, v)
    one, _ = ops.block_attention("single_row", q, k, v)
    near = [(np.abs(c - want).max(-1) <= 2.0 ** -11 * np.abs(want).max(-1)).mean() for c in (got, one)]
    assert near[0] >= near[1] - 0.02 > 0.9


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("magnitude", [3e-7, 1e-3, 3e4, 3e8])
def test_span_attention_takes_values_of_any_size(ops, magnitude, dtype):
    if dtype == np.float16 and magnitude > 65504:
        pytest.skip("beyond the cache's type")
    q, k, v = inputs(70, 10, 6, 2, 128, dtype, 6)
    v = np.clip(v * magnitude / 2, -65504 if dtype == np.float16 else None, 65504 if dtype == np.float16 else None).astype(dtype)
    if magnitude > 65504:   # what adds up to a finite fp16 context
        v[0::2, :, :] = v[0, :, :]
        v[1::2, :, :] = -v[0, :, :]
        q[:] = 0.0
    want = exact(q, k, v)
    fits = np.abs(want) < 65000
    got, _ = ops.block_attention("span", q, k, v)
    assert np.isfinite(got[fits]).all() and fits.mean() > 0.3
    # fp16 ends at 2^-25 below its normal numbers; values cancel to an fp32 sum's 2^-22 of their size
    assert (np.abs(got - want)[fits] <= 2.0 ** -11 * np.abs(want)[fits] + 2.0 ** -25 + 2.0 ** -22 * np.abs(v).max()).all()


@pytest.mark.parametrize("kernel,heads,kv_heads,size,sets", [("span", 6, 2, 128, 0), ("span", 8, 1, 64, 0), ("prompt", 8, 2, 128, 1), ("prompt", 8, 2, 128, 2), ("prompt", 2, 2, 64, 1),
                                                             ("prompt", 4, 2, 64, 1)])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_what_a_row_does_not_see_does_not_reach_it(ops, kernel, heads, kv_heads, size, sets, dtype, bad):
    """A value that is not finite poisons the rows that see it and no others; so does a key."""
    rows, first, at = 75, 13, 60
    ops.set_tuning("prompt_attention_key_sets", sets)
    q, k, v = inputs(rows, first, heads, kv_heads, size, dtype, 7)
    clean = exact(q, k, v)
    limit = 2e-3 if kernel == "prompt" and dtype == np.float32 else 2.0 ** -11   # that kernel rounds operands to fp16
    for which in (v, k):
        kept = which[at, 0, 5]
        which[at, 0, 5] = bad
        for planes in ([False, True] if heads * size % 256 == 0 and (kernel == "span" or dtype == np.float16) else [False]):
            got, _ = ops.block_attention(kernel, q, k, v, split_rows=planes)
            unseen = got[:at - first]
            assert np.isfinite(unseen).all()
            assert np.abs(unseen - clean[:at - first]).max() <= limit * np.abs(clean).max()
            share = heads // kv_heads
            if which is v:
                assert not np.isfinite(got[at - first:, :share, 5]).any()
                rest = got[at - first:, :share, :5]
                assert np.abs(rest - clean[at - first:, :share, :5]).max() <= limit * np.abs(clean).max()
            else:   # a score of -inf is a key that counts for nothing; any other poisons
                with np.errstate(all="ignore"):
                    want = exact(q[at - first:, :share], k[:, :1], v[:, :1])
                assert (np.isfinite(got[at - first:, :share]) == np.isfinite(want)).all()
        which[at, 0, 5] = kept


@pytest.mark.parametrize("size,planes", [(128, False), (64, True)])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_a_query_that_is_not_finite_is_its_own_row_alone(ops, size, planes, dtype, bad):
    q, k, v = inputs(45, 20, 8, 1, size, dtype, 9)
    want = exact(q, k, v)
    q[33, 5, size - 1] = q[2, 0, 0] = bad
    got, _ = ops.block_attention("span", q, k, v, split_rows=planes)
    assert np.isnan(got[33, 5]).all() and np.isnan(got[2, 0]).all()
    got[33, 5], got[2, 0] = want[33, 5], want[2, 0]
    assert np.abs(got - want).max() <= 2.0 ** -11 * np.abs(want).max()


@pytest.mark.parametrize("kernel", ["span", "prompt"])
def test_fp32_values_beyond_fp16_that_add_up(ops, kernel):
    """fp32 caches hold more than fp16: rows whose weighted sum fits come out finite."""
    q, k, v = inputs(40, 9, 4, 2, 64, np.float32, 8)
    q[:] = 0.0
    v[:] = np.where(np.arange(49)[:, None, None] % 2 == 0, 9e4, -9e4)
    want = exact(q, k, v)
    got, _ = ops.block_attention(kernel, q, k, v)
    assert np.abs(want).max() < 65504 and np.isfinite(got).all()
    assert np.abs(got - want).max() <= 2.0 ** -11 * np.abs(want).max()


# One workgroup a head (64 dims, fp16 caches, contexts of up to 256, 192 rows x heads and more), four slices and a merge, and the kernel of longer contexts; keys that end at, before and behind a pass of
# eight wavefronts (128 or 256 keys) and several passes
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("rows,first,heads,kv_heads,size", [
    (1, 0, 4, 4, 128), (3, 124, 8, 2, 128), (3, 125, 8, 8, 128), (2, 127, 6, 2, 64), (4, 253, 6, 2, 128), (5, 254, 4, 1, 128), (16, 300, 12, 4, 128), (3, 480, 32, 8, 128), (16, 496, 16, 16, 64), (8, 381, 9, 3, 64),
    (32, 200, 8, 2, 128), (6, 500, 32, 8, 128), (7, 600, 8, 2, 64)])
def test_steps_are_as_exact_as_fp32(ops, rows, first, heads, kv_heads, size, dtype):
    for sharp in (1.0, 60.0):
        q, k, v = inputs(rows, first, heads, kv_heads, size, dtype, rows + first, sharp)
        want = exact(q, k, v)
        got, _ = ops.block_attention("step", q, k, v)
        one, _ = ops.block_attention("single_row", q, k, v)
        off = lambda c: np.sqrt(np.mean((c - want) ** 2))  # noqa: E731
        # fp32 arithmetic as above, the context rounded to fp16 once (2^-11 at most); the kernel of longer contexts rounds likewise
        assert off(got) <= 2.0 ** -24 * (np.sqrt(size) * sharp + 8) + 2.0 ** -11 * np.sqrt(np.mean(want ** 2)), sharp
        assert off(got) <= 1.02 * off(one) + 2.0 ** -24 * np.sqrt(size) * sharp, sharp
