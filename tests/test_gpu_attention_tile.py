"""Attention over many tokens (the prompt tiles) and over a step's few query rows
against the oracle, bit for bit: tile sizes 8, 16 and 32, partial tiles, a past,
passes of fewer queries than a tile, head widths 64 and 128, tokens of several
cache rows or lengths, masked keys and values that reach the host's results, the
tiles' outputs quantised in the decoder, and its steps on both sides of the
length at which their kernel changes."""
import sys

import numpy as np
import pytest

from oracle import oracle
import tensomite_hip as th

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return th.HIPDevice(0)


def attend(dev, q, k, v, table):
    tokens, heads, width = q.shape
    rows, kv_heads, capacity, _ = k.shape
    scale = float(np.float32(1.0 / np.sqrt(width)))
    out = dev.attention(dev.from_array(q), tokens, heads, dev.from_array(k), dev.from_array(v), rows, kv_heads,
                        capacity, width, dev.from_array(np.array(table, np.int32)), scale)
    return dev.to_array(out, np.float32, q.size).reshape(q.shape), scale


def same(got, want):
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])


def inputs(seed, tokens, heads, kv_heads, width, capacity, rows=1):
    rng = np.random.default_rng(seed)
    cache = (rows, kv_heads, capacity, width)
    q, k, v = (rng.normal(0, 1, s).astype(np.float32) for s in ((tokens, heads, width), cache, cache))
    q[tokens // 2] *= 40.0  # sharp softmax: many exponentials underflow to 0
    return q, k, v


# tokens · heads from one round of workgroups up; tiles of 8, 16 and 32 tokens
# (their count times heads against two a compute unit), whole and partial; the
# last two: score rows too long for all a tile's queries, and one position
@pytest.mark.parametrize("tokens,heads,kv_heads,width,past,capacity", [
    (24, 32, 32, 64, 0, 24), (97, 9, 3, 64, 0, 512), (130, 8, 2, 64, 3, 140), (257, 32, 4, 64, 1, 300),
    (512, 32, 32, 64, 0, 512), (100, 12, 4, 128, 30, 131), (330, 32, 2, 128, 0, 400), (160, 52, 4, 64, 1240, 1400),
    (16, 48, 48, 64, 0, 2048)])
def test_prompt_tiles(dev, tokens, heads, kv_heads, width, past, capacity):
    print("prompt tiles", tokens, heads, kv_heads, width, past, capacity, flush=True)
    q, k, v = inputs(tokens + past, tokens, heads, kv_heads, width, capacity)
    table = [(0, past + t, past + tokens) for t in range(tokens)]
    got, scale = attend(dev, q, k, v, table)
    dev.sync()
    same(got, oracle.attention(q, k, v, table, scale))


def test_tiles_of_several_rows(dev):
    # tokens 0-15 a whole tile, 16-39 each its own row and length, the rest
    # of the second row; one row's ends in no order
    tokens, heads, capacity = 72, 16, 90
    q, k, v = inputs(5, tokens, heads, 4, 64, capacity, rows=3)
    rng = np.random.default_rng(6)
    table = [(0, int(rng.integers(0, 60)), 60) for _ in range(16)]
    for t in range(16, 40):
        length = int(rng.integers(1, capacity + 1))
        table.append((t % 3, int(rng.integers(0, length)), length))
    table += [(1, t, 80) for t in range(tokens - 40)]
    got, scale = attend(dev, q, k, v, table)
    dev.sync()
    same(got, oracle.attention(q, k, v, table, scale))


# Tokens of several cache rows in one call: as many sequences as tokens (a decode
# step's), more query rows than a round of workgroups takes with every tile
# mixed, and whole tiles beside mixed ones.
@pytest.mark.parametrize("width", [64, 128])
@pytest.mark.parametrize("tokens,heads,rows,run", [(24, 32, 24, 1), (200, 32, 5, 3), (150, 24, 4, 40)])
def test_tokens_of_several_rows(dev, width, tokens, heads, rows, run):
    print("several rows", width, tokens, heads, rows, run, flush=True)
    capacity = 70
    q, k, v = inputs(tokens, tokens, heads, 8, width, capacity, rows=rows)
    rng = np.random.default_rng(tokens)
    table = []
    for t in range(tokens):
        length = int(rng.integers(1, capacity + 1))
        table.append((t // run % rows, int(rng.integers(0, length)), length))
    got, scale = attend(dev, q, k, v, table)
    dev.sync()
    same(got, oracle.attention(q, k, v, table, scale))


# Tokens of one row with a length each: a token does not see what lies past its
# own length, masked or not, whatever the others see of it.
@pytest.mark.parametrize("width", [64, 128])
@pytest.mark.parametrize("beyond", [1.0, np.nan, np.inf])
def test_tiles_of_own_lengths(dev, width, beyond):
    print("own lengths", width, beyond, flush=True)
    tokens, heads, capacity, past = 100, 16, 160, 40
    q, k, v = inputs(17, tokens, heads, 8, width, capacity)
    v[0, 3, past + 60, 5] = beyond
    k[0, 2, past + 75, 9] = beyond
    table = [(0, past + t, min(capacity, past + t + 1 + (t % 7) * 3)) for t in range(tokens)]
    with np.errstate(all="ignore"):
        got, scale = attend(dev, q, k, v, table)
        dev.sync()
        same(got, oracle.attention(q, k, v, table, scale))


def test_tile_entry_out_of_range(dev):
    # the entry's token gets zeros and a report, the others their attention
    tokens, heads, capacity = 64, 16, 64
    q, k, v = inputs(8, tokens, heads, 16, 64, capacity)
    table = [(0, t, tokens) for t in range(tokens)]
    good = oracle.attention(q, k, v, table, float(np.float32(0.125)))
    table[37] = (0, 3, capacity + 1)
    got, _ = attend(dev, q, k, v, table)
    with pytest.raises(th.ExecutionError):
        dev.sync()
    assert np.all(got[37] == 0)
    keep = np.arange(tokens) != 37
    same(got[keep], good[keep])


@pytest.mark.parametrize("poison", ["value nan", "value inf", "key nan", "key inf", "key huge", "seen nan", "query huge"])
def test_masked_keys_and_values(dev, poison):
    # the host's masked positions take part: a masked value that is not
    # finite times a zero weight, a masked score that is NaN or +inf - inf
    print("masked", poison, flush=True)
    tokens, heads, capacity, past = 96, 16, 160, 40
    q, k, v = inputs(11, tokens, heads, 8, 64, capacity)
    at = past + 70  # masked for the first 70 tokens
    if poison.startswith("value"):
        v[0, 3, at, 5] = np.nan if poison.endswith("nan") else -np.inf
    elif poison.startswith("key"):
        k[0, 3, at, 5] = {"nan": np.nan, "inf": np.inf, "huge": 3e38}[poison.split()[1]]
    elif poison == "seen nan":
        k[0, 2, 0, 9] = np.nan
        v[0, 5, 7, 1] = np.inf
    else:
        q[20, 4] *= np.float32(1e37)
    table = [(0, past + t, past + tokens) for t in range(tokens)]
    with np.errstate(all="ignore"):
        got, scale = attend(dev, q, k, v, table)
        dev.sync()
        same(got, oracle.attention(q, k, v, table, scale))


# One workgroup a query row and head: positions of one, two and more rounds of
# value blocks, whole and partial blocks, capacities on both sides of 2048, few
# and many heads; the last past the causal end (masked positions).
@pytest.mark.parametrize("width", [64, 128])
@pytest.mark.parametrize("capacity,lengths", [
    (70, [1, 63, 64, 65, 70]), (600, [128, 129, 511, 512, 513, 600]), (1100, [1024, 1025, 1040, 1100]),
    (2048, [2048, 1537, 16]), (3000, [3000, 2049, 17]), (5200, [5200])])
def test_few_query_rows(dev, width, capacity, lengths):
    print("few rows", width, capacity, lengths, flush=True)
    heads, kv_heads = 4, 2
    q, k, v = inputs(capacity + width, len(lengths), heads, kv_heads, width, capacity, rows=len(lengths))
    for seen in (1.0, 0.6):
        table = [(i, max(0, int(n * seen) - 1), n) for i, n in enumerate(lengths)]
        got, scale = attend(dev, q, k, v, table)
        dev.sync()
        same(got, oracle.attention(q, k, v, table, scale))
    k[0, 0, 0, 3] = np.nan  # a NaN at position 0 reaches every weight of its head
    v[-1, 1, lengths[-1] - 1, 2] = np.inf
    table = [(i, n - 1, n) for i, n in enumerate(lengths)]
    with np.errstate(all="ignore"):
        got, scale = attend(dev, q, k, v, table)
        dev.sync()
        same(got, oracle.attention(q, k, v, table, scale))


# Rows of one block of 64 positions (one wave's): groups of 16 whole and partial, the
# causal end before the length, a NaN first score, values that are not finite seen and
# masked, an entry out of range beside them; and in the decoder, quantised.
def test_rows_of_one_block(dev):
    lengths = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65]
    q, k, v = inputs(3, len(lengths), 8, 2, 64, 70, rows=len(lengths))
    k[4, 1, 0, 7] = np.nan
    v[6, 0, 31, 3] = np.inf
    k[8, 1, 46, 2] = -np.inf
    v[9, 1, 40, 5] = np.nan
    for seen in (1.0, 0.6):
        table = [(i, max(0, int(n * seen) - 1), n) for i, n in enumerate(lengths)]
        with np.errstate(all="ignore"):
            got, scale = attend(dev, q, k, v, table)
            dev.sync()
            want = oracle.attention(q, k, v, table, scale)
        same(got, want)
    table[3] = (3, 16, 16)
    with np.errstate(all="ignore"):
        got, _ = attend(dev, q, k, v, table)
    with pytest.raises(th.ExecutionError):
        dev.sync()
    assert np.all(got[3] == 0)
    keep = np.arange(len(lengths)) != 3
    same(got[keep], want[keep])


@pytest.mark.parametrize("tokens", [3, 16, 33, 64])
def test_prompt_of_one_block_quantised(dev, tokens):
    from llama_fixtures import random_llama
    config = dict(layers=2, width=64, heads=4, kv_heads=2, head_width=64, hidden=64, vocab=96, context=80, eps=1e-5,
                  theta=10000.0, kind="Q4_0")
    weights = random_llama(config, seed=tokens, std=0.2)
    ids = np.random.default_rng(tokens).integers(0, 96, tokens).astype(np.int32)
    want = oracle.Llama(config, weights).forward([int(i) for i in ids])
    same(th.HIPLlama(dev, config, weights, max_tokens=tokens).forward(ids), want)


# Capacities whose scores fill the workgroup's LDS: the last one with room for
# two waves' keys, the first without, the first without room for one's, and the
# largest the entry point takes.
@pytest.mark.parametrize("width,capacity", [(64, 32256), (64, 32257), (64, 36353), (64, 39356),
                                            (128, 32000), (128, 32001), (128, 36097), (128, 38264)])
def test_capacities_that_fill_lds(dev, width, capacity):
    print("capacity", width, capacity, flush=True)
    lengths = [capacity, 700, 1]
    q, k, v = inputs(capacity, len(lengths), 2, 1, width, capacity, rows=len(lengths))
    table = [(i, n - 1, n) for i, n in enumerate(lengths)]
    got, scale = attend(dev, q, k, v, table)
    dev.sync()
    same(got, oracle.attention(q, k, v, table, scale))


@pytest.mark.parametrize("head_width,capacity", [(64, 1200), (128, 700), (64, 2600)])
def test_decode_past_several_rounds(dev, head_width, capacity):
    # the decode step's form (RoPE, the cache write and the new position
    # inside): one-id forwards after a long prompt against one forward
    from llama_fixtures import random_llama
    config = dict(layers=1, width=128, heads=4, kv_heads=2, head_width=head_width, hidden=64, vocab=64,
                  context=capacity, eps=1e-5, theta=10000.0, kind="Q8_0")
    weights = random_llama(config, seed=capacity, std=0.2)
    ids = np.random.default_rng(3).integers(0, 64, capacity).astype(np.int32)
    want = oracle.Llama(config, weights).forward([int(i) for i in ids])
    model = th.HIPLlama(dev, config, weights, max_tokens=512)
    at = 0
    for upto in [u for u in (0, 60, 63, 127, 511, 513, 1023, 1025) if u < capacity - 3] + [capacity - 2]:
        if upto > at:
            model.forward(ids[at:upto], last_only=True)
            at = upto
        for _ in range(2):
            got = model.forward(ids[at:at + 1])
            assert np.array_equal(got.view(np.uint32)[0], want.view(np.uint32)[at]), at
            at += 1


# The decoder's prompts: the tiles' outputs quantised for the o product, whose
# staging takes a score row as wide as a query's outputs although the first tiles'
# positions are fewer. Tiles of 8, 16 and 32 tokens (one, two and four queries a
# wave); the last cases' whole cache is shorter than 64 positions.
@pytest.mark.parametrize("head_width", [64, 128])
@pytest.mark.parametrize("heads,tokens,capacity", [
    (16, 40, 256), (32, 64, 256), (32, 65, 256), (16, 200, 200), (32, 250, 256), (64, 250, 250), (32, 20, 20), (64, 60, 60)])
def test_prompt_tiles_quantised(dev, head_width, heads, tokens, capacity):
    from llama_fixtures import random_llama
    print("quantised tiles", head_width, heads, tokens, capacity, flush=True)
    config = dict(layers=1, width=64, heads=heads, kv_heads=4, head_width=head_width, hidden=32, vocab=96,
                  context=capacity, eps=1e-5, theta=10000.0, kind="Q8_0")
    weights = random_llama(config, seed=tokens + heads, std=0.2)
    ids = np.random.default_rng(tokens).integers(0, 96, tokens).astype(np.int32)
    want = oracle.Llama(config, weights).forward([int(i) for i in ids])
    got = th.HIPLlama(dev, config, weights, max_tokens=tokens).forward(ids)
    same(got, want)


# Decode steps on both sides of the length at which the step's attention kernel
# changes (256 positions of the longest row), the shorter rows far from it: tokens
# from step graphs of either kernel (the second time both captured), and eager
# ones.
@pytest.mark.parametrize("rows,heads,longest", [(2, 4, 250), (8, 32, 250), (8, 32, 506)])
def test_steps_across_the_attention_kernels(dev, rows, heads, longest):
    from llama_fixtures import random_llama
    print("steps", rows, heads, longest, flush=True)
    config = dict(layers=2, width=64, heads=heads, kv_heads=4, head_width=64, hidden=64, vocab=96,
                  context=600, eps=1e-5, theta=10000.0, kind="Q8_0")
    weights = random_llama(config, seed=longest, std=0.2)
    rng = np.random.default_rng(longest)
    prompts = [[int(i) for i in rng.integers(0, 96, max(1, longest - 80 * r))] for r in range(rows)]
    cpu = oracle.Llama(config, weights)
    want = [cpu.generate(p, 12) for p in prompts]
    model = th.HIPLlama(dev, config, weights, rows=rows, max_tokens=512)
    for graph in (True, True, False):
        for r, p in enumerate(prompts):
            model.reset(r)
            model.forward(p, row=r, last_only=True)
        got = model.generate(12, graph=graph)
        assert [list(t) for t in got] == want, graph
