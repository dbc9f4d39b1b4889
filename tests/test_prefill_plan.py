"""The plan of prefill launches that run as ranges of equal work, on the CPU:
every range walked with the kernel's own arithmetic, each tile's counts
covered once, each split tile's description naming its pieces."""
import heapq

import numpy as np
import pytest

from prefill_plan import (BY_CLASS, LIST_ORDER, LIST_PARTS, SEQUENCES, check_walk, item_order, route,
                          tile_order)


def equal(f32, n, heads, kvh, q, k, d=128):
    r = route(f32, n, heads, kvh, q, k, d)
    return r, (check_walk(r, [q] * n, [k] * n, heads, kvh) if r.ranges else 0)


# f32, sequences, q heads, kv heads, queries each: shapes whose counts pass
# 2^24 at long contexts.
LONG = [
    (False, 1, 32, 8, 512), (False, 2, 32, 8, 512), (False, 63, 32, 8, 64),
    (False, 22, 32, 32, 200), (False, 15, 32, 8, 128), (False, 2, 32, 8, 960),
    (False, 20, 32, 8, 192), (True, 1, 16, 8, 512), (True, 3, 16, 8, 300),
]


@pytest.mark.parametrize("case", LONG, ids=lambda c: f"f32-{c[0]}-n{c[1]}-kvh{c[3]}-q{c[4]}")
def test_ranges_hold_up_to_the_longest_context_they_are_taken_for(case):
    """Every context for the last 1,500 keys that ranges are taken for (they
    end where the counts' products would leave 32 bits), and around the
    largest that an unbounded product would allow."""
    f32, n, heads, kvh, q = case
    lo, hi = 4096, 1 << 20
    assert not route(f32, n, heads, kvh, q, hi, 128).ranges
    # The last context, on a grid coarse enough that equal shares taken here
    # and there below it don't matter.
    ks = [k for k in range(lo, hi, 997) if route(f32, n, heads, kvh, q, k, 128).ranges]
    assert ks
    for k in range(max(ks[-1] - 1500, q), ks[-1] + 2000, 7):
        r, bad = equal(f32, n, heads, kvh, q, k)
        assert bad == 0, (k, r)
    # Ragged: one sequence at that length, the others anywhere below.
    rng = np.random.default_rng(n)
    for _ in range(20):
        k = ks[-1] - int(rng.integers(0, 300))
        r = route(f32, n, heads, kvh, q, k, 128)
        lens_q = [int(x) for x in rng.integers(1, q + 1, n)]
        lens_k = [int(x) for x in rng.integers(q, k + 1, n)]
        lens_q[0], lens_k[-1] = q, k
        for wl, wr in ((-1, 0), (-1, -1), (5000, 0)):
            if r.ranges:
                assert check_walk(r, lens_q, lens_k, heads, kvh, wl, wr) == 0


@pytest.mark.parametrize("f32", [False, True])
def test_ranges_hold_over_ragged_batches(f32):
    rng = np.random.default_rng(7 + f32)
    taken = 0
    for _ in range(4000):
        n = int(rng.integers(1, 65))
        kvh = int(rng.choice([1, 2, 3, 4, 8, 32]))
        heads = kvh * int(rng.choice([1, 2, 4, 7, 16]))
        q = int(np.exp(rng.uniform(np.log(2), np.log(3000))))
        k = q + int(np.exp(rng.uniform(0, np.log(60000))))
        d = int(rng.choice([64, 128]))
        ws = (1 << 64) - 1 if rng.random() < 0.5 else int(np.exp(rng.uniform(9, 19)))
        r = route(f32, n, heads, kvh, q, k, d, True, ws)
        if not r.ranges:
            continue
        taken += 1
        assert r.range_bytes <= ws
        lens_q = [int(x) for x in rng.integers(0, q + 1, n)]
        lens_k = [max(l, int(x)) for l, x in zip(lens_q, rng.integers(0, k + 1, n))]
        lens_q[-1], lens_k[-1] = q, k
        wl = -1 if rng.random() < 0.7 else int(rng.integers(0, k))
        wr = int(rng.choice([-1, 0, 0, 5]))
        assert check_walk(r, lens_q, lens_k, heads, kvh, wl, wr) == 0, (r, lens_q, lens_k, wl, wr)
    assert taken > 200


def test_lengths_past_the_hosts_bound_stay_within_the_counts():
    """max_seqlen_k below the real lengths costs balance, not coverage."""
    for n, q, k in ((3, 512, 8192), (10, 100, 9000), (1, 512, 400000)):
        r = route(False, n, 32, 8, q, k, 128)
        assert r.ranges
        assert check_walk(r, [q] * n, [1 << 24] * n, 32, 8) == 0
        assert check_walk(r, [q] * n, [k] * (n - 1) + [1 << 30], 32, 8) == 0


MIB16 = 16 << 20


def test_a_small_workspace_does_not_run_a_launch_on_fewer_cus():
    """16 MiB hold 62 ranges: a launch that fills the GPU with its tiles keeps
    them, whatever ranges would save with all the workspace asked for."""
    for n, heads, kvh, q, k in ((5, 32, 8, 512, 4096), (3, 32, 8, 512, 8192),
                                (6, 28, 4, 1000, 8000)):
        assert route(False, n, heads, kvh, q, k, 128).ranges == 256
        assert route(False, n, heads, kvh, q, k, 128, True, MIB16).ranges == 0
    assert route(True, 5, 16, 8, 512, 4096, 128).ranges == 256
    assert route(True, 5, 16, 8, 512, 4096, 128, True, MIB16).ranges == 0


def test_f32_batches_of_few_rows_get_the_ranges_their_workspace_is_for():
    """Where the split kernel runs as ranges but not as tiles: the workspace asked
    for holds them all."""
    for n, heads, kvh, q, k in ((40, 8, 4, 59, 862), (40, 16, 8, 59, 862), (33, 8, 4, 40, 2000)):
        r = route(True, n, heads, kvh, q, k, 128)
        assert r.ranges == 256
        assert route(True, n, heads, kvh, q, k, 128, True, r.range_bytes).ranges == 256


def test_ranges_of_a_small_workspace_beat_its_tiles_or_shares():
    """A range's steps are at most those of the rounds of tiles or shares that
    the same workspace allows, all sequences as long as the longest."""
    rng = np.random.default_rng(3)
    taken = 0
    for _ in range(20000):
        n, kvh = int(rng.integers(1, 65)), int(rng.choice([1, 2, 4, 8, 32]))
        heads = kvh * int(rng.choice([1, 4, 7]))
        q = int(np.exp(rng.uniform(np.log(2), np.log(2000))))
        k = q + int(np.exp(rng.uniform(0, np.log(30000))))
        ws = int(np.exp(rng.uniform(np.log(1 << 20), np.log(128 << 20))))
        r = route(False, n, heads, kvh, q, k, 128, True, ws)
        if not r.ranges:
            continue
        taken += 1
        rounds = -(-r.items * r.n_split // 256)
        assert r.items / r.ranges <= rounds / r.n_split, (r, n, q, k, ws)
    assert taken > 100


def test_a_launch_by_classes_takes_every_tile_once_from_the_longest_down():
    """Over ragged batches: no tile comes before one that has two classes (of
    16) more work, and tiles of nearly equal work keep their sequences together."""
    rng = np.random.default_rng(5)
    for i in range(300):
        n, step = int(rng.integers(2, 65)), int(rng.choice([1, 3, 16, 36, 64, 256]))
        top = int(np.exp(rng.uniform(np.log(step), np.log(30000))))
        lens_q = [int(x) for x in rng.integers(0, min(top, 40 * step) + 1, n)]
        lens_k = [q + int(x) for q, x in zip(lens_q, rng.integers(0, top + 1, n))]
        if i % 3 == 0:
            lens_k = lens_q
        tiles = [-(-q // step) for q in lens_q]
        if sum(tiles) > 700:
            continue
        order = tile_order(lens_k, tiles, step)
        work = [lens_k[s] - (tiles[s] - 1 - t) * step for s, t in order]
        longest = max([k for k, t in zip(lens_k, tiles) if t] + [1])
        if min(work + [longest]) < longest // 2:
            after = -10 ** 9
            for w in reversed(work):  # (thresholds are multiples of longest // 16)
                assert w >= after - 2 * (longest // 16) - 16
                after = max(after, w)
        else:
            assert order == sorted(order, key=lambda x: (-lens_k[x[0]], x[0], -x[1]))


def rounds(order, lens_k, tiles, step, kvh, cus=32):
    """When the last CU of an XCD ends, in keys, its tiles dealt in order."""
    end = 0
    items = [(s, t) for s, t in order for _ in range(kvh)]
    for x in range(8):
        free = [0] * cus
        for s, t in items[x::8]:
            heapq.heapreplace(free, free[0] + lens_k[s] - (tiles[s] - 1 - t) * step)
        end = max(end, max(free))
    return end


@pytest.mark.parametrize("heads,kvh,n", [(16, 2, 4), (8, 1, 8), (32, 1, 3)])
def test_equal_fresh_prompts_end_within_a_quarter_of_an_even_division(heads, kvh, n):
    """With one or two kv heads, where whole sequences one after the other
    ended up to half past it."""
    assert route(False, n, heads, kvh, 2000, 2000, 128, False).order == BY_CLASS
    step = 256 // (heads // kvh)
    tiles = [-(-2000 // step)] * n
    order = tile_order([2000] * n, tiles, step)
    even = sum(2000 - (tiles[s] - 1 - t) * step for s, t in order) * kvh / 256
    assert rounds(order, [2000] * n, tiles, step, kvh) <= 1.25 * even
    whole = sorted(order, key=lambda x: (x[0], -x[1]))
    assert rounds(whole, [2000] * n, tiles, step, kvh) > 1.25 * even


@pytest.mark.parametrize("heads,kvh,n", [(16, 16, 40), (24, 12, 40), (8, 8, 64)])
def test_ragged_sequences_of_one_tile_each_do_not_end_on_a_long_one(heads, kvh, n):
    """A round or more of items: the launch ends within a sixth of the longest
    item past an even division, where the list dealt as it is ends a fifth or more
    of one past it."""
    rng = np.random.default_rng(4)
    lens = [int(x) for x in np.clip(np.exp(rng.normal(np.log(300), 0.75, n)), 33, 4000)]
    lens[-1] = max(lens) + 1
    r = route(False, n, heads, kvh, 20, max(lens), 128, False)
    assert r.qtiles == 1 and r.order == SEQUENCES
    walk = sorted(range(n), key=lambda i: -lens[i])
    even = max(sum(lens) * kvh / 256, max(lens))
    assert rounds([(s, 0) for s in walk], lens, [1] * n, 1, kvh) <= even + max(lens) / 6
    assert rounds([(s, 0) for s in range(n)], lens, [1] * n, 1, kvh) > even + max(lens) / 5


def test_short_sequences_keep_list_order():
    """Where the sort costs more than it gives (few keys, all items at once, or
    many rounds of them), and a sequence's tiles stay on one XCD."""
    for n, heads, kvh, q, k, d, want in ((64, 16, 16, 32, 32, 128, LIST_PARTS),
                                         (64, 32, 8, 12, 600, 64, LIST_PARTS),
                                         (64, 32, 32, 12, 600, 128, LIST_ORDER),
                                         (64, 16, 16, 12, 600, 128, LIST_ORDER),
                                         (130, 32, 32, 50, 50, 128, LIST_ORDER),
                                         (130, 32, 32, 50, 50, 80, LIST_PARTS),
                                         (64, 28, 4, 64, 64, 128, LIST_PARTS),
                                         (130, 28, 4, 50, 50, 64, LIST_PARTS),
                                         (40, 28, 4, 128, 128, 128, SEQUENCES)):
        kernel_d = 64 if d <= 64 else 128
        assert route(False, n, heads, kvh, q, k, kernel_d, False, pool_dim=d).order == want
    # f32: as listed with one tile, walked with several.
    assert route(True, 40, 16, 8, 128, 128, 64, False).order == LIST_ORDER
    assert route(True, 10, 64, 8, 63, 63, 128, False).order == SEQUENCES
    for n, qtiles, kvh in ((64, 2, 4), (130, 2, 4), (20, 1, 16), (3, 5, 3)):
        items = item_order(n, qtiles, kvh)
        assert sorted(items) == [(s, h, t) for s in range(n) for h in range(kvh)
                                 for t in range(qtiles)]
        xcds = [{(i, s) for i, (s, h, t) in enumerate(items) if i % 8 == x} for x in range(8)]
        # A sequence on two XCDs at most, where each holds a sequence or more.
        if n >= 8:
            assert max(sum(any(s == q for _, q in x) for x in xcds) for s in range(n)) <= 2
