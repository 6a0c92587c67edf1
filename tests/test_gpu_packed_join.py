"""GPU parity of joins whose keys are packed into one u32 (their own slots, mixed, or too wide: the dictionaries) and of
the small build sides (bucket sort, keys with more rows than a bucket holds, the fallback where its sample misleads), against
numpy: inner joins in left-row-major, right-row order, semi and anti joins as the left rows with and without a match."""
from collections import defaultdict

import numpy as np
import pytest

from test_gpu_sort_block import launches, unlucky  # noqa: F401  (launches: a fixture)
from xlog_amd import JOIN_ANTI, JOIN_INNER, JOIN_SEMI

pytestmark = pytest.mark.gpu


def _check(p, left, right, lk, rk):
    L = p.create_buffer_from_u32_columns(left)
    R = p.create_buffer_from_u32_columns(right)
    rows = defaultdict(list)
    for j, key in enumerate(zip(*[right[c].tolist() for c in rk])):
        rows[key].append(j)
    li, ri, hit = [], [], []
    for i, key in enumerate(zip(*[left[c].tolist() for c in lk])):
        m = rows.get(key, [])
        li += [i] * len(m)
        ri += m
        hit.append(bool(m))
    hit = np.array(hit)
    if len(left) + len(right) <= 8:
        out = p.hash_join_v2(L, R, lk, rk, JOIN_INNER)
        want = [c[li] for c in left] + [c[ri] for c in right]
        assert out.num_rows() == len(li)
        for c, w in enumerate(want):
            assert np.array_equal(p.download_column(out, c), w), c
    for kind, keep in ((JOIN_SEMI, hit), (JOIN_ANTI, ~hit)):
        out = p.hash_join_v2(L, R, lk, rk, kind)
        for c, w in enumerate(left):
            assert np.array_equal(p.download_column(out, c), w[keep]), (kind, c)


def _cols(rng, n, tops):
    return [rng.integers(0, t, n).astype(np.uint32) for t in tops]


# the key columns' ranges: 9 bits (their own slots), 27 and 31 bits (mixed), 32, 33 and 64 bits (dictionaries)
@pytest.mark.parametrize("tops", [(40, 8), (1 << 21, 64), (1 << 16, 1 << 15), (1 << 16, 1 << 16), (1 << 32, 2),
                                  (1 << 32, 1 << 32)])
@pytest.mark.parametrize("nl,nr", [(1, 1), (300, 70), (20000, 16384), (5000, 30000)])
def test_two_keys(provider, tops, nl, nr):
    rng = np.random.default_rng(nl + nr)
    pool = [rng.integers(0, t, max(4, nr // 3)) for t in tops]  # values that meet
    left = [rng.choice(q, nl).astype(np.uint32) for q in pool] + _cols(rng, nl, (1 << 32,))
    right = _cols(rng, nr, (1 << 32,)) + [rng.choice(q, nr).astype(np.uint32) for q in pool] + _cols(rng, nr, (9,))
    _check(provider, left, right, [0, 1], [1, 2])
    _check(provider, left[:2], right[1:3], [1, 0], [1, 0])  # nothing beside the keys


def test_probe_bits_outside_the_build_side(provider):
    """Left values with bits that no right row has must not match through the packing."""
    left = [np.array([0, 1, 2, 3, 4, 0xFFFFFFFF, 3, 7], np.uint32), np.array([0, 1, 2, 3, 0, 0xFFFFFFFF, 7, 3], np.uint32)]
    right = [np.array([0, 3, 2], np.uint32), np.array([0, 3, 2], np.uint32)]
    _check(provider, left, right, [0, 1], [0, 1])
    _check(provider, left, [np.zeros(2, np.uint32)] * 2, [0, 1], [0, 1])  # keys of no bits


@pytest.mark.parametrize("arity", [(2, 2), (1, 2), (2, 1), (3, 2), (2, 4), (4, 4)])
@pytest.mark.parametrize("nr", [100, 16385, 60000])
def test_one_key(provider, arity, nr):
    rng = np.random.default_rng(nr)
    nl = 9000
    left = _cols(rng, nl, (1 << 32,) * (arity[0] - 1)) + [rng.integers(0, nr // 2, nl).astype(np.uint32)]
    right = [rng.integers(0, nr // 2, nr).astype(np.uint32)] + _cols(rng, nr, (1 << 32,) * (arity[1] - 1))
    _check(provider, left, right, [arity[0] - 1], [0])


@pytest.mark.parametrize("wide", [False, True])
def test_hub_keys(provider, wide):
    """Keys with thousands of rows on the build side, all ones among them."""
    rng = np.random.default_rng(2)
    key = rng.permutation(np.concatenate([np.full(9000, 0xFFFFFFFF), np.full(30000, 5), np.arange(20000)])).astype(np.uint32)
    right = [key] + _cols(rng, len(key), (1 << 32,) * (2 if wide else 1))
    left = [np.array([5, 6, 0xFFFFFFFF, 1 << 31, 7], np.uint32), np.arange(5, dtype=np.uint32)]
    _check(provider, left, right, [0], [0])


@pytest.mark.parametrize("keys", [1, 2])
@pytest.mark.parametrize("nr", [16385, 60000, 3 << 17, (3 << 17) + 1])
def test_unlucky_sample(provider, launches, keys, nr):
    """A build side whose sample sees one key only: the index that was begun is dropped, and the second one sorts by
    digit passes at once, as larger build sides of one key column do."""
    rng = np.random.default_rng(nr)
    one = unlucky(rng.integers(1, 250, nr).astype(np.uint32))
    right = [one] + _cols(rng, nr, (200, 1 << 32) if keys == 2 else (1 << 32,))
    left = [np.arange(0, 300, 7, dtype=np.uint32)] + _cols(rng, 43, (250,))
    L, R = provider.create_buffer_from_u32_columns(left), provider.create_buffer_from_u32_columns(right)
    on = list(range(keys))
    ran = launches(lambda: provider.hash_join_v2(L, R, on, on, JOIN_INNER))
    assert ran["sort_segments"] == (keys > 1 or nr <= 3 << 17) and ran["sort_pass"] > 0
    if nr < 1 << 17:
        _check(provider, left, right, on, on)
    else:  # the pairs of left and right rows alone
        out = provider.hash_join_v2(L, R, on, on, JOIN_INNER)
        code = lambda cols: sum(c.astype(np.int64) << (16 * i) for i, c in enumerate(cols[:keys]))  # noqa: E731
        order = np.argsort(code(right), kind="stable")
        lo, hi = (np.searchsorted(code(right)[order], code(left), s) for s in ("left", "right"))
        want = np.concatenate([order[a:b] for a, b in zip(lo, hi)])
        assert np.array_equal(provider.download_column(out, len(left) + keys), right[keys][want])


@pytest.mark.parametrize("key", ["equal", "two", "hub", "collide"])
@pytest.mark.parametrize("nr", [1, 1023, 1025, 40000, 600000])
def test_key_set_of_repeats(provider, key, nr):
    """Semi and anti joins against keys that most build rows share, with single rows of other keys among them."""
    rng = np.random.default_rng(nr)
    if key == "equal":
        k = np.full(nr, 0xFFFFFFFF, dtype=np.uint32)
    elif key == "two":
        k = rng.choice(np.array([0, 77], np.uint32), nr)
    elif key == "hub":
        k = np.where(rng.random(nr) < 0.9, 5, rng.integers(0, 1 << 32, nr)).astype(np.uint32)
    else:  # a few hundred keys in turn, so that the keys last seen change all the time
        k = (np.arange(nr, dtype=np.uint32) * np.uint32(2654435761)) % np.uint32(499) * np.uint32(8192)
    left = [np.concatenate([k[:: max(1, nr // 2000)], rng.integers(0, 1 << 32, 500, dtype=np.uint32)]).astype(np.uint32)]
    left.append(np.arange(len(left[0]), dtype=np.uint32))
    L, R = provider.create_buffer_from_u32_columns(left), provider.create_buffer_from_u32_columns([k, k])
    hit = np.isin(left[0], k)
    for kind, keep in ((JOIN_SEMI, hit), (JOIN_ANTI, ~hit)):
        out = provider.hash_join_v2(L, R, [0], [0], kind)
        assert np.array_equal(provider.download_column(out, 1), left[1][keep])
