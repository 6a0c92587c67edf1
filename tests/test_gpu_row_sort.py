"""GPU parity of the sort and dedup of rows by key columns (any arity, any key list) against a stable numpy sort: the
prefix of the key's bits that one u64 holds, runs of equal prefix ordered by the rest, runs too long for that, and the
tile and size edges."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(p, cols, keys):
    n = len(cols[0])
    R = p.create_buffer_from_u32_columns(cols)
    order = np.lexsort([cols[c] for c in reversed(keys)])  # stable
    s = p.sort(R, keys)
    for c, col in enumerate(cols):
        assert np.array_equal(p.download_column(s, c), col[order]), ("sort", c)
    first = np.ones(n, bool)
    first[1:] = np.any([cols[c][order][1:] != cols[c][order][:-1] for c in keys], axis=0)
    d = p.dedup(R, keys)
    assert d.num_rows() == int(first.sum())
    for c, col in enumerate(cols):
        assert np.array_equal(p.download_column(d, c), col[order][first]), ("dedup", c)
    for c, col in enumerate(cols):
        assert np.array_equal(p.download_column(R, c), col)  # the input is left as it is


def _rows(rng, n, arity, kind):
    if kind == "wide":      # more bits than a prefix holds, few ties
        tops = [1 << 32] * arity
    elif kind == "narrow":  # the prefix holds every bit
        tops = [7, 1, 300, 2, 5, 3, 2, 9][:arity]
    elif kind == "ties":    # equal prefixes in short runs, told apart by the rest
        tops = [max(2, n // 5)] + [1 << 32] * (arity - 1)
    else:                   # "runs": equal prefixes in long runs
        tops = [2] * (arity - 1) + [1 << 32]
    cols = [rng.integers(0, t, n).astype(np.uint32) for t in tops]
    if kind in ("ties", "runs"):
        for c in range(1, max(1, arity - 1)):
            cols[c] = (cols[c] % 2 * 0xFFFFFFFF).astype(np.uint32)  # 32 used bits, two values
    if n > 3:  # repeated rows
        src = rng.integers(0, n, n // 4)
        dst = rng.integers(0, n, n // 4)
        for c in cols:
            c[dst] = c[src]
    return cols


@pytest.mark.parametrize("kind", ["wide", "narrow", "ties", "runs"])
@pytest.mark.parametrize("arity", [1, 2, 3, 4, 5, 6, 7, 8])
def test_all_columns(provider, kind, arity):
    for n in (2, 3, 1000, 20011):
        _check(provider, _rows(np.random.default_rng(n + arity), n, arity, kind), list(range(arity)))


@pytest.mark.parametrize("kind", ["wide", "narrow", "ties", "runs"])
@pytest.mark.parametrize("keys", [[0], [1], [2, 0], [3, 1, 0], [1, 1, 3], [3, 2, 1, 0]])
def test_key_lists(provider, kind, keys):
    for n in (1023, 1024, 1025, 1088, 1089, 30000):
        _check(provider, _rows(np.random.default_rng(n), n, 4, kind), keys)


@pytest.mark.parametrize("run", [2, 63, 64, 65, 66, 1024])
def test_run_lengths(provider, run):
    """Runs of one prefix at the longest length that is ordered on chip, across tile edges, and past it."""
    rng = np.random.default_rng(run)
    n = 5000
    cols = [(np.arange(n) // run * 7919).astype(np.uint32)] + [rng.integers(0, 1 << 32, n).astype(np.uint32) for _ in range(3)]
    cols[0][0] = 0xFFFFFFFF
    _check(provider, [c[rng.permutation(n)] if i else c for i, c in enumerate(cols)], [0, 1, 2, 3])


def _hashed(rng, n, distinct):
    """A column of 32-bit values, `distinct` of them (0: any)."""
    if not distinct:
        return rng.integers(0, 1 << 32, n).astype(np.uint32)
    return rng.choice(rng.integers(0, 1 << 32, distinct), n).astype(np.uint32)


# distinct values of each column: the first has few, all have few, a first that hardly splits the rows
@pytest.mark.parametrize("distinct", [(3, 0, 0), (100, 0, 0, 0), (20, 20, 20, 20), (1, 0, 5, 0), (2, 2, 2, 0, 2, 2),
                                      (7, 7, 7, 7, 7, 7, 7, 7), (50, 1000, 3, 1000)])
@pytest.mark.parametrize("n", [16384, 16385, 70001, (1 << 20) + 3])
def test_long_runs(provider, distinct, n):
    """Runs of equal prefix that are sorted again by the key's next bits, once or several times, and those that go by
    pieces of the whole key."""
    rng = np.random.default_rng(n)
    _check(provider, [_hashed(rng, n, d) for d in distinct], list(range(len(distinct))))


@pytest.mark.parametrize("share", [0.001, 0.1, 0.9, 1.0])
def test_hub_among_short_runs(provider, share):
    """The rows of one value are sorted again and the others stay where the first sort put them."""
    n = 200003
    rng = np.random.default_rng(9)
    cols = [_hashed(rng, n, 0) for _ in range(4)]
    cols[0][rng.random(n) < share] = 0xFFFFFFFF
    cols[1][rng.random(n) < 0.3] = 0
    src, dst = rng.integers(0, n, n // 4), rng.integers(0, n, n // 4)
    for c in cols:
        c[dst] = c[src]
    _check(provider, cols, [0, 1, 2, 3])
    _check(provider, cols, [0, 3])
    _check(provider, cols[:3], [0, 2, 1])


@pytest.mark.parametrize("n", [(1 << 20) + 7, (1 << 22) + 1])
def test_large(provider, n):
    _check(provider, _rows(np.random.default_rng(5), n, 3, "ties"), [0, 1, 2])
