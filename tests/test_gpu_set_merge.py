"""GPU parity of the set operations of an iteration on canonical relations against numpy: the union by merge alone (sets
that share nothing) and with its repeats dropped, and the difference by the merge path, at tile edges (2,048 merged keys),
shared keys on both sides of a tile edge, and the size ratios where the difference changes its kernel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel(p, keys):
    r = p.dedup_full_row(p.create_buffer_from_packed(np.asarray(keys, dtype=np.uint64)))
    assert r.is_canonical()
    return r


def _check(p, a, b):
    A, B = _rel(p, a), _rel(p, b)
    for x, y, X, Y in ((a, b, A, B), (b, a, B, A)):
        u = p.union_gpu(X, Y)
        assert np.array_equal(p.download_packed(u), np.union1d(x, y)) and u.is_canonical()
        d = p.diff_gpu(X, Y)
        assert np.array_equal(p.download_packed(d), np.setdiff1d(x, y)) and d.is_canonical()


@pytest.mark.parametrize("na,nb", [(1, 1), (1, 2047), (2048, 2048), (4095, 4096), (4096, 4097), (5000, 20000),
                                   (4096, 131072), (4096, 131073), (70000, 300000)])
@pytest.mark.parametrize("kind", ["apart", "overlap", "equal", "one", "ends"])
def test_union_diff(provider, na, nb, kind):
    rng = np.random.default_rng(na + nb)
    b = np.unique(rng.integers(0, 1 << 40, nb, dtype=np.uint64) * np.uint64(2))
    if kind == "apart":
        a = np.unique(rng.integers(0, 1 << 40, na, dtype=np.uint64) * np.uint64(2) + np.uint64(1))
    elif kind == "overlap":
        a = np.unique(np.concatenate([rng.choice(b, na // 2 + 1), rng.integers(0, 1 << 41, na // 2, dtype=np.uint64)]))
    elif kind == "equal":
        a = b[: min(na, len(b))].copy()
    elif kind == "one":  # one shared key, at the end
        a = np.unique(np.concatenate([rng.integers(0, 1 << 40, na, dtype=np.uint64) * np.uint64(2) + np.uint64(1), b[-1:]]))
    else:  # 0 and all ones on both sides
        a = np.unique(np.concatenate([rng.integers(0, 1 << 41, na, dtype=np.uint64), np.array([0, 2**64 - 1], np.uint64)]))
        b = np.unique(np.concatenate([b, np.array([0, 2**64 - 1], np.uint64)]))
    _check(provider, a, b)


def test_every_tile_edge(provider):
    """Equal pairs at every offset around the tile edges of the merge."""
    b = np.arange(0, 3 * 8192, dtype=np.uint64)
    for shift in range(5):
        a = b[shift :: 5][:4999]
        _check(provider, a, b)


@pytest.mark.parametrize("shared", ["none", "one", "first tile", "half", "all"])
def test_shared_keys_of_many_tiles(provider, shared):
    """Hundreds of tiles with shared keys in none, one or all of them."""
    b = np.arange(0, 2_000_000, dtype=np.uint64) * np.uint64(4)
    a = b[: 1_000_000] * np.uint64(2) + np.uint64(1)
    if shared == "one":
        a[500_000] += np.uint64(3)
    elif shared == "first tile":
        a[:10] = b[:20:2]
    elif shared == "half":
        a[::2] += np.uint64(3)
    elif shared == "all":
        a = b[: 1_000_000].copy()
    assert len(np.intersect1d(a, b)) == {"none": 0, "one": 1, "first tile": 10, "half": 500_000, "all": 1_000_000}[shared]
    _check(provider, np.unique(a), b)
