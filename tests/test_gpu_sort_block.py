"""GPU parity of the one-workgroup sort (up to 16,384 keys) and the bucket sort (up to 2^20) against numpy: its wave, round and size edges, keys whose
bins are short (hashed, dense ids) and long (hubs, few values: the digit passes in LDS), and the stable sort by one
column that a join's build side takes."""
import numpy as np
import pytest

from xlog_amd import pack

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 63, 64, 65, 1023, 1024, 1025, 4097, 16383, 16384, 16385]


def _keys(kind, n, rng):
    if kind == "hashed":
        return rng.integers(0, 1 << 64, n, dtype=np.uint64)
    if kind == "dense":
        return pack(rng.integers(0, 1000, n), rng.integers(0, 700, n))
    if kind == "hub":
        return pack(np.where(rng.random(n) < 0.6, 7, rng.integers(0, 1 << 32, n)), rng.integers(0, 3000, n))
    if kind == "few":
        return rng.choice(np.array([0, 1, (1 << 64) - 1, 1 << 63], dtype=np.uint64), n)
    return np.full(n, 0xFFFFFFFF00000000, dtype=np.uint64)  # equal


@pytest.mark.parametrize("kind", ["hashed", "dense", "hub", "few", "equal"])
def test_sort_and_dedup(provider, kind):
    for n in SIZES:
        k = _keys(kind, n, np.random.default_rng(n))
        R = provider.create_buffer_from_packed(k)
        assert np.array_equal(provider.download_packed(provider.sort(R, [0, 1])), np.sort(k)), n
        d = provider.dedup_full_row(R)
        assert np.array_equal(provider.download_packed(d), np.unique(k)), n
        assert d.is_canonical()
        assert np.array_equal(provider.download_packed(R), k), n  # the input is left as it is


@pytest.mark.parametrize("digits", [2, 3, 5, 8])
@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_longest_bin(provider, digits, extra):
    """One bin (a value of the top 12 bits that vary) holds as many keys as are ranked, one fewer, one more; the low
    word of the keys varies whole before the high word does."""
    rng = np.random.default_rng(digits * 3 + extra)
    below, long = 8 * digits - 12, 14 * digits + extra
    top = np.concatenate([np.arange(4096), np.full(long - 1, 77)]).astype(np.uint64)
    low = rng.integers(0, 1 << below, len(top), dtype=np.uint64)
    k = rng.permutation((top << np.uint64(below)) | low)
    R = provider.create_buffer_from_packed(k)
    assert np.array_equal(provider.download_packed(provider.sort(R, [0, 1])), np.sort(k))
    assert np.array_equal(provider.download_packed(provider.dedup_full_row(R)), np.unique(k))


@pytest.mark.parametrize("kind", ["hashed", "dense", "hub", "few", "equal"])
@pytest.mark.parametrize("n", [1, 65, 1025, 16384])
def test_stable_by_column(provider, kind, n):
    """The rows of a run of equal join keys come in input order."""
    k = _keys(kind, n, np.random.default_rng(n))
    col = (k >> np.uint64(32)).astype(np.uint32)
    some = np.unique(col)[:8]
    out = provider.hash_join_v2(provider.create_buffer_from_u32_columns([some]),
                                provider.create_buffer_from_u32_columns([col, np.arange(n, dtype=np.uint32)]), [0], [0])
    want = np.concatenate([np.nonzero(col == v)[0] for v in some])
    assert np.array_equal(provider.download_column(out, 2), want.astype(np.uint32))


@pytest.mark.parametrize("kind", ["hashed", "dense", "hub", "few", "equal"])
@pytest.mark.parametrize("n", [16385, 32768, 32769, 100003, (1 << 20) - 1, 1 << 20, (1 << 20) + 1])
def test_bucket_sort(provider, kind, n):
    """The bucket sort at its size edges and where the number of buckets changes."""
    k = _keys(kind, n, np.random.default_rng(n))
    R = provider.create_buffer_from_packed(k)
    assert np.array_equal(provider.download_packed(provider.sort(R, [0, 1])), np.sort(k))
    assert np.array_equal(provider.download_packed(provider.dedup_full_row(R)), np.unique(k))
    assert np.array_equal(provider.download_packed(R), k)


@pytest.fixture
def launches(provider):
    """A function giving the launches of each kernel kind in a call."""
    def count(call):
        provider.profile_enable(True)
        try:
            provider.profile_reset()
            call()
            return {k: v["launches"] for k, v in provider.profile_read().items()}
        finally:
            provider.profile_enable(False)
    return count


@pytest.mark.parametrize("kind", ["few", "equal", "equal 0", "equal ends", "hub", "hubs", "next to hubs"])
@pytest.mark.parametrize("n", [20000, 100003, 1 << 20])
def test_bucket_sort_repeats(provider, launches, kind, n):
    """Values with more repeats than a bucket's region holds (4,096 keys) are sorted without digit passes."""
    rng = np.random.default_rng(n)
    top = (1 << 64) - 1
    if kind == "equal 0":
        k = np.zeros(n, dtype=np.uint64)
    elif kind == "equal ends":
        k = rng.choice(np.array([0, top], dtype=np.uint64), n)
    elif kind in ("few", "equal"):
        k = _keys(kind, n, rng)
    else:  # among hashed keys: one value, four with the ends, and values whose neighbours are there, too
        k = rng.integers(0, 1 << 64, n, dtype=np.uint64)
        hubs = {"hub": [12345 << 30], "hubs": [0, 1 << 40, (1 << 40) + 1, top],
                "next to hubs": [(5 << 40) + d for d in (-1, 0, 1)]}[kind]
        at = rng.random(n) < 0.6
        k[at] = rng.choice(np.array(hubs, dtype=np.uint64), int(at.sum()))
    R = provider.create_buffer_from_packed(k)
    out = {}
    ran = launches(lambda: out.update(s=provider.sort(R, [0, 1]), d=provider.dedup_full_row(R)))
    assert np.array_equal(provider.download_packed(out["s"]), np.sort(k))
    assert np.array_equal(provider.download_packed(out["d"]), np.unique(k))
    assert ran["sort_pass"] == 0 and ran["sort_segments"] == 2


def unlucky(k):
    """The keys with the smallest one's repeats where the bucket sort takes its sample: one bucket gets the others."""
    n = len(k)
    bits = next(b for b in range(1, 32) if (n >> b) <= 1024)
    i = np.arange(8 << bits, dtype=np.uint64)
    step = np.uint64(n // (8 << bits))
    at = i * step + (((i * np.uint64(0x9E3779B1)) & np.uint64(0xFFFFFFFF)) >> np.uint64(8)) % step
    k = k.copy()
    k[at] = k.min()
    return k


@pytest.mark.parametrize("n", [16385, 100003, 1 << 20])
def test_bucket_sort_unlucky_sample(provider, launches, n):
    """A bucket that outgrows its region: the digit passes sort the keys instead."""
    k = unlucky(np.random.default_rng(n).integers(0, 1 << 64, n, dtype=np.uint64))
    R = provider.create_buffer_from_packed(k)
    out = {}
    ran = launches(lambda: out.update(s=provider.sort(R, [0, 1]), d=provider.dedup_full_row(R)))
    assert np.array_equal(provider.download_packed(out["s"]), np.sort(k))
    assert np.array_equal(provider.download_packed(out["d"]), np.unique(k))
    assert np.array_equal(provider.download_packed(R), k)
    assert ran["sort_pass"] > 0 and ran["sort_segments"] == 2


@pytest.mark.parametrize("order", ["ascending", "descending", "runs"])
def test_bucket_sort_ordered_input(provider, order):
    """Inputs whose order the sample's stretches follow."""
    n = 200001
    k = np.sort(np.random.default_rng(1).integers(0, 1 << 64, n, dtype=np.uint64))
    k = {"ascending": k, "descending": k[::-1], "runs": np.roll(np.repeat(k[:: 7], 7)[:n], 3)}[order].copy()
    R = provider.create_buffer_from_packed(k)
    assert np.array_equal(provider.download_packed(provider.dedup_full_row(R)), np.unique(k))


@pytest.mark.parametrize("misled", [False, True])
def test_fixpoint_with_repeated_facts(provider, misled):
    """One fact repeated 60,000 times inside a program, and one where the sample sees no other, so that the buckets do
    not fit."""
    import oracle
    from xlog_amd import datagen, tc_plan

    s, d = datagen.random_digraph(3000, 4000, 5)
    e = np.concatenate([pack(s, d), np.full(60000, pack(s[:1], d[:1])[0], dtype=np.uint64)])
    if misled:
        e = np.roll(np.sort(np.tile(np.unique(e), 16)), 7)
        e = unlucky(e)
        s, d = (e >> np.uint64(32)).astype(np.uint32), e.astype(np.uint32)
    outs, st = provider.fixpoint(tc_plan(), [provider.create_buffer_from_packed(e), None])
    ref = oracle.bfs_tc(3000, s, d)
    assert np.array_equal(provider.download_packed(outs[1]), ref["relation"]) and st["iterations"] == ref["iterations"]
