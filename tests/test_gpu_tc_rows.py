"""GPU parity of the closure by walks from every source (closure_rows.hip) against the CPU oracle, over ids of the whole
32-bit range: sources at the capacities of its three sets and of their frontiers, walks at the largest number of layers
of the first two (the third's needs more sources on its list than fit it below 1.4e7 edges), the sources that outgrow
all of them and what the loop over hash sets makes of those, runs of 255 edges and more, cycles, the smallest relations,
what it gives up on, and the iteration limit.  The counts of each list come from the trace line."""
import re

import numpy as np
import pytest

import oracle
from xlog_amd import XlogError, pack, tc_plan

pytestmark = pytest.mark.gpu

ITERATION_LIMIT = 4
AUTO_WAITS = 8  # read-backs of a call that takes the walks; the loop over hash sets has one per 8 iterations more


def _spread(edges, seed=1, shuffle=True):
    """distinct ids over the whole range for 0..n-1 (ascending unless shuffled), the two ends among them"""
    n = int(edges.max()) + 1 if edges.size else 1
    ids = np.unique(np.random.default_rng(seed).integers(1, 2**32 - 1, 2 * n + 8, dtype=np.uint64))[: max(n - 2, 0)]
    ids = np.concatenate([[0], ids, [2**32 - 1]]).astype(np.uint32)
    if shuffle:
        np.random.default_rng(seed + 1).shuffle(ids)
    return ids[edges]


def _padding(first, n):  # edges that no other touches
    return np.arange(first, first + 2 * n).reshape(n, 2)


def _check(p, edges, plan=None, shuffle=True):
    edges = np.asarray(edges, dtype=np.int64).reshape(-1, 2)
    e = _spread(edges, shuffle=shuffle)
    E = np.unique(pack(e[:, 0], e[:, 1]))
    outs_o, it_o, deltas_o = oracle.seminaive(tc_plan(), [E, None])
    outs, st = p.fixpoint(plan or tc_plan(), [p.create_buffer_from_packed(E), None])
    assert np.array_equal(p.download_packed(outs[1]), outs_o[1])
    assert st["iterations"] == it_o and st["delta_sizes"] == deltas_o
    return st


def _star(root, first, n):
    return np.stack([np.full(n, root), np.arange(first, first + n)], 1)


@pytest.mark.parametrize("n", [1, 2, 23, 24, 25, 48, 49, 300, 5000])
def test_random(provider, n):
    rng = np.random.default_rng(n)
    st = _check(provider, rng.integers(0, n + 1, (n, 2)) if n < 300 else rng.integers(0, int(1.3 * n), (n, 2)))
    assert st["host_waits"] <= AUTO_WAITS or n < 300  # (a few edges may follow each other too often)


@pytest.fixture
def lists(monkeypatch, capfd):
    """A function giving what the last call's walks did: sources listed, listed for the largest sets, handed back; None
    when they gave up or did not run."""
    monkeypatch.setenv("XLOG_HIP_TRACE", "1")

    def read():
        found = re.findall(r"closure walks: (\d+) sources listed, (\d+) for the largest sets, (\d+) handed back(.*)",
                           capfd.readouterr().err)
        assert len(found) <= 1
        return tuple(int(v) for v in found[0][:3]) if found and not found[0][3] else None
    return read


def _alone(runs, first):
    """Edges where each of the runs (source, targets) begins a batch of 24 edges with nothing else in it; the sources are
    numbered in the order of the runs.  Between them are edges that no other touches, from vertex `first` on."""
    at = np.cumsum([0] + [len(t) + (-len(t)) % 24 for _, t in runs])  # the number of each run's first edge
    n = int(at[-1])
    number, edges, extra = {s: int(a) for a, (s, _) in zip(at, runs)}, [], n + first
    for a, (s, t) in zip(at, runs):
        for v in t:
            edges.append((number[s], number.get(v, v + n)))
        for k in range((-len(t)) % 24):
            edges.append((int(a) + 1 + k, extra))
            extra += 1
    return np.array(edges)


def _comb(reach, width):
    """A spine s0 -> s1 -> ... whose vertices have width - 1 leaves each: s0 reaches `reach` vertices, at most `width`
    of them a layer; runs for _alone and the first number free for it."""
    runs, leaf, left = [], 1000, reach
    while left > 0:
        more = left > width
        k = width - 1 if more else left
        runs.append((-len(runs) - 1, ([-len(runs) - 2] if more else []) + list(range(leaf, leaf + k))))
        leaf += k
        left -= width
    return runs, leaf


# the first width fits every frontier up to its tier's (256, 512, 2048 edges), so that the pairs (896, 1792, 7168) decide
@pytest.mark.parametrize("tier,width,reach", [(t, w, r + d) for t, w, r in ((0, 201, 896), (1, 401, 1792), (2, 1901, 7168))
                                              for d in (-1, 0, 1)])
def test_pairs_at_the_capacities(provider, lists, tier, width, reach):
    runs, first = _comb(reach, width)
    edges = _alone(runs, first)
    _check(provider, edges, shuffle=False)
    n = len(runs)
    reaches = [reach - width * i for i in range(n)]
    over = [sum(r > cap for r in reaches) for cap in (896, 1792, 7168)]
    if tier > 0:  # wider than the frontiers before
        over[0] = sum(min(r, width) > 256 for r in reaches)
    if tier > 1:
        over[1] = sum(min(r, width) > 512 for r in reaches)
    assert lists() == tuple(over)
    assert over[tier] == (reach > (896, 1792, 7168)[tier])


@pytest.mark.parametrize("width", [255, 256, 257, 511, 512, 513, 2047, 2048, 2049])
def test_frontiers(provider, lists, width):
    """A run alone, and one that a single edge leads to."""
    runs = [(-1, list(range(1000, 1000 + width))), (-2, [-3]), (-3, list(range(9000, 9000 + width)))]
    _check(provider, _alone(runs, 20000), shuffle=False)
    # (the second shares its batch with 23 sources that no other touches)
    assert lists() == (26 * (width > 256), 3 * (width > 512), 3 * (width > 2048))


@pytest.mark.parametrize("layers", [127, 128, 129, 511, 512, 513])
def test_layers_of_single_sources(provider, lists, layers):
    """A path whose sources are alone in their batches: before each lies a run of 47 edges."""
    edges = []
    for i in range(layers):
        edges += [(2 * i, 5000 + 47 * i + k) for k in range(47)] + [(2 * i + 1, 2 * i + 3 if i + 1 < layers else 4000)]
    _check(provider, edges, shuffle=False)
    assert lists() == (max(0, layers - 128), max(0, layers - 512), 0)


@pytest.mark.parametrize("n_back", [1, 3, 20, 60])
def test_sources_handed_back(provider, lists, n_back):
    """Sources that outgrow the largest sets, and ones that reach them, go through the loop over hash sets; the others
    stay with the walks.  Cycles and long paths among both, so that either part has the more iterations."""
    rng = np.random.default_rng(n_back)
    parts, first = [], 0

    def add(edges, size):
        nonlocal first
        parts.append(np.asarray(edges, dtype=np.int64).reshape(-1, 2) + first)
        first += size

    hub = first
    add(_star(0, 1, 3000), 3001)                       # too many edges
    for k in range(n_back - 1):                        # they lead to it
        add([[0, hub - first]], 1)
    path = min(100, 40 * n_back)
    add([[i, i + 1] for i in range(path)], path + 1)
    add([[i, (i + 1) % 9] for i in range(9)], 9)
    add(rng.integers(0, 9000, (4000, 2)), 9000)
    edges = np.concatenate(parts)
    edges = np.concatenate([edges, _padding(first, 3600 * n_back)])  # (so that few edges follow an edge on average)
    edges = np.concatenate([edges, [[hub + 5, hub + 3001 + n_back - 1]]])  # from one of its targets along the path
    st = _check(provider, edges)
    got = lists()
    assert got is not None and got[2] == n_back
    e = _spread(edges)
    E = provider.create_buffer_from_packed(np.unique(pack(e[:, 0], e[:, 1])))
    provider.fixpoint(tc_plan(), [E, None], max_iterations=st["iterations"])
    assert lists() == got
    with pytest.raises(XlogError) as ex:
        provider.fixpoint(tc_plan(), [E, None], max_iterations=st["iterations"] - 1)
    assert ex.value.status == ITERATION_LIMIT
    del ex


@pytest.mark.parametrize("reach", [254, 255, 256, 895, 896, 897, 1791, 1792, 1793, 7167, 7168, 7169])
def test_stars(provider, reach):
    # 2 -> 3 -> (reach - 1 targets): sources with reach and reach - 1 pairs, the second through its run's length
    star = _star(3, 4, reach - 1)
    st = _check(provider, np.concatenate([[[2, 3], [0, 1]], star, _padding(4 + reach, 40 + reach // 4)]))
    assert st["host_waits"] <= AUTO_WAITS or reach > 2048  # (the loop over hash sets takes the larger ones)


@pytest.mark.parametrize("layers", [127, 128, 129, 511, 512, 513])
def test_layers(provider, layers):
    # the path's sources lie together, so few other sources share their batches
    path = np.stack([np.arange(layers), np.arange(1, layers + 1)], 1)
    st = _check(provider, np.concatenate([path, _padding(layers + 1, 2000)]), shuffle=False)
    assert st["host_waits"] <= AUTO_WAITS


def test_cycles_and_both_rule_forms(provider):
    edges = np.concatenate([[[i, (i + 1) % 40] for i in range(40)], [[50, 50], [51, 52], [52, 51], [51, 0]]])
    _check(provider, edges)
    t = np.array([[i, (i * 7 + 3) % 101] for i in range(101)])
    _check(provider, t)


def test_gives_up(provider):
    rng = np.random.default_rng(5)
    _check(provider, rng.integers(0, 700, (1400, 2)))  # most sources reach most of it


@pytest.mark.parametrize("small,large", [(40, 0), (40, 1), (40, 20), (0, 40)])
def test_large_runs_among_the_listed_sources(provider, small, large):
    """The largest sets' launch with many sources: runs that its frontier holds (up to 2,048 edges) and runs that it
    refuses at their first push, when other workgroups of the launch are still starting and find the attempt ended."""
    stars, first = [], 0
    for k in range(small + large):
        n = 600 + 30 * k if k < small else 2049 + 17 * k
        stars.append(_star(first, first + 1, n))
        first += n + 1
    _check(provider, np.concatenate(stars[::2] + stars[1::2] + [_padding(first, 3000)]))


def test_iteration_limit(provider):
    path = np.stack([np.arange(60), np.arange(1, 61)], 1)
    e = _spread(np.concatenate([path, _padding(61, 100)]))
    E = provider.create_buffer_from_packed(np.unique(pack(e[:, 0], e[:, 1])))
    outs, st = provider.fixpoint(tc_plan(), [E, None], max_iterations=60)
    assert st["iterations"] == 60 and st["delta_sizes"] == [160] + list(range(59, -1, -1))
    with pytest.raises(XlogError) as ex:
        provider.fixpoint(tc_plan(), [E, None], max_iterations=59)
    assert ex.value.status == ITERATION_LIMIT
    del ex
