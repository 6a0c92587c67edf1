"""GPU parity of the closure by walks from every source (closure_rows.hip) against the CPU oracle, over ids of the whole
32-bit range: sources at the capacities of its three sets and their neighbours, walks at the largest number of layers
of each, runs of 255 edges and more, cycles, the smallest relations, what it gives up on, and the iteration limit."""
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


@pytest.mark.parametrize("reach", [254, 255, 256, 895, 896, 897, 1791, 1792, 1793, 7167, 7168, 7169])
def test_reach_at_the_capacities(provider, reach):
    # 2 -> 3 -> (reach - 1 targets): sources with reach and reach - 1 pairs, the second through its run's length
    star = _star(3, 4, reach - 1)
    st = _check(provider, np.concatenate([[[2, 3], [0, 1]], star, _padding(4 + reach, 40 + reach // 4)]))
    assert st["host_waits"] <= AUTO_WAITS or reach > 7168


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
