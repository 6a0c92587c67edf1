"""GPU parity of the column-blocked closure (closure_columns.hip) against the CPU oracle: domains at the edges of its
64-row slices, 1024-row instances and 32-column blocks, hubs (slices read a row at a time, targets with many sources),
iterations that push and that pull, a separate seed relation, and the iteration limit."""
import numpy as np
import pytest

import oracle
from xlog_amd import XlogError, copy_points_to_plan, datagen, pack, tc_plan

pytestmark = pytest.mark.gpu

ITERATION_LIMIT = 4


def _check(p, plan, rels, idb):
    outs_o, it_o, deltas_o = oracle.seminaive(plan, rels)
    dev = [p.create_buffer_from_packed(r) if r is not None else None for r in rels]
    outs, st = p.fixpoint(plan, dev)
    assert np.array_equal(p.download_packed(outs[idb]), outs_o[idb])
    assert st["iterations"] == it_o and st["delta_sizes"] == deltas_o


# the last vertex has an edge, so the domain is n
def _graph(n, m, seed):
    rng = np.random.default_rng(seed)
    e = np.stack([rng.integers(0, n, m), rng.integers(0, n, m)], 1)
    return np.unique(np.concatenate([pack(e[:, 0], e[:, 1]), pack([n - 1], [0])]))


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 63, 64, 65, 1023, 1024, 1025, 2048, 2049, 4096, 4097, 8193])
def test_domains(provider, n):
    _check(provider, tc_plan(), [_graph(n, int(1.3 * n) + 1, n), None], 1)


@pytest.mark.parametrize("n,m", [(16400, 18000), (24600, 24000), (32800, 30000), (38912, 35000)])
def test_large_instances(provider, n, m):
    e = _graph(n, m, n)
    ref = oracle.bfs_tc(n, (e >> np.uint64(32)).astype(np.uint32), e.astype(np.uint32))
    outs, st = provider.fixpoint(tc_plan(), [provider.create_buffer_from_packed(e), None])
    assert np.array_equal(provider.download_packed(outs[1]), ref["relation"])
    assert st["iterations"] == ref["iterations"]


@pytest.mark.parametrize("hub", ["sources", "targets"])
def test_hubs(provider, hub):
    n = 5000
    rng = np.random.default_rng(7)
    many = np.concatenate([rng.permutation(n)[:k] for k in (4000, 900, 70, 17, 16)])
    one = np.repeat([5, 1900, 1901, 77, n - 1], [4000, 900, 70, 17, 16])
    s, d = (one, many) if hub == "sources" else (many, one)
    e = np.unique(np.concatenate([pack(s, d), _graph(n, n // 2, 8)]))
    _check(provider, tc_plan(), [e, None], 1)


@pytest.mark.parametrize("n", [40, 5000])
def test_separate_seed(provider, n):
    _check(provider, copy_points_to_plan(), [_graph(n, n // 2, 3), _graph(n, 2 * n, 4), None], 2)


def test_iteration_limit(provider):
    s, d = datagen.chain(600)
    E = provider.create_buffer_from_u32_columns([s, d])
    outs, st = provider.fixpoint(tc_plan(), [E, None], max_iterations=599)
    assert st["iterations"] == 599 and st["delta_sizes"] == list(range(599, -1, -1))
    with pytest.raises(XlogError) as ex:
        provider.fixpoint(tc_plan(), [E, None], max_iterations=598)
    assert ex.value.status == ITERATION_LIMIT
    assert ex.value.stats["iterations"] == 598 and ex.value.stats["delta_sizes"] == list(range(599, 0, -1))
    del ex
