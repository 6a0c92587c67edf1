"""GPU parity of linear closures by row gathers over bit matrices, which the column-blocked closure leaves to them: more
than 32 edges a row (64 from 12,288 ids), and domains above 38,912 ids; several iterations, a separate seed relation, and
the iteration limit.  The launches show the route: products are queued several at a time, the columns take one in all."""
import numpy as np
import pytest

import oracle
from xlog_amd import XlogError, copy_points_to_plan, datagen, pack, tc_plan

pytestmark = pytest.mark.gpu

ITERATION_LIMIT = 4


def _run(p, plan, rels, columns=False, **kw):
    dev = [p.create_buffer_from_packed(r) if r is not None else None for r in rels]
    p.profile_enable(True)
    try:
        p.profile_reset()
        outs, st = p.fixpoint(plan, dev, **kw)
        ran = p.profile_read()["chain_product"]["launches"]
    finally:
        p.profile_enable(False)
    assert (ran == 1) == columns and ran >= 1, ran
    return outs, st


def _check(p, plan, rels, idb):
    outs_o, it_o, deltas_o = oracle.seminaive(plan, rels)
    outs, st = _run(p, plan, rels)
    assert np.array_equal(p.download_packed(outs[idb]), outs_o[idb])
    assert st["iterations"] == it_o and st["delta_sizes"] == deltas_o


def _layers(width, n, extra=0, seed=0):
    """n layers of `width` vertices, each vertex with an edge to every one of the next layer; `extra` random edges"""
    a, b = np.meshgrid(np.arange(width), np.arange(width), indexing="ij")
    s = np.concatenate([a.ravel() + i * width for i in range(n - 1)])
    d = np.concatenate([b.ravel() + (i + 1) * width for i in range(n - 1)])
    rng = np.random.default_rng(seed)
    s, d = (np.concatenate([x, rng.integers(0, width * n, extra)]) for x in (s, d))
    perm = rng.permutation(width * n)
    return np.unique(pack(perm[s], perm[d]))


@pytest.mark.parametrize("width,n,extra", [(40, 10, 0), (50, 3, 0), (43, 24, 0), (70, 15, 0), (70, 15, 3), (34, 60, 500),
                                           (130, 5, 40)])
def test_many_edges_a_row(provider, width, n, extra):
    e = _layers(width, n, extra)
    assert len(e) > 32 * width * n
    _check(provider, tc_plan(), [e, None], 1)


def test_many_edges_a_row_above_12288_ids(provider):
    one = _layers(100, 4)
    e = np.concatenate([one + np.uint64((400 * k << 32) + 400 * k) for k in range(31)])
    assert len(e) > 64 * 12400
    ref = oracle.bfs_tc(12400, (e >> np.uint64(32)).astype(np.uint32), e.astype(np.uint32))
    outs, st = _run(provider, tc_plan(), [e, None])
    assert np.array_equal(provider.download_packed(outs[1]), ref["relation"]) and st["iterations"] == ref["iterations"]


@pytest.mark.parametrize("nv,m", [(38912, 30000), (38913, 30000), (50001, 45000), (1 << 17, 100000)])
def test_domains_beside_the_columns(provider, nv, m):
    s, d = datagen.random_digraph(nv - 1, m, nv)
    s, d = np.append(s, nv - 1).astype(np.uint32), np.append(d, 0).astype(np.uint32)  # the largest id has an edge
    ref = oracle.bfs_tc(nv, s, d)
    outs, st = _run(provider, tc_plan(), [np.unique(pack(s, d)), None], nv == 38912)
    assert np.array_equal(provider.download_packed(outs[1]), ref["relation"]) and st["iterations"] == ref["iterations"]


def test_separate_seed(provider):
    rng = np.random.default_rng(4)
    f = _layers(45, 12)
    seed = np.unique(pack(rng.integers(0, 540, 300), rng.integers(0, 540, 300)))
    _check(provider, copy_points_to_plan(), [seed, f, None], 2)


def test_iteration_limit(provider):
    e = _layers(40, 10)
    outs, st = _run(provider, tc_plan(), [e, None], max_iterations=9)
    assert st["iterations"] == 9 and st["delta_sizes"] == [1600 * k for k in range(9, -1, -1)]
    with pytest.raises(XlogError) as ex:
        provider.fixpoint(tc_plan(), [provider.create_buffer_from_packed(e), None], max_iterations=8)
    assert ex.value.status == ITERATION_LIMIT
    assert ex.value.stats["iterations"] == 8
    del ex
