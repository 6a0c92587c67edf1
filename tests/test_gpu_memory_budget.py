"""GPU checks of the context's device memory budget (the reference's
MemoryBudget::with_limit, crates/xlog-core/src/config.rs:39-45, enforced by
GpuMemoryManager, crates/xlog-cuda/src/memory.rs:756-770): an allocation past
it fails closed with OOM, the context stays usable, and the fixpoint's AUTO
route choice keeps its bit matrices within it (the result, iteration count
and delta sizes stay those of the oracle)."""
import gc
import sys

import numpy as np
import pytest

import oracle
from xlog_amd import ROUTE_AUTO, ROUTE_BITMAP, ROUTE_HASH, ROUTE_JOIN, XlogError, datagen, pack, tc_plan

pytestmark = pytest.mark.gpu
OOM = 5


def _note(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture
def p():
    """A context of its own: its pool holds nothing of the other tests (the
    session context keeps per-context look-back state sized by the largest
    sort it ran), so the budget counts only what these tests allocate."""
    from xlog_amd import HipKernelProvider

    gc.collect()
    prov = HipKernelProvider(0)
    try:
        yield prov
    finally:
        gc.collect()
        prov.close()


def test_budget_refuses_then_recovers(p):
    rng = np.random.default_rng(5)
    keys = rng.integers(0, 1 << 64, 1 << 20, dtype=np.uint64)
    rel = p.create_buffer_from_packed(keys)  # 8 MiB held
    p.trim()
    p.set_memory_budget(4 << 20)  # below what a sort of it needs
    with pytest.raises(XlogError) as ex:
        p.dedup_full_row(rel)
    assert ex.value.status == OOM
    assert "budget" in ex.value.message
    p.set_memory_budget(0)
    d = p.dedup_full_row(rel)
    assert np.array_equal(p.download_packed(d), oracle.sort_dedup(keys))
    # a budget that allows the operation gives the same result, within the budget
    p.set_memory_budget(256 << 20)
    d2 = p.dedup_full_row(rel)
    assert np.array_equal(p.download_packed(d2), oracle.sort_dedup(keys))
    st = p.memory_stats()
    assert st["in_use"] + st["cached"] <= 256 << 20, st
    p.set_memory_budget(0)


def test_budget_steers_auto_off_the_bitmap_route(p):
    """A transitive closure over 2^17 ids takes the bitmap route (2 GiB bit
    matrices) without a budget; with a 1 GiB budget AUTO takes the hash-set
    route instead, with the same relation, iterations and delta sizes."""
    nv = 1 << 17
    src, dst = datagen.random_digraph(nv, nv // 2, 77)  # sparse: short paths, small closure
    e = pack(src, dst)
    b = oracle.bfs_tc(nv, src, dst)
    it = b["iterations"]
    deltas = [int(x) for x in b["dist_count"][1:it + 1]] + [0]
    for budget, route in ((0, ROUTE_BITMAP), (1 << 30, ROUTE_HASH)):
        _note(f"budget {budget}: tc over {nv} ids")
        p.trim()
        p.set_memory_budget(budget)
        outs, st = p.fixpoint(tc_plan(), [p.create_buffer_from_packed(e), None], route=ROUTE_AUTO)
        assert st["route"] == route
        assert np.array_equal(p.download_packed(outs[1]), b["relation"])
        assert (st["iterations"], st["delta_sizes"]) == (it, deltas)
        del outs
    p.set_memory_budget(0)
    # an explicit bitmap request under a budget too small for it fails closed
    p.trim()
    p.set_memory_budget(1 << 30)
    with pytest.raises(XlogError) as ex:
        p.fixpoint(tc_plan(), [p.create_buffer_from_packed(e), None], route=ROUTE_BITMAP)
    assert ex.value.status == OOM
    p.set_memory_budget(0)


@pytest.mark.parametrize("where", ["rule2", "rule3_second_join"])
def test_failed_fixpoint_frees_its_device_memory(p, where):
    """A fixpoint stopped by the join-row limit (CAPACITY_OVERFLOW, the
    reference's relational.rs:4550-4555) gives back every block it took.  The
    limit trips in the first recursive iteration either on rule 2's join or on
    rule 3's second join, when rule 2's head tuples and rule 3's first join
    are held (join sizes from the oracle's counts, as for C5 at its stated
    size)."""
    from xlog_amd import andersen_plan

    f = datagen.andersen(2000, 8000, 1.5, datagen.seed_for(5))
    assign, addr, load = (oracle.sort_dedup(pack(*f[k])) for k in ("assign", "addressOf", "load"))
    r2 = oracle.chain2_counts(assign, addr, np.zeros(0, np.uint64))
    r3 = oracle.chain2_counts(load, addr, addr)
    if where == "rule2":
        limit = r2["bag1"] - 1
    else:
        limit = max(r2["bag1"], r3["bag1"])
        assert r3["bag2_over_bag1"] > limit
    rels = [p.create_buffer_from_u32_columns(list(f[k])) for k in ("assign", "addressOf", "load", "store")]

    def fail_once():
        with pytest.raises(XlogError) as ex:
            p.fixpoint(andersen_plan(), rels + [None], route=ROUTE_JOIN, max_join_rows=limit)
        assert ex.value.status == 3  # CAPACITY_OVERFLOW
        assert ex.value.stats["iterations"] == 1
        del ex
        gc.collect()
        return p.memory_stats()["in_use"]

    # the first run also sizes the context's persistent look-back state; the
    # second must end with exactly the live bytes it started with
    before = fail_once()
    assert fail_once() == before


def _block(nbytes):
    """What the pool takes for an allocation: four size classes per power of two."""
    if nbytes < 256:
        return 256
    q = 1 << max(0, nbytes.bit_length() - 3)
    return -(-nbytes // q) * q


@pytest.fixture
def within(p):
    """A function that runs a call with a budget of some bytes above what is held."""
    def run(nbytes, call):
        gc.collect()
        p.trim()
        p.set_memory_budget(p.memory_stats()["in_use"] + nbytes)
        try:
            return call()
        finally:
            p.set_memory_budget(0)
    return run


SLACK = 5 << 19  # counters and the digit passes' look-back state


@pytest.mark.parametrize("n", [100000, 1000000])
def test_sorts_in_two_buffers(p, within, n):
    """Sizes of the bucket sort, whose regions are four times the keys: without room for them the digit passes do."""
    keys = np.random.default_rng(n).integers(0, 1 << 64, n, dtype=np.uint64)
    rel = p.create_buffer_from_packed(keys)
    need = 2 * _block(8 * n) + SLACK
    assert np.array_equal(p.download_packed(within(need, lambda: p.dedup_full_row(rel))), np.unique(keys))
    assert np.array_equal(p.download_packed(within(need, lambda: p.sort(rel, [0, 1]))), np.sort(keys))


@pytest.mark.parametrize("arity,first", [(3, 1 << 32), (4, 1 << 32), (6, 3), (8, 1 << 32), (4, 1)])
@pytest.mark.parametrize("keys", ["all", "one"])
@pytest.mark.parametrize("n", [12000, 700000])
def test_row_sorts_without_a_copy_of_the_rows(p, within, arity, first, keys, n):
    """Room for four bytes per row beside the sorted rows, or for two words: the rows are not copied and the key goes by
    pieces."""
    rng = np.random.default_rng(n + arity)
    cols = [rng.integers(0, first if c == 0 else 1 << 32, n).astype(np.uint32) for c in range(arity)]
    rel = p.create_buffer_from_u32_columns(cols)
    by = list(range(arity)) if keys == "all" else [1]
    words = (arity + 1) // 2
    need = max(words * _block(8 * n) + _block(4 * n), 2 * _block(8 * n)) + (SLACK if n > 16384 else 1 << 16)
    out = within(need, lambda: p.sort(rel, by))
    order = np.lexsort([cols[c] for c in reversed(by)])
    for c in range(arity):
        assert np.array_equal(p.download_column(out, c), cols[c][order]), c
    del out
    cols[0][:] = cols[0][0]
    rel = p.create_buffer_from_u32_columns([np.concatenate([c, c]) for c in cols])  # every row twice
    out = within((3 * words + 1) * _block(16 * n) + SLACK, lambda: p.dedup(rel, by))
    order = np.lexsort([cols[c] for c in reversed(by)])
    first_of = np.ones(n, bool)
    first_of[1:] = np.any([cols[c][order][1:] != cols[c][order][:-1] for c in by], axis=0)
    for c in range(arity):
        assert np.array_equal(p.download_column(out, c), cols[c][order][first_of]), c


# bytes per build row above the inputs that each join took as an index over its sorted keys (one key) or by dictionaries
@pytest.mark.parametrize("kind,per_row", [("one", 100), ("few", 34), ("two", 96), ("two keys only", 96), ("wide", 92),
                                          ("direct", 104), ("two few", 30)])
@pytest.mark.parametrize("n", [300000, 1000000])
def test_joins_without_room_for_packed_keys(p, within, kind, per_row, n):
    """Joins and semi joins within what they took before keys were packed, by whatever route fits."""
    rng = np.random.default_rng(n)
    cols = lambda rows, *tops: [rng.integers(0, t, rows).astype(np.uint32) for t in tops]  # noqa: E731
    nl, on = n, [0, 1]
    if kind in ("one", "few"):
        on, nl = [0], n if kind == "one" else 1000
        tops = [100 if kind == "few" else n // 2, 1 << 32]
    elif kind == "wide":
        on, tops = [2], [50, 64, n]
    else:
        tops = [{"direct": 4 * n // 64, "two few": 50}.get(kind, n // 64), 64] + ([] if "only" in kind else [1 << 32])
        nl = 1000 if kind == "two few" else n
    left, right = cols(nl, *tops), cols(n, *tops)
    L, R = p.create_buffer_from_u32_columns(left), p.create_buffer_from_u32_columns(right)
    code = lambda c: sum(c[k].astype(np.int64) << (32 * i) for i, k in enumerate(on))  # noqa: E731
    hit = np.isin(code(left), code(right))
    from xlog_amd import JOIN_ANTI, JOIN_INNER, JOIN_SEMI

    semi_row = {"two": 40, "direct": 40, "two keys only": 31, "wide": 40}.get(kind, per_row)
    for how, keep in ((JOIN_SEMI, hit), (JOIN_ANTI, ~hit)):
        out = within(semi_row * n + SLACK, lambda: p.hash_join_v2(L, R, on, on, how))
        assert np.array_equal(p.download_column(out, 0), left[0][keep])
        del out
    if kind in ("few", "two few"):
        return  # (outputs of many rows a key)
    want = p.hash_join_v2(L, R, on, on, JOIN_INNER)
    want = [p.download_column(want, c) for c in range(want.arity)]
    got = within(per_row * n + SLACK, lambda: p.hash_join_v2(L, R, on, on, JOIN_INNER))
    for c, w in enumerate(want):
        assert np.array_equal(p.download_column(got, c), w), c


@pytest.mark.parametrize("nv,m,need", [(300, 300, 80_000), (1000, 900, 800_000), (1000, 1000, 900_000)])
def test_small_closures_without_room_for_column_lists(p, within, nv, m, need):
    """A closure over a small dense domain within what its bit matrices take."""
    src, dst = datagen.random_digraph(nv, m, 3)
    e = p.dedup_full_row(p.create_buffer_from_packed(pack(src, dst)))
    outs_o, it_o, deltas_o = oracle.seminaive(tc_plan(), [np.unique(pack(src, dst)), None])
    for budget in (need, 64 << 20):
        outs, st = within(budget, lambda: p.fixpoint(tc_plan(), [e, None]))
        assert np.array_equal(p.download_packed(outs[1]), outs_o[1])
        assert st["iterations"] == it_o and st["delta_sizes"] == deltas_o
        assert st["route"] == ROUTE_BITMAP
        del outs


def test_difference_in_its_own_output(p, within):
    """The difference of sets by merge keeps a flag per key; without room for it the keys' windows are searched."""
    rng = np.random.default_rng(1)
    a, b = (np.unique(rng.integers(0, 1 << 22, 2_000_000, dtype=np.uint64)) for _ in range(2))
    A, B = (p.dedup_full_row(p.create_buffer_from_packed(k)) for k in (a, b))
    want = np.setdiff1d(a, b)
    assert np.array_equal(p.download_packed(p.diff_gpu(A, B)), want)  # (sizes the context's look-back state)
    assert np.array_equal(p.download_packed(within(_block(8 * len(a)) + (1 << 17), lambda: p.diff_gpu(A, B))), want)
