"""What the framework is timed on: the work a Datalog program gives it, through the provider's public methods.

A case is a dict of plain values whose "op" names one of these kinds of work:

  closure     transitive closure to its fixpoint (HipKernelProvider.fixpoint, route chosen by the library) of a random
              digraph; ids dense from 0 or, with "sparse", spread over the whole 32-bit range
  points_to   Andersen points-to (four mutually recursive rules) to its fixpoint
  triangles   a cyclic rule body over one edge relation, to its fixpoint
  join_dedup  one rule contribution: join, project, dedup in one call (join_project_dedup), Zipf keys on the left
  join        hash_join_v2 on one or two key columns, inner, semi (a filter) or anti (a negated atom)
  dedup       dedup of rows that repeat, on the whole row or on its first column
  delta       the set operations of one semi-naive iteration: new = candidates \\ full, full' = full + new

Inputs are made on the GPU from the seed and handed over as device columns; relations and provider are what a program
keeps between calls.  Outputs are tensors over the result relations' own words (8 bytes per two columns).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from xlog_amd import JOIN_ANTI, JOIN_INNER, JOIN_SEMI, HipKernelProvider, andersen_plan, datagen, tc_plan

_JOIN_TYPES = {"inner": JOIN_INNER, "semi": JOIN_SEMI, "anti": JOIN_ANTI}
# tri(X,Z) :- e(X,Y), e(Y,Z), e(X,Z)
_TRIANGLES = [1, 1, 0, 2, 3, 0, 0, 1, 0, 1, 2, 0, 0, 2]


def listed():
    return [
        # the smallest program: a call graph or a type hierarchy of a thousand names, bound by launches and read-backs
        {"name": "closure_small", "op": "closure", "vertices": 1000, "edges": 5000, "sparse": False},
        # the headline: reachability over a dense id domain, about 9.5e8 result tuples
        {"name": "closure_large", "op": "closure", "vertices": 32768, "edges": 98304, "sparse": False},
        # reachability over ids that are hashes or addresses, so no dense domain; many short iterations
        {"name": "closure_sparse_ids", "op": "closure", "vertices": 1 << 20, "edges": 943718, "sparse": True},
        # pointer analysis: non-linear, mutually dependent rules
        {"name": "points_to", "op": "points_to", "variables": 10_000, "facts": 40_000},
        # a cyclic body, which no chain of products evaluates
        {"name": "triangles", "op": "triangles", "vertices": 100_000, "edges": 3_000_000},
        # the heaviest rule contribution: 2^24 rows a side, skewed probe keys, about 2.7e8 output rows
        {"name": "join_dedup_large", "op": "join_dedup", "left": 1 << 24, "right": 1 << 24, "distinct": 1 << 20},
        # a single operator call of an operator-by-operator executor, at the reference benchmark's 100K rows a side
        {"name": "join_small", "op": "join", "type": "inner", "left": 100_000, "right": 100_000, "distinct": 50_000,
         "left_arity": 2, "right_arity": 2, "keys": 1},
        # joins of wider facts on a compound key (function and offset, relation and argument)
        {"name": "join_two_keys", "op": "join", "type": "inner", "left": 1 << 22, "right": 1 << 21,
         "distinct": 1 << 20, "left_arity": 3, "right_arity": 3, "keys": 2},
        # fact loading and rule results: a few thousand rows with repeats, a size that fills no tile
        {"name": "dedup_small", "op": "dedup", "rows": 5003, "arity": 2, "keys": "row"},
        # the same at the scale of a bulk load, 2^28 pairs
        {"name": "dedup_large", "op": "dedup", "rows": 1 << 28, "arity": 2, "keys": "row"},
        # facts of four columns
        {"name": "dedup_wide", "op": "dedup", "rows": 10_000_019, "arity": 4, "keys": "row"},
        # one iteration's set operations against a full relation that is far larger than the candidates
        {"name": "delta", "op": "delta", "full": 1 << 25, "candidates": 1 << 22, "ids": 1 << 20},
    ]


def _log_between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["closure", "closure_sparse", "points_to", "triangles", "join_dedup", "join", "join", "dedup",
                     "dedup", "delta"])
    if op == "closure":
        v = _log_between(rng, 500, 30_000)
        return {"op": "closure", "vertices": v, "edges": int(v * rng.uniform(1.2, 4.0)), "sparse": False}
    if op == "closure_sparse":
        v = _log_between(rng, 2_000, 1 << 20)
        return {"op": "closure", "vertices": v, "edges": int(v * rng.uniform(0.4, 0.9)), "sparse": True}
    if op == "points_to":
        v = _log_between(rng, 500, 10_000)
        return {"op": "points_to", "variables": v, "facts": 4 * v}
    if op == "triangles":
        v = _log_between(rng, 2_000, 100_000)
        return {"op": "triangles", "vertices": v, "edges": int(v * rng.uniform(5.0, 30.0))}
    if op == "join_dedup":
        right = _log_between(rng, 1_000, 1 << 24)
        return {"op": "join_dedup", "left": _log_between(rng, 1_000, 1 << 24), "right": right,
                "distinct": max(64, int(right / rng.uniform(4.0, 16.0)))}
    if op == "join":
        keys = rng.choice([1, 2])
        right = _log_between(rng, 1_000, 1 << 22)
        return {"op": "join", "type": rng.choice(["inner", "inner", "semi", "anti"]),
                "left": _log_between(rng, 1_000, 1 << 22), "right": right,
                "distinct": max(16, int(right / rng.uniform(1.0, 4.0))), "left_arity": rng.choice([2, 2, 3, 4]),
                "right_arity": rng.choice([2, 2, 3, 4]), "keys": keys}
    if op == "dedup":
        arity = rng.choice([1, 2, 2, 3, 4, 6])
        keys = rng.choice(["row", "row", "row", "first"]) if arity > 1 else "row"
        hi = 1 << 27 if arity <= 2 and keys == "row" else 10_000_000
        return {"op": "dedup", "rows": _log_between(rng, 1_000, hi), "arity": arity, "keys": keys}
    full = _log_between(rng, 10_000, 1 << 25)
    return {"op": "delta", "full": full, "candidates": max(1_000, int(full / rng.uniform(4.0, 64.0))),
            "ids": max(1 << 10, 1 << (full.bit_length() * 3 // 4))}


# -- inputs -------------------------------------------------------------------------------------------------

_state = {}


def _provider():
    if "p" not in _state:
        _state["p"] = HipKernelProvider(0)
    return _state["p"]


def _u32(col):
    """An int64 column of ids below 2^32 as the 32-bit words the library reads."""
    return torch.where(col >= 1 << 31, col - (1 << 32), col).to(torch.int32).contiguous()


def _relation(cols):
    p = _provider()
    words = [_u32(c) for c in cols]
    torch.cuda.synchronize()
    rel = p.create_buffer_from_device_columns([w.data_ptr() for w in words], len(words[0]))
    p.synchronize()
    return rel


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _ints(g, n, hi):
    return torch.randint(0, int(hi), (int(n),), generator=g, device="cuda", dtype=torch.int64)


def _order(g, n):
    return torch.argsort(torch.rand(int(n), generator=g, device="cuda", dtype=torch.float64))


def _spread(ids):
    """A bijection of the 32-bit ids: small dense ids become values from all over the range."""
    lo = (ids & 0xFFFF) * datagen.SPARSE_ID_MUL
    hi = (((ids >> 16) * datagen.SPARSE_ID_MUL) & 0xFFFF) << 16
    return (lo + hi + datagen.SPARSE_ID_ADD) & 0xFFFFFFFF


def _labels(g, top):
    """A seeded bijection of the ids below `top` (a power of two)."""
    odd, add = (int(v) for v in _ints(g, 2, top).tolist())
    return lambda ids: (ids * ((odd | 1) & 0x7FFFFFFF) + add) & (top - 1)


def _distinct_pairs(g, n, draw_col):
    """n distinct (a, b), a != b, in random order; draw_col(k) draws k ids."""
    got = torch.empty(0, dtype=torch.int64, device="cuda")
    while len(got) < n:
        k = int((n - len(got)) * 1.2) + 64
        a, b = draw_col(k), draw_col(k)
        got = torch.unique(torch.cat([got, ((a << 32) | b)[a != b]]))
    got = got[_order(g, len(got))[:n]]
    return got >> 32, got & 0xFFFFFFFF


def _by_rank(g, n, ranks, exponent):
    """n ranks with P(k) ~ (k + 1)^-exponent."""
    cdf = np.cumsum(np.arange(1, ranks + 1, dtype=np.float64) ** -exponent)
    cdf = torch.from_numpy(cdf / cdf[-1]).cuda()
    u = torch.rand(int(n), generator=g, device="cuda", dtype=torch.float64)
    return torch.searchsorted(cdf, u).clamp_(max=ranks - 1)


def _power_of_two(n):
    return 1 << max(1, int(n - 1).bit_length())


def prepare(case, seed):
    """The inputs' structure (which rows repeat, which ids meet) comes from the case, so that every seed has results of
    the same sizes; the seed gives the ids and the order of the rows."""
    g0, g, op = _generator(20240229), _generator(seed), case["op"]
    if op in ("closure", "triangles", "points_to"):
        n = case["variables"] if op == "points_to" else case["vertices"]
        name = _order(g, n)
        spread = _labels(g, 1 << 32)

        def facts(pairs):
            mix = _order(g, len(pairs[0]))
            cols = [name[c[mix]] for c in pairs]
            return _relation([spread(_spread(c)) for c in cols] if case.get("sparse") else cols)

        if op == "points_to":
            sizes = [case["facts"] * s // 10 for s in (4, 2, 2, 2)]  # assign, addressOf, load, store
            rels = [facts(_distinct_pairs(g0, s, lambda k: _by_rank(g0, k, n, 1.5))) for s in sizes]
            return {"op": "fixpoint", "plan": andersen_plan(), "rels": rels + [None], "idb": 4}
        edges = facts(_distinct_pairs(g0, case["edges"], lambda k: _ints(g0, k, n)))
        return {"op": "fixpoint", "plan": tc_plan() if op == "closure" else _TRIANGLES, "rels": [edges, None], "idb": 1}
    if op == "join_dedup":
        key, a, c = _labels(g, 1 << 32), _labels(g, 1 << 32), _labels(g, 1 << 32)
        r_b = key(_spread(_by_rank(g0, case["left"], case["distinct"], 1.1)))
        s_b = key(_spread(_ints(g0, case["right"], case["distinct"])))
        return {"op": op, "left": _relation([a(_ints(g0, case["left"], 1 << 32)), r_b]),
                "right": _relation([s_b, c(_ints(g0, case["right"], 1 << 32))])}
    if op == "join":
        d, sides = case["distinct"], []
        high = _labels(g, 1 << 32 if case["keys"] == 1 else _power_of_two(d + d // 4))
        low = _labels(g, 64)
        for rows, arity in ((case["left"], case["left_arity"]), (case["right"], case["right_arity"])):
            k = _ints(g0, rows, d if len(sides) else d + d // 4)  # a fifth of the left keys have no match
            key = [high(_spread(k))] if case["keys"] == 1 else [high(k >> 6), low(k & 63)]
            sides.append(_relation(key + [_ints(g, rows, 1 << 32) for _ in range(arity - len(key))]))
        return {"op": op, "left": sides[0], "right": sides[1], "on": list(range(case["keys"])),
                "type": _JOIN_TYPES[case["type"]]}
    if op == "dedup":
        rows, arity = case["rows"], case["arity"]
        fresh = rows - rows * 3 // 10  # three rows in ten repeat another
        pick = torch.cat([torch.arange(fresh, device="cuda"), _ints(g0, rows - fresh, fresh)])[_order(g, rows)]
        # pairs of hashed ids; of wider facts, a subject with a few rows, then attributes of small and large domains
        subjects = _power_of_two(fresh // 3)
        tops = [subjects if case["keys"] == "first" else 1 << 32, 1 << 32] if arity <= 2 else \
            [subjects, 1 << 12, 1 << 20, 1 << 32, 1 << 8, 1 << 16]
        cols = []
        for top in tops[:arity]:
            label = _labels(g, top)
            cols.append(label(_ints(g0, fresh, top))[pick])
        return {"op": op, "rel": _relation(cols), "cols": [0] if case["keys"] == "first" else None}
    label = _labels(g, case["ids"])
    full = [_ints(g0, case["full"], case["ids"]) for _ in range(2)]
    known = _ints(g0, case["candidates"] // 2, case["full"])  # half of the candidates are known already
    fresh = [_ints(g0, case["candidates"] - len(known), case["ids"]) for _ in range(2)]
    mix = _order(g, case["candidates"])
    candidates = [label(torch.cat([full[c][known], fresh[c]])[mix]) for c in range(2)]
    return {"op": op, "full": _provider().dedup_full_row(_relation([label(c) for c in full])),
            "candidates": _relation(candidates)}


# -- one pass -----------------------------------------------------------------------------------------------

class _Words:
    """One word array of a relation as torch reads device memory; keeps the relation alive."""

    def __init__(self, rel, word, rows):
        self.rel = rel
        self.__cuda_array_interface__ = {"shape": (rows,), "typestr": "<i8", "version": 2,
                                         "data": (_provider().device_words(rel, word), False)}


def _tensors(rel):
    rows = rel.num_rows()
    if rows == 0:
        return [torch.empty(0, dtype=torch.int64, device="cuda")]
    return [torch.as_tensor(_Words(rel, w, rows), device="cuda") for w in range((rel.arity + 1) // 2)]


def run(state):
    p, op = _provider(), state["op"]
    if op == "fixpoint":
        outs, stats = p.fixpoint(state["plan"], state["rels"])
        return {"tuples": _tensors(outs[state["idb"]]), "iterations": stats["iterations"],
                "deltas": np.asarray(stats["delta_sizes"], dtype=np.int64)}
    if op == "join_dedup":
        return _tensors(p.join_project_dedup(state["left"], state["right"], 1, 0, [0, 3]))
    if op == "join":
        return _tensors(p.hash_join_v2(state["left"], state["right"], state["on"], state["on"], state["type"]))
    if op == "dedup":
        if state["cols"] is None:
            return _tensors(p.dedup_full_row(state["rel"]))
        return _tensors(p.dedup(state["rel"], state["cols"]))
    new = p.diff_gpu(state["candidates"], state["full"])
    return {"new": _tensors(new), "full": _tensors(p.union_gpu(state["full"], new))}


# -- what a pass cannot do without ----------------------------------------------------------------------------

def _closure_tuples(n, degree):
    """Expected closure size of G(n, degree n): pairs of the giant component above degree 1, small trees below."""
    if degree < 1.0:
        return min(float(n) * n, n * degree / (1.0 - degree))
    s = 0.5
    for _ in range(200):
        s = 1.0 - math.exp(-degree * s)
    return max(1.0, (s * n) ** 2)


def _row_bytes(arity):
    return 8 * ((arity + 1) // 2)


def work(case):
    op = case["op"]
    if op == "closure":
        out = _closure_tuples(case["vertices"], case["edges"] / case["vertices"])
        moved = 8 * (case["edges"] + out)
    elif op == "points_to":
        moved = 8 * (case["facts"] + 5.8e6 * (case["variables"] / 1e4) ** 1.76)
    elif op == "triangles":
        m, n = case["edges"], case["vertices"]
        moved = 8 * (m + m * (1.0 - math.exp(-m * m / (float(n) ** 3))))
    elif op == "join_dedup":
        moved = 8 * (case["left"] + case["right"] + case["left"] * case["right"] / case["distinct"])
    elif op == "join":
        out = case["left"] * 0.8
        arity = case["left_arity"]
        if case["type"] == "inner":
            out, arity = out * case["right"] / case["distinct"], arity + case["right_arity"]
        elif case["type"] == "anti":
            out = case["left"] * 0.2
        moved = (case["left"] * _row_bytes(case["left_arity"]) + case["right"] * _row_bytes(case["right_arity"])
                 + out * _row_bytes(arity))
    elif op == "dedup":
        kept = 0.7 if case["keys"] == "row" else 0.3
        moved = case["rows"] * _row_bytes(case["arity"]) * (1.0 + kept)
    else:  # candidates and full read, new and full' written
        moved = 8 * (case["candidates"] * 1.5 + case["full"] * 2 + case["candidates"] * 0.5)
    return {"bytes": float(moved), "flops": 0.0}


def tolerance(case):
    """Relations are sets or bags of whole numbers in a fixed row order: every bit is the same."""
    return "exact"
