"""The work a user of this framework has it do, as cases that can be timed and
compared: Datalog programs run to their fixed point through the program-building
calls of parallel-ra_amd/pra_amd.py, the batched and served forms, and the two
device steps a program can call alone (bucket partition, relation load).

A case is a dict of plain values.  `prepare` makes its inputs from a seed,
`run` is one pass through the public entry points and returns its outputs
whole (result rows with their intern ids, delta history, counts), `work` the
bytes that the pass cannot do without.  Every output is a whole number.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "parallel-ra_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "parallel-ra_amd"))

import pra_amd  # noqa: E402

DELTA, FULL = pra_amd.DELTA, pra_amd.FULL


def listed():
    return [
        # a one-shot program on a tiny graph: context, program, fixed point and
        # rows once, as a test or a small query does; launches and host calls
        dict(name="one_shot_tc_v40", program="tc", graph="random", n=40, m=60, buckets=3, batch=1, context="new"),
        # the smallest and a middle request of the batched / served size range,
        # solved alone in a context that stays
        dict(name="tc_random_v1000", program="tc", graph="random", n=1000, m=1300, buckets=8, batch=1, context="kept"),
        dict(name="tc_random_v10007", program="tc", graph="random", n=10007, m=13009, buckets=8, batch=1,
             context="kept"),
        # a large random graph on one bucket, the fixed-point test every ten
        # iterations (LIE's own batch size)
        dict(name="tc_random_v20000_b10", program="tc", graph="random", n=20000, m=26000, buckets=1, batch=10,
             context="kept"),
        # the benchmark's own workload: the 150 x 150 grid, eight buckets
        dict(name="tc_grid150", program="tc", graph="grid", n=150, buckets=8, batch=1, context="kept"),
        # same generation on a layered DAG: joins, an acopy re-key and a filter
        dict(name="same_generation_v10000", program="sg", n=10000, layers=12, m=14000, buckets=8, batch=1),
        # doubling transitive closure: few iterations, many join pairs a tuple,
        # a join side that grows every iteration
        dict(name="doubling_tc_grid28", program="nltc", n=28, buckets=4, batch=1),
        # field-sensitive points-to analysis: eight relations, ten rules,
        # rows of two and three columns, long runs of small iterations
        dict(name="points_to_v4000", program="points_to", n=4000, buckets=3, batch=1),
        # sixty small programs in lock step in one context
        dict(name="lock_step_60", program="batch", count=60, nmin=200, nmax=1500, buckets=8),
        # a burst of requests to the server, rows read back
        dict(name="serve_24", program="serve", count=24, nmin=200, nmax=1500, buckets=8, slots=8),
        # the bucket partition of an exchange, alone, on device rows
        dict(name="partition_24m", program="partition", n=24000000, w=3, jcc=1, buckets=8, noalloc=False),
        # a relation loaded from host rows and walked in trie order
        dict(name="load_w4_2m", program="load", n=2000003, w=4, jcc=1, buckets=8, span=1 << 40),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tc", "tc", "tc", "grid", "grid", "sg", "nltc", "points_to", "batch", "serve", "partition",
                       "partition", "load", "load"])
    buckets = rng.choice([1, 2, 3, 4, 5, 8, 8, 13, 16])
    if kind == "tc":
        n = _log_int(rng, 30, 19000)
        return dict(program="tc", graph="random", n=n, m=int(n * rng.uniform(1.2, 1.35)), buckets=buckets,
                    batch=rng.choice([1, 1, 2, 10]), context=rng.choice(["kept", "kept", "new"]))
    if kind == "grid":
        return dict(program="tc", graph="grid", n=_log_int(rng, 5, 140), buckets=buckets,
                    batch=rng.choice([1, 1, 2, 10]), context=rng.choice(["kept", "kept", "new"]))
    if kind == "sg":
        n = _log_int(rng, 300, 10000)
        return dict(program="sg", n=n, layers=rng.randint(5, 13), m=int(n * rng.uniform(1.1, 1.4)), buckets=buckets,
                    batch=rng.choice([1, 3]))
    if kind == "nltc":
        return dict(program="nltc", n=rng.randint(4, 28), buckets=buckets, batch=rng.choice([1, 2]))
    if kind == "points_to":
        return dict(program="points_to", n=_log_int(rng, 100, 4500), buckets=buckets, batch=rng.choice([1, 10]))
    if kind == "batch":
        nmin = _log_int(rng, 40, 400)
        return dict(program="batch", count=rng.randint(2, 60), nmin=nmin, nmax=int(nmin * rng.uniform(1, 4)),
                    buckets=buckets)
    if kind == "serve":
        nmin = _log_int(rng, 40, 400)
        return dict(program="serve", count=rng.randint(2, 24), nmin=nmin, nmax=int(nmin * rng.uniform(1, 4)),
                    buckets=buckets, slots=rng.randint(1, 12))
    if kind == "partition":
        w = rng.randint(2, 6)
        noalloc = rng.random() < 0.4
        n = _log_int(rng, 1000, 8000000 if noalloc else 64000000 // w)
        return dict(program="partition", n=n, w=w, jcc=rng.randint(1, min(w - 1, 3)),
                    buckets=rng.choice([2, 3, 8, 16, 64, 200]), noalloc=noalloc)
    w = rng.randint(2, 6)
    return dict(program="load", n=_log_int(rng, 300, 6000000 // w), w=w, jcc=rng.randint(1, w - 1), buckets=buckets,
                span=rng.choice([1 << 12, 1 << 24, 1 << 40, 1 << 63]))


# ------------------------------------------------------------------ inputs ---

def _ids(rng, n):
    """n distinct uint64 values in random order"""
    ids = np.empty(0, dtype=np.uint64)
    while ids.size < n:
        more = rng.integers(0, 2**64 - 1, size=n + 64, dtype=np.uint64, endpoint=True)
        ids = np.unique(np.concatenate([ids, more]))
    return ids[rng.permutation(ids.size)[:n]]


def _with_id(pairs):
    """rows as a program loads them: the columns, then the row id"""
    p = np.asarray(pairs, dtype=np.uint64)
    return np.ascontiguousarray(np.column_stack([p, np.arange(len(p), dtype=np.uint64)]))


def _distinct(cols):
    """the distinct rows among integer columns, in first-draw order"""
    a = np.stack(cols, axis=1)
    _, first = np.unique(a, axis=0, return_index=True)
    return a[np.sort(first)]


def _random_edges(rng, n, m):
    """m distinct edges (fewer on a graph that has not so many) without self-loops"""
    m = min(m, n * (n - 1) // 2)
    k = 2 * m + 64
    while True:
        u, v = rng.integers(0, n, size=k), rng.integers(0, n, size=k)
        e = u[u != v] * n + v[u != v]
        _, first = np.unique(e, return_index=True)
        if first.size >= m:
            e = e[np.sort(first)[:m]]
            return np.stack([e // n, e % n], axis=1)
        k *= 2


def _grid_edges(n):
    idx = np.arange(n * n, dtype=np.int64).reshape(n, n)
    return np.concatenate([np.stack([idx[:, :-1].ravel(), idx[:, 1:].ravel()], axis=1),
                           np.stack([idx[:-1, :].ravel(), idx[1:, :].ravel()], axis=1)])


def _layered_edges(rng, n, layers, m):
    """m random edges from each layer of a DAG to the next"""
    bounds = (np.arange(layers + 1, dtype=np.int64) * n) // layers
    last = bounds[layers - 1]
    u = rng.integers(0, last, size=m + m // 4 + 16)
    layer = np.searchsorted(bounds, u, side="right") - 1
    lo, hi = bounds[layer + 1], bounds[layer + 2]
    v = lo + (rng.random(u.size) * (hi - lo)).astype(np.int64)
    return _distinct([u, v])[:m]


def _points_to_input(rng, ids, n):
    """n variables, n / 4 objects, four fields: allocations, assignments that
    mostly stay inside a function of forty variables, loads and stores"""
    nobj = max(2, n // 4)
    objs = np.arange(nobj)
    new = np.stack([rng.integers(0, n, size=nobj), objs + n], axis=1)

    def near(u):
        """a variable of u's function, or any variable for one in twelve"""
        f = np.minimum(u // 40 * 40 + rng.integers(0, 40, size=u.size), n - 1)
        return np.where(rng.random(u.size) < 1 / 12, rng.integers(0, n, size=u.size), f)

    s = rng.integers(0, n, size=int(0.95 * n))
    assign = _distinct([s, near(s)])
    assign = assign[assign[:, 0] != assign[:, 1]]
    b = rng.integers(0, n, size=max(2, n // 6))
    load = _distinct([b, rng.integers(0, 4, size=b.size) + n + nobj, near(b)])
    b = rng.integers(0, n, size=max(2, n // 6))
    store = _distinct([b, rng.integers(0, 4, size=b.size) + n + nobj, near(b)])
    ids = _ids(ids, n + nobj + 4)
    return {k: _with_id(ids[v]) for k, v in (("new", new), ("assign", assign), ("load", load), ("store", store))}


def _sizes(case):
    """vertex counts of a batch's or a burst's graphs, spread evenly over the
    logarithm of the range"""
    lo, hi, k = case["nmin"], max(case["nmax"], case["nmin"]), case["count"]
    return [int(round(lo * (hi / lo) ** (i / max(1, k - 1)))) for i in range(k)]


def _tc_edges(rng, ids, n, m=None, graph="random"):
    if graph == "grid":
        return _with_id(_ids(ids, n * n)[_grid_edges(n)])
    return _with_id(_ids(ids, n)[_random_edges(rng, n, int(1.3 * n) if m is None else m)])


# ---------------------------------------------------------------- programs ---

def _build_tc(c, edges):
    """T(z, x) for every path x -> z: seeded by a copy of the edges, closed by
    the join of T's delta with the edges"""
    T, G = c.rel_create(2, 1, 257), c.rel_create(2, 1, 256)
    c.load_rows(G, edges, FULL)
    fix = c.scc_create(True, 1)
    c.scc_add_relation(fix, G, False)
    c.scc_add_relation(fix, T, True)
    c.add_join(fix, T, T, DELTA, G, FULL, [3, 1])
    seed = c.scc_create(False, 2)
    c.scc_add_relation(seed, G, False)
    c.scc_add_relation(seed, T, True)
    c.add_copy(seed, T, G, FULL, [1, 0])
    c.add_dependency(seed, fix)
    return [T], fix


def _build_sg(c, edges):
    """sg(x, y) :- edge(p, x), edge(p, y), x != y
    sg(x, y) :- edge(a, x), sg(a, b), edge(b, y)"""
    E, sib, SG = c.rel_create(2, 1, 300), c.rel_create(2, 1, 301), c.rel_create(2, 1, 302)
    A, B = c.rel_create(2, 1, 303), c.rel_create(2, 1, 304)
    c.load_rows(E, edges, FULL)
    base = c.scc_create(False, 1)
    c.scc_add_relation(base, E, False)
    c.scc_add_relation(base, sib, False)
    c.add_join(base, sib, E, FULL, E, FULL, [1, 3])
    filt = c.scc_create(False, 2)
    c.scc_add_relation(filt, sib, True)
    c.scc_add_relation(filt, SG, False)
    c.add_copy_filter(filt, SG, sib, DELTA, [0, 1], pra_amd.F_NEQ)
    rec = c.scc_create(True, 3)
    c.scc_add_relation(rec, E, False)
    for r, move in ((SG, True), (A, False), (B, False)):
        c.scc_add_relation(rec, r, move)
    c.add_join(rec, A, SG, DELTA, E, FULL, [3, 1])
    c.add_acopy(rec, B, A, DELTA, [1, 0, 2])
    c.add_join(rec, SG, B, DELTA, E, FULL, [1, 3])
    c.add_dependency(base, filt)
    c.add_dependency(filt, rec)
    return [SG, A], rec


def _build_nltc(c, edges):
    """t(x, z) :- t(x, y), t(y, z), through an index of t on its second column"""
    T, R = c.rel_create(2, 1, 410), c.rel_create(2, 1, 411)
    c.load_rows(T, edges, FULL)
    s = c.scc_create(True, 1)
    c.scc_add_relation(s, T, True)
    c.scc_add_relation(s, R, False)
    c.add_acopy(s, R, T, DELTA, [1, 0, 2])
    c.add_join(s, T, R, DELTA, T, FULL, [1, 3])
    c.add_join(s, T, R, FULL, T, DELTA, [1, 3])
    return [T, R], s


def _build_points_to(c, e):
    """pt(v, o) :- new(v, o)                     pt(d, o) :- assign(s, d), pt(s, o)
    la(o, f, d) :- load(b, f, d), pt(b, o)    pt(d, q) :- la(o, f, d), heap(o, f, q)
    sa(s, o, f) :- store(b, f, s), pt(b, o)   heap(o, f, q) :- sa(s, o, f), pt(s, q)
    each rule over two recursive relations as DELTA x FULL, FULL x DELTA and
    DELTA x DELTA"""
    new, assign = c.rel_create(2, 1, 500), c.rel_create(2, 1, 501)
    load, store = c.rel_create(3, 1, 502), c.rel_create(3, 1, 503)
    pt, la = c.rel_create(2, 1, 504), c.rel_create(3, 2, 505)
    sa, heap = c.rel_create(3, 1, 506), c.rel_create(3, 2, 507)
    for r, k in ((new, "new"), (assign, "assign"), (load, "load"), (store, "store")):
        c.load_rows(r, e[k], FULL)
    base = c.scc_create(False, 1)
    c.scc_add_relation(base, new, False)
    c.scc_add_relation(base, pt, False)
    c.add_copy(base, pt, new, FULL, [0, 1])
    rec = c.scc_create(True, 2)
    for r in (assign, load, store):
        c.scc_add_relation(rec, r, False)
    for r, move in ((pt, True), (la, False), (sa, False), (heap, False)):
        c.scc_add_relation(rec, r, move)
    c.add_join(rec, pt, pt, DELTA, assign, FULL, [3, 1])
    c.add_join(rec, la, pt, DELTA, load, FULL, [1, 3, 4])
    c.add_join(rec, sa, pt, DELTA, store, FULL, [4, 1, 3])
    for v0, v1 in ((DELTA, FULL), (FULL, DELTA), (DELTA, DELTA)):
        c.add_join(rec, pt, la, v0, heap, v1, [2, 4])
        c.add_join(rec, heap, sa, v0, pt, v1, [1, 2, 4])
    c.add_dependency(base, rec)
    return [pt, heap, la, sa], rec


_BUILD = {"tc": _build_tc, "sg": _build_sg, "nltc": _build_nltc, "points_to": _build_points_to}


class _Words:
    """device rows as the array interface shows them (int64, since sums and
    comparisons of unsigned words are not everywhere).  The tensor made of one
    keeps it, and it keeps the context whose memory the rows are in."""

    def __init__(self, c, ptr, n, w):
        self.context = c
        self.__cuda_array_interface__ = {"shape": (n, w), "typestr": "<i8", "data": (ptr, False), "version": 2,
                                         "strides": None}


def _device_rows(c, rel):
    """a relation's full rows in trie order, where they lie on the device"""
    ptr, n = ctypes.POINTER(ctypes.c_uint64)(), ctypes.c_uint64()
    c._chk(c.L.pra_rel_device_rows(c.rels[rel], FULL, ctypes.byref(ptr), ctypes.byref(n)), "device_rows")
    if not n.value:
        return torch.empty((0, c.arity[rel] + 1), dtype=torch.int64, device="cuda")
    return torch.as_tensor(_Words(c, ctypes.cast(ptr, ctypes.c_void_p).value, n.value, c.arity[rel] + 1),
                           device="cuda")


def prepare(case, seed):
    """The seed draws the values; the shape of a graph is its case's, so that
    every seed closes to as many rows."""
    ids = np.random.default_rng(seed)
    rng = np.random.default_rng([case.get("n", case.get("nmin")), case.get("m", 0), case["buckets"]])
    p = case["program"]
    state = {"case": case}
    if p == "tc":
        state["input"] = _tc_edges(rng, ids, case["n"], case.get("m"), case["graph"])
    elif p == "sg":
        state["input"] = _with_id(_ids(ids, case["n"])[_layered_edges(rng, case["n"], case["layers"], case["m"])])
    elif p == "nltc":
        state["input"] = _tc_edges(rng, ids, case["n"], graph="grid")
    elif p == "points_to":
        state["input"] = _points_to_input(rng, ids, case["n"])
    elif p in ("batch", "serve"):
        sizes = _sizes(case)
        state["input"] = [_tc_edges(rng, ids, n) for n in [sizes[i] for i in rng.permutation(len(sizes))]]
    elif p == "partition":
        n, w = case["n"], case["w"]
        g = torch.Generator(device="cuda").manual_seed(int(seed))
        state["input"] = torch.randint(-2**63, 2**63 - 1, (n, w), dtype=torch.int64, device="cuda", generator=g)
        state["rows"] = torch.empty_like(state["input"])
        state["bounds"] = torch.empty(case["buckets"] + 1, dtype=torch.int64, device="cuda")
    else:
        a = ids.integers(0, case["span"], size=(case["n"], case["w"] - 1), dtype=np.uint64)
        state["input"] = _with_id(a)
    if case.get("context") != "new" and p != "serve":
        state["ctx"] = pra_amd.Context(nbuckets=case["buckets"], batch_size=case.get("batch", 1))
        state["ctx"].synchronize()
    return state


def _solve(c, build, data):
    out, scc = build(c, data)
    c.execute()
    return out, scc


def run(state):
    case = state["case"]
    p = case["program"]
    if p == "partition":
        c, x = state["ctx"], state["input"]
        f = c.partition_rows_noalloc if case["noalloc"] else c.partition_rows
        f(x.data_ptr(), case["n"], case["w"], case["jcc"], state["rows"].data_ptr(), state["bounds"].data_ptr())
        if case["noalloc"]:
            c.synchronize()   # calls from several contexts must not overlap on the shared scratch
        return state["rows"], state["bounds"]
    if p == "serve":
        s = pra_amd.Server(nbuckets=case["buckets"], slots=case["slots"], keep_rows=True)
        tickets = [s.submit(e) for e in state["input"]]
        res = [s.wait(t) for t in tickets]
        rows = [s.rows(t) for t in tickets]
        s.close()
        counts = np.array([[r["status"], r["tuples"], r["joined"], r["iterations"]] for r in res], dtype=np.int64)
        return np.concatenate(rows).view(np.int64), counts
    if case.get("context") == "new":
        c = state["ctx"] = pra_amd.Context(nbuckets=case["buckets"], batch_size=case["batch"])
    else:
        c = state["ctx"]
        for g in range(state.get("groups", 1)):
            c.release_group(g)
    if p == "load":
        c.set_group(0)
        r = c.rel_create(case["w"] - 1, case["jcc"], 1)
        c.load_rows(r, state["input"], FULL)
        return _device_rows(c, r)
    if p == "batch":
        state["groups"] = len(state["input"])
        made = []
        for g, e in enumerate(state["input"]):
            c.set_group(g)
            made.append(_build_tc(c, e))
        c.execute()
        rows = [_device_rows(c, out[0]) for out, _ in made]
        joined = [c.group_joined(g) for g in range(len(made))]
        return rows, np.array(joined, dtype=np.int64)
    c.set_group(0)
    out, scc = _solve(c, _BUILD[p], state["input"])
    return [_device_rows(c, r) for r in out], np.array(c.history(scc), dtype=np.int64), c.group_joined(0)


def work(case):
    """Inputs read once, results written once (24 bytes a binary row).  Sizes
    of results: exact for grids; 0.18 n^2 paths on random graphs of 1.3 edges a
    vertex, and measured growth laws for the others."""
    p = case["program"]

    def tc(n):
        return 24 * (1.3 * n + 0.18 * n * n)

    if p in ("tc", "nltc") and case.get("graph", "grid") == "grid":
        n = case["n"]
        facts = (n * (n + 1) // 2) ** 2 - n * n
        b = 24 * (2 * n * (n - 1) + facts * (2 if p == "nltc" else 1))
    elif p == "tc":
        b = tc(case["n"])
    elif p == "sg":
        b = 24 * (case["m"] + 200 * case["n"])
    elif p == "points_to":
        b = 24 * 60 * case["n"]
    elif p in ("batch", "serve"):
        b = sum(tc(n) for n in _sizes(case))
    elif p == "partition":
        b = 2 * 8 * case["n"] * case["w"]
    else:
        b = 2 * 8 * case["n"] * case["w"]
    return {"bytes": float(b), "flops": 0.0}
