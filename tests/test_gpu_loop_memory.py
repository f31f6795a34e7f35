"""One-block iterations (k_rank_loop) whose memory ends: logs that outgrow
their room, and device memory budgets that refuse the log, its tables or the
delta between them.  A run that ends well equals the oracle's; one that is
refused leaves rows of the closure only, delta and full."""
import os

import numpy as np
import pytest

import oracle as O
import pra_amd
from programs import DELTA, FULL, distinct_u64, random_graph, tc_program, with_rowid

pytestmark = pytest.mark.gpu


def path(n, count=1):
    """`count` separate paths of n vertices"""
    ids = distinct_u64(n * count, n)
    return with_rowid([(ids[p * n + i], ids[p * n + i + 1]) for p in range(count) for i in range(n - 1)])


def fan(n, chain, degree, levels):
    """n sources into a chain that ends in a tree: the deltas are small until
    the sources reach the tree"""
    e = [(s, n) for s in range(n)] + [(n + i, n + i + 1) for i in range(chain - 1)]
    front, top = [n + chain - 1], n + chain
    for _ in range(levels):
        e += [(v, top + degree * i + j) for i, v in enumerate(front) for j in range(degree)]
        front = list(range(top, top + degree * len(front)))
        top = front[-1] + 1
    ids = distinct_u64(top, n)
    return with_rowid([(ids[a], ids[b]) for a, b in e])


def context(k, loop=True, budget=0):
    """fixed variants, so that a run's memory does not depend on timings"""
    os.environ["PRA_AUTOTUNE"], os.environ["PRA_RANK_LOOP"] = "0", str(int(loop))
    try:
        return pra_amd.Context(nbuckets=k, batch_size=1, hbm_budget=budget)
    finally:
        del os.environ["PRA_AUTOTUNE"], os.environ["PRA_RANK_LOOP"]


def closure(edges, k):
    o = O.Oracle(k)
    T, _, fix, _ = tc_program(o, edges)
    o.execute(1)
    return o.rows(T), o.history(fix), o.joined()


@pytest.mark.parametrize("k", [1, 8])
def test_log_outgrows_its_room(k):
    edges = path(700, 6)
    want = closure(edges, k)
    g = context(k)
    try:
        g.set_profiling(True)
        T, _, fix, _ = tc_program(g, edges)
        print(f"[loop memory] six paths of 700, k={k}", flush=True)
        g.execute()
        np.testing.assert_array_equal(g.rows(T), want[0])
        assert g.history(fix) == want[1] and g.joined() == want[2]
        # 256 iterations a launch at most, and one more wherever the log is full
        assert g.kernel_stats()["rank_loop"]["launches"] > (len(want[1]) + 255) // 256
    finally:
        g.close()


@pytest.mark.parametrize("name,edges", [("fan", fan(300, 6, 5, 3)), ("path600", path(600)),
                                        ("random400", random_graph(400, 600, 5))], ids=lambda v: v if isinstance(v, str) else "")
def test_a_refused_run_leaves_rows_of_the_closure(name, edges):
    want = closure(edges, 3)
    keys = {tuple(r) for r in want[0].tolist()}
    g = context(3)
    tc_program(g, edges)
    g.execute()
    peak = g.device_bytes()[1]
    g.close()
    outcomes = set()
    for i in range(60):
        budget = int(peak * 0.07 * 15 ** (i / 59))   # (the fan's delta is refused at about a tenth)
        print(f"[loop memory] {name} budget={budget}", flush=True)
        try:
            g = context(3, budget=budget)
        except pra_amd.PraError:
            continue
        try:
            T, _, fix, _ = tc_program(g, edges)
            try:
                g.execute()
            except pra_amd.PraError as e:
                assert "budget" in str(e)
                outcomes.add("refused")
                for v in (DELTA, FULL):
                    try:
                        rows = g.rows(T, v)
                    except pra_amd.PraError as e:
                        assert "budget" in str(e)
                        continue
                    assert {tuple(r) for r in rows.tolist()} <= keys
                continue
            outcomes.add("done")
            assert g.history(fix) == want[1]
            try:
                rows = g.rows(T)
            except pra_amd.PraError as e:
                assert "budget" in str(e)
                continue
            np.testing.assert_array_equal(rows, want[0])
        except pra_amd.PraError as e:
            assert "budget" in str(e)   # the load itself
        finally:
            g.close()
    assert outcomes == {"refused", "done"}


def outcome(edges, k, loop, budget):
    """rows and peak bytes, None when the budget refused them"""
    g = context(k, loop, budget)
    try:
        T = tc_program(g, edges)[0]
        try:
            g.execute()
            rows = g.rows(T)
        except pra_amd.PraError as e:
            assert budget and "budget" in str(e)
            return None
        return rows, g.device_bytes()[1]
    finally:
        g.close()


@pytest.mark.parametrize("edges", [random_graph(1100, 1430, 5), random_graph(2300, 2990, 5), random_graph(200, 500, 5),
                                   path(600)], ids=["random1100", "random2300", "random200", "path600"])
def test_budgets_that_the_general_launches_manage_with(edges):
    want, general = outcome(edges, 8, False, 0)
    loop = max(outcome(edges, 8, True, 0)[1], int(1.3 * general))
    for i in range(24):
        budget = int(general + (loop - general) * i / 23)
        print(f"[loop memory] budget={budget}", flush=True)
        for by_block in (False, True):
            got = outcome(edges, 8, by_block, budget)
            assert got is not None, (by_block, budget, general)
            np.testing.assert_array_equal(got[0], want)


def triples(b, edges):
    """the closure P of `edges`, and W(a, b, c) :- P(a, b), edge(a, c): a rank
    space of three columns beside it"""
    E, P, W = b.rel_create(2, 1, 500), b.rel_create(2, 1, 501), b.rel_create(3, 1, 502)
    b.load_rows(E, edges, FULL)
    seed = b.scc_create(False, 1)
    b.scc_add_relation(seed, E, False)
    b.scc_add_relation(seed, P, True)
    b.add_copy(seed, P, E, FULL, [1, 0])
    rec = b.scc_create(True, 2)
    for r, move in ((E, False), (P, True), (W, False)):
        b.scc_add_relation(rec, r, move)
    b.add_join(rec, P, P, DELTA, E, FULL, [3, 1])
    b.add_join(rec, W, P, DELTA, E, FULL, [0, 1, 3])
    b.add_dependency(seed, rec)
    return P, W


def test_ranked_membership_yields_to_a_budget():
    """its bitmap of new keys, a bit for every triple of values, is done
    without where that is what a budget lacks"""
    edges = random_graph(600, 700, 5)
    o = O.Oracle(3)
    want = triples(o, edges)
    o.execute(1)
    want = [o.rows(r) for r in want]
    g = context(3)
    rels = triples(g, edges)
    g.execute()
    peak = g.device_bytes()[1]
    g.close()
    bitmap = len(np.unique(edges[:, :2])) ** 3 // 8
    for tenths in range(10):
        budget = peak - bitmap * tenths // 10
        print(f"[loop memory] budget={budget} of {peak}", flush=True)
        g = context(3, budget=budget)
        try:
            rels = triples(g, edges)
            g.execute()
            for r, w in zip(rels, want):
                np.testing.assert_array_equal(g.rows(r), w)
        finally:
            g.close()
