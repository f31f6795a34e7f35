"""A value dictionary whose rebuild is refused by the memory budget: the rows
of a relation that was finished before, with a membership bitmap by the last
dictionary's ranks, are then put in order without it."""
import os

import numpy as np
import pytest

import oracle as O
import pra_amd
from programs import DELTA, FULL, layered_dag, random_graph, tc_program

pytestmark = pytest.mark.gpu


def program(b, edges, dag):
    """the closure of `edges`, then a fixpoint over `dag` whose rows carry the
    ids of earlier rows as key columns: values that no dictionary has yet"""
    T, _, fix, _ = tc_program(b, edges)
    X, H = b.rel_create(2, 1, 400), b.rel_create(2, 1, 401)
    b.load_rows(H, dag, FULL)
    seed = b.scc_create(False, 1)
    b.scc_add_relation(seed, H, False)
    b.scc_add_relation(seed, X, True)
    b.add_copy(seed, X, H, FULL, [1, 2])
    ids = b.scc_create(True, 2)
    b.scc_add_relation(ids, H, False)
    b.scc_add_relation(ids, X, True)
    b.add_join(ids, X, X, DELTA, H, FULL, [3, 2])
    b.add_dependency(fix, seed)
    b.add_dependency(seed, ids)
    return T


def context(k, budget=0):
    """fixed variants, so that a run's memory does not depend on timings"""
    os.environ["PRA_AUTOTUNE"] = "0"
    try:
        return pra_amd.Context(nbuckets=k, batch_size=1, hbm_budget=budget)
    finally:
        del os.environ["PRA_AUTOTUNE"]


@pytest.mark.parametrize("k", [1, 3])
@pytest.mark.parametrize("n,m", [(20, 420), (150, 7000)])
def test_finished_rows_after_a_refused_dictionary(n, m, k):
    edges, dag = random_graph(n, int(1.3 * n), n), layered_dag(6, nvert=m * 5 // 7, nlayers=6, nedges=m)
    o = O.Oracle(k)
    To = program(o, edges, dag)
    o.execute(1)
    want = o.rows(To)
    g = context(k)
    Tg = program(g, edges, dag)
    g.execute()
    np.testing.assert_array_equal(g.rows(Tg), want)
    peak = g.device_bytes()[1]
    g.close()
    refused = read = 0
    for i in range(100):
        budget = int(peak * (0.3 + 0.72 * i / 99))
        print(f"[dictionary] n={n} m={m} k={k} budget={budget}", flush=True)
        try:
            g = context(k, budget)
        except pra_amd.PraError:
            continue
        try:
            Tg = program(g, edges, dag)
            try:
                g.execute()
            except pra_amd.PraError as e:
                assert "budget" in str(e)
                refused += 1
                if g.count(Tg, DELTA) or g.count(Tg) != len(want):
                    continue   # refused before the closure's end
            rows = g.rows(Tg)
            read += 1
            np.testing.assert_array_equal(rows, want)
        except pra_amd.PraError as e:
            assert "budget" in str(e)
        finally:
            g.close()
    assert refused and read
