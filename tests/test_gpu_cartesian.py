"""Joins without join columns (every pair of rows matches) over relations that
change in the SCC, whose runs are searched in sorted rows: FULL and DELTA
inners of fewer and more rows than the four that are compared at once, with
values on either side of the outer rows'.  Rows, ids included, per-batch
deltas and join pairs must equal the oracle's."""
import numpy as np
import pytest

import oracle as O
from programs import DELTA, FULL, distinct_u64, with_rowid

pytestmark = pytest.mark.gpu


def cartesian_program(b, base, seed):
    """P(a, d) :- P(a, b), P(c, d) from `base` in P's full version and `seed`
    as its first delta"""
    P, S = b.rel_create(2, 0, 310), b.rel_create(2, 0, 311)
    b.load_rows(P, base, FULL)
    b.load_rows(S, seed, FULL)
    s = b.scc_create(True, 1)
    b.scc_add_relation(s, P, False)
    b.scc_add_relation(s, S, True)
    b.add_copy(s, P, S, DELTA, [0, 1])
    for v0, v1 in ((DELTA, FULL), (FULL, DELTA), (DELTA, DELTA)):
        b.add_join(s, P, P, v0, P, v1, [0, 4])
    return P, s


@pytest.mark.parametrize("k", [1, 3, 8])
@pytest.mark.parametrize("nbase,nseed", [(1, 1), (3, 2), (4, 4), (5, 3), (9, 1), (40, 6)])
def test_cartesian_join_of_a_changing_relation(nbase, nseed, k):
    import pra_amd
    ids = distinct_u64(2 * (nbase + nseed), 17 * nbase + nseed).reshape(-1, 2)
    base, seed = with_rowid(ids[:nbase]), with_rowid(ids[nbase:])
    o = O.Oracle(k)
    Po, so = cartesian_program(o, base, seed)
    o.execute(1)
    assert o.rows(Po).shape[0] == (nbase + nseed) ** 2
    g = pra_amd.Context(nbuckets=k, batch_size=1)
    try:
        Pg, sg = cartesian_program(g, base, seed)
        print(f"[cartesian] base={nbase} seed={nseed} k={k}", flush=True)
        g.execute()
        np.testing.assert_array_equal(g.rows(Pg), o.rows(Po))
        assert g.history(sg) == o.history(so)
        assert g.joined() == o.joined()
    finally:
        g.close()


@pytest.mark.parametrize("k", [1, 3])
@pytest.mark.parametrize("n", [1, 5, 4096, 4097])
def test_cartesian_join_with_a_static_relation(n, k):
    import pra_amd
    ids = distinct_u64(2 * (n + 3), n).reshape(-1, 2)
    rows, few = with_rowid(ids[:n]), with_rowid(ids[n:])

    def program(b):
        Q, S, T = b.rel_create(2, 0, 310), b.rel_create(2, 0, 311), b.rel_create(2, 1, 312)
        b.load_rows(Q, rows, FULL)
        b.load_rows(S, few, FULL)
        s = b.scc_create(True, 1)
        b.scc_add_relation(s, Q, False)
        b.scc_add_relation(s, S, True)
        b.scc_add_relation(s, T, False)
        b.add_join(s, T, S, DELTA, Q, FULL, [0, 4])
        return T, s

    o = O.Oracle(k)
    To, so = program(o)
    o.execute(1)
    g = pra_amd.Context(nbuckets=k, batch_size=1)
    try:
        Tg, sg = program(g)
        print(f"[cartesian] static inner of {n} rows, k={k}", flush=True)
        g.execute()
        np.testing.assert_array_equal(g.rows(Tg), o.rows(To))
        assert g.history(sg) == o.history(so)
        assert g.joined() == o.joined()
    finally:
        g.close()
