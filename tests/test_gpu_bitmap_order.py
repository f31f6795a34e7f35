"""Results put into trie order through the membership bitmap: rank spaces
around the 256-bit blocks and 64-bit words of the bitmap, one and several
buckets, one, two and three key columns.  Rows, ids included, must equal the
oracle's."""
import numpy as np
import pytest

import oracle as O
import pra_amd
from programs import DELTA, FULL, distinct_u64, tc_program, with_rowid

pytestmark = pytest.mark.gpu


def chain(b, n):
    ids = distinct_u64(n, 17 * n)
    T, _, _, _ = tc_program(b, with_rowid([(ids[i], ids[i + 1]) for i in range(n - 1)] + [(ids[n - 1], ids[0])]))
    return [T]


def columns(b, n, arity, jcc):
    """rows of `arity` columns copied out of a relation, three passes long"""
    rng = np.random.default_rng(n + arity)
    vals = distinct_u64(n, n)
    rows = np.unique(vals[rng.integers(0, n, size=(6 * n, arity))], axis=0)
    src, out = b.rel_create(arity, 1, 40), b.rel_create(arity, jcc, 41)
    b.load_rows(src, np.column_stack([rows, np.arange(len(rows), dtype=np.uint64)]), FULL)
    s = b.scc_create(True, 1)
    b.scc_add_relation(s, src, True)
    b.scc_add_relation(s, out, False)
    b.add_copy(s, out, src, DELTA, list(range(arity - 1, -1, -1)))
    if arity > 1:
        b.add_copy(s, out, out, DELTA, [1, 0] + list(range(2, arity)))
    return [out]


CASES = [(f"chain{n}", lambda b, n=n: chain(b, n)) for n in (2, 15, 16, 17, 33, 64, 90)] + [
    (f"cols{a}_{j}_{n}", lambda b, n=n, a=a, j=j: columns(b, n, a, j))
    for a, j in ((1, 1), (2, 1), (2, 2), (3, 1), (3, 2)) for n in (7, 40)]


@pytest.mark.parametrize("k", [1, 3, 16])
@pytest.mark.parametrize("name,build", CASES, ids=[c[0] for c in CASES])
def test_rows_equal_oracle(name, build, k):
    print(f"[bitmap order] {name} k={k}", flush=True)
    g, o = pra_amd.Context(k, batch_size=1), O.Oracle(k)
    try:
        gr, orr = build(g), build(o)
        g.execute()
        o.execute(1)
        for a, b in zip(gr, orr):
            np.testing.assert_array_equal(g.rows(a), o.rows(b))
    finally:
        g.close()
