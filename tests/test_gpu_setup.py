"""The dictionary and the join index of an instance, each built by one block up
to a size and by the general kernels above it: value and row counts on both
sides of those sizes and of a block's chunks, the value of all ones (the LDS
table's empty mark), and more relations than one launch reads.  Rows, ids
included, per-batch deltas and join pairs must equal the oracle's."""
import threading

import numpy as np
import pytest

import oracle as O
import pra_amd
from programs import FULL, distinct_u64, tc_program, with_rowid

pytestmark = pytest.mark.gpu


def layers(values, rows):
    """rows edges over exactly `values` values, the last of them 2^64 - 1,
    three layers deep, some sources with many targets"""
    ids = [v for v in distinct_u64(values, values) if v != 2**64 - 1][:values - 1] + [2**64 - 1]
    ids += [v for v in range(7) if v not in ids][:values - len(ids)]
    m = values // 3
    a, b, c, rest = ids[:m], ids[m:2 * m], ids[2 * m:3 * m], ids[3 * m:]
    if not m:
        return with_rowid([(ids[0], ids[1])])
    e = [(a[i], b[i]) for i in range(m)] + [(b[i], c[i]) for i in range(m)] + [(a[0], r) for r in rest]
    j = 1
    while len(e) < rows:
        e += [(a[i], b[(i + j) % m]) for i in range(min(rows - len(e), m))]
        j += 1
    assert len(set(e)) == len(e)
    return with_rowid(e)


def check(build, k):
    g, o = pra_amd.Context(k, batch_size=1), O.Oracle(k)
    try:
        Tg, fg = build(g)
        To, fo = build(o)
        g.execute()
        o.execute(1)
        np.testing.assert_array_equal(g.rows(Tg), o.rows(To))
        assert g.history(fg) == o.history(fo)
        assert g.joined() == o.joined()
    finally:
        g.close()


SIZES = [(2, 1), (3, 2), (64, 80), (1500, 1024), (1500, 1025), (700, 4096), (700, 4097), (4095, 4000), (4096, 4096),
         (4097, 4097), (6000, 4095)]


@pytest.mark.parametrize("k", [1, 3, 256])
@pytest.mark.parametrize("values,rows", SIZES)
def test_tc_equals_oracle(values, rows, k):
    print(f"[setup] values={values} rows={rows} k={k}", flush=True)
    edges = layers(values, rows)

    def build(b):
        T, _, fix, _ = tc_program(b, edges)
        return T, fix

    check(build, k)


@pytest.mark.parametrize("more", [13, 14, 15, 16])
def test_many_relations(more):
    """relations beside the program's two, with values of their own"""
    edges = layers(64, 80)

    def build(b):
        for r in range(more):
            b.load_rows(b.rel_create(2, 1, 300 + r), np.array([[r, r + 1, r]], dtype=np.uint64), FULL)
        T, _, fix, _ = tc_program(b, edges)
        return T, fix

    check(build, 3)


def test_contexts_that_come_and_go():
    """contexts made, used and closed by three threads at once take over each
    other's streams, pinned blocks and idle device blocks"""
    want = {}
    for n in (64, 700):
        o = O.Oracle(3)
        T, *_ = tc_program(o, layers(n, n + 20))
        o.execute(1)
        want[n] = o.rows(T)
    bad = []

    def user(k):
        for i in range(12):
            n = (64, 700)[(i + k) % 2]
            g = pra_amd.Context(3, batch_size=1)
            T, *_ = tc_program(g, layers(n, n + 20))
            g.execute()
            if not np.array_equal(g.rows(T), want[n]):
                bad.append((k, i))
            g.close()

    users = [threading.Thread(target=user, args=(k,)) for k in range(3)]
    for u in users:
        u.start()
    for u in users:
        u.join()
    assert not bad


@pytest.mark.parametrize("k", [1, 3])
def test_instances_of_all_sizes(k):
    """one launch for the small instances of a context, the general kernels for
    the others"""
    sizes = SIZES + [(64, 80)] * 5
    g = pra_amd.Context(k, batch_size=1)
    made = []
    for i, (values, rows) in enumerate(sizes):
        g.set_group(i)
        T, _, fix, _ = tc_program(g, layers(values, rows))
        made.append((T, fix))
    g.execute()
    for i, (values, rows) in enumerate(sizes):
        o = O.Oracle(k)
        T, _, fix, _ = tc_program(o, layers(values, rows))
        o.execute(1)
        np.testing.assert_array_equal(g.rows(made[i][0]), o.rows(T))
        assert g.history(made[i][1]) == o.history(fix)
        assert g.group_joined(i) == o.joined()
    g.close()
