"""Relation loads through the sorts of rows by (bucket, columns): one block up
to 2,048 rows, then keyed counting passes and LDS segments, then (segments too
large for a block) byte passes.  Sizes around the changes of path and of block,
keys of one word and of several, rows that share their leading word, skewed
and constant columns, duplicates.  The loaded rows must equal numpy's sort by
(bucket, columns)."""
import numpy as np
import pytest

import pra_amd
from partition_expect import partition_expect
from programs import FULL

pytestmark = pytest.mark.gpu


def rows_of(kind, n, w, rng):
    if kind == "wide":            # random 64-bit columns: keys of several words, mostly told apart by the first
        a = rng.integers(0, 2**64 - 1, size=(n, w), dtype=np.uint64, endpoint=True)
    elif kind == "shared":        # few leading values: rows of a segment share their first word
        a = rng.integers(0, 2**64 - 1, size=(n, w), dtype=np.uint64, endpoint=True)
        a[:, 0] = a[rng.integers(0, max(1, n // 40), size=n), 0]
    elif kind == "narrow":        # the whole key in one word, duplicates among the rows
        a = rng.integers(0, 7, size=(n, w), dtype=np.uint64)
        a[:, 0] = rng.integers(0, max(2, n // 2), size=n)
    elif kind == "hub":           # one leading value: a single segment, too large for a block beyond 8,192 rows
        a = rng.integers(0, 2**64 - 1, size=(n, w), dtype=np.uint64, endpoint=True)
        a[:, 0] = 5
    else:                         # constant but for one bit of the last column
        a = np.full((n, w), 3, dtype=np.uint64)
        a[:, w - 1] ^= rng.integers(0, 2, size=n, dtype=np.uint64) << np.uint64(40)
    return a


@pytest.mark.parametrize("k", [1, 5])
@pytest.mark.parametrize("n", [1, 2, 63, 1025, 2047, 2048, 2049, 4100, 20000, 262144, 262145, 400000])
@pytest.mark.parametrize("kind,w,jcc", [("wide", 4, 2), ("shared", 3, 1), ("narrow", 3, 1), ("hub", 3, 1),
                                        ("constant", 3, 2)])
def test_loaded_rows(kind, w, jcc, n, k):
    print(f"[keyed sort] {kind} n={n} k={k}", flush=True)
    a = rows_of(kind, n, w, np.random.default_rng(n + w))
    want = np.unique(a, axis=0)
    want = partition_expect(want, jcc, k)[0] if k > 1 else want
    c = pra_amd.Context(k)
    try:
        r = c.rel_create(w - 1, jcc, 1)
        c.load_rows(r, a, FULL)
        np.testing.assert_array_equal(c.rows(r), want)
    finally:
        c.close()
