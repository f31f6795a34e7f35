"""The bucket partition around its sub-tiles (512 or 256 rows through LDS) and
tiles (2,048 rows), for every row width class, with few and many buckets; the
allocation-free form alike."""
import numpy as np
import pytest

from partition_expect import partition_expect
from test_gpu_partition import run_partition

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 511, 512, 513, 2047, 2049, 5000])
@pytest.mark.parametrize("w,jcc,k", [(1, 1, 2), (2, 1, 200), (3, 1, 3), (4, 2, 8), (5, 3, 64), (6, 1, 64), (8, 2, 13), (9, 2, 7), (32, 4, 256)])
def test_widths(w, jcc, k, n):
    import pra_amd
    print("case", n, w, jcc, k, flush=True)
    rows = np.random.default_rng(n + w).integers(0, 50, size=(n, w), dtype=np.uint64)
    want, wbnd = partition_expect(rows, jcc, k)
    ctx = pra_amd.Context(nbuckets=k)
    try:
        for noalloc in (False, True):
            got, bnd = run_partition(ctx, rows, w, jcc, noalloc=noalloc)
            np.testing.assert_array_equal(bnd, wbnd)
            np.testing.assert_array_equal(got, want)
    finally:
        ctx.close()
