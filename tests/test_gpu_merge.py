"""Full versions kept sorted by merges, several relations an iteration: doubling
transitive closure on chains and rings around the searches' four-row and the
merge's block steps.  Rows, ids included, must equal the oracle's."""
import numpy as np
import pytest

import oracle as O
import pra_amd
from programs import distinct_u64, nonlinear_tc_program, with_rowid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 5])
@pytest.mark.parametrize("ring", [False, True])
@pytest.mark.parametrize("n", [2, 4, 5, 17, 24, 65])
def test_doubling_closure(n, ring, k):
    print(f"[merge] n={n} ring={ring} k={k}", flush=True)
    ids = distinct_u64(n + 1, n)
    e = with_rowid([(ids[i], ids[(i + 1) % n if ring else i + 1]) for i in range(n)])
    g, o = pra_amd.Context(k, batch_size=1), O.Oracle(k)
    try:
        rg, ro = nonlinear_tc_program(g, e), nonlinear_tc_program(o, e)
        g.execute()
        o.execute(1)
        for a, b in zip(rg[:2], ro[:2]):
            np.testing.assert_array_equal(g.rows(a), o.rows(b))
        assert g.history(rg[2]) == o.history(ro[2])
    finally:
        g.close()
