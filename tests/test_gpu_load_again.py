"""Several loads into one relation: rows equal to loaded ones are dropped
whichever sort puts them in order, and a load that sees no equal rows keeps all
of them."""
import numpy as np
import pytest

import oracle as O
import pra_amd
from programs import FULL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 3])
@pytest.mark.parametrize("span", [3, 1 << 20, 1 << 63])
@pytest.mark.parametrize("n", [1, 2, 512, 513, 2049, 20000, 300000])
def test_loads_into_one_relation(n, span, k):
    rng = np.random.default_rng([n, span % 1000, k])
    rows = np.column_stack([rng.integers(0, span, size=(n, 2), dtype=np.uint64), rng.integers(0, 4, size=n, dtype=np.uint64)])
    fresh = np.column_stack([rows[:, :2], rows[:, 2] + np.uint64(7)])
    g, o = pra_amd.Context(nbuckets=k, batch_size=1), O.Oracle(k)
    try:
        Rg, Ro = g.rel_create(2, 1, 300), o.rel_create(2, 1, 300)
        print(f"[load again] n={n} span={span} k={k}", flush=True)
        for part in (rows, rows[::2], fresh, np.concatenate([fresh[: n // 2 + 1], rows[:1]])):
            for b, R in ((g, Rg), (o, Ro)):
                b.load_rows(R, part, FULL)
            np.testing.assert_array_equal(g.rows(Rg), o.rows(Ro))
    finally:
        g.close()
