"""Ranked membership (new keys placed by their bitmap's prefix counts) where
its parts change over: candidate counts around one tile, rank spaces around one
and several superblocks (32,768 bits) and scan chunks, bucket counts on both
sides of the wave look-back, duplicates from several predecessors.  Rows, ids
included, per-batch deltas and join pairs must equal the oracle's."""
import numpy as np
import pytest

import oracle as O
import pra_amd
from programs import distinct_u64, random_graph, tc_program, with_rowid

pytestmark = pytest.mark.gpu


def hubs(n, nhub):
    """n sources into each of nhub hubs, every hub into one sink: n * nhub
    candidates for n keys in one iteration"""
    ids = distinct_u64(n + nhub + 1, n + nhub)
    e = [(ids[i], ids[n + h]) for h in range(nhub) for i in range(n)]
    return with_rowid(e + [(ids[n + h], ids[n + nhub]) for h in range(nhub)])


CASES = [(f"hub{n}_{h}", hubs(n, h)) for n, h in ((2047, 1), (2048, 1), (2049, 1), (683, 3), (1025, 4))] + [
    (f"random{n}", random_graph(n, int(1.3 * n), n)) for n in (181, 182, 256, 724, 725, 1100)]


@pytest.mark.parametrize("k", [1, 3, 33, 200])
@pytest.mark.parametrize("name,edges", CASES, ids=[c[0] for c in CASES])
def test_tc_equals_oracle(name, edges, k):
    print(f"[ranked] {name} k={k}", flush=True)
    g, o = pra_amd.Context(k, batch_size=1), O.Oracle(k)
    try:
        Tg, _, fg, _ = tc_program(g, edges)
        To, _, fo, _ = tc_program(o, edges)
        g.execute()
        o.execute(1)
        np.testing.assert_array_equal(g.rows(Tg), o.rows(To))
        assert g.history(fg) == o.history(fo)
        assert g.joined() == o.joined()
    finally:
        g.close()
