"""pra_ctx_step makes one iteration of every instance in progress, also the
empty ones that end a batch: as many steps as the oracle makes iterations."""
import numpy as np
import pytest

import oracle as O
from programs import small_random_graph, tc_program

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 3, 10])
def test_a_step_is_an_iteration(batch):
    import pra_amd
    edges = small_random_graph(3)
    o = O.Oracle(3)
    To, _, fo, _ = tc_program(o, edges)
    o.execute(batch)
    g = pra_amd.Context(nbuckets=3, batch_size=batch)
    try:
        Tg, _, fg, _ = tc_program(g, edges)
        print(f"[steps] batch={batch}", flush=True)
        made = []
        while True:
            left = g.step()
            made.append(g.iterations_run())
            if not left:
                break
        assert made == list(range(1, o.iterations_run() + 1))
        np.testing.assert_array_equal(g.rows(Tg), o.rows(To))
        assert g.history(fg) == o.history(fo)
    finally:
        g.close()
