"""A fixpoint SCC without rules: its delta moves into full in its first
iteration and its first batch ends it, alone and beside instances with rules.
Rows, per-batch deltas and iterations must equal the oracle's."""
import numpy as np
import pytest

import oracle as O
from programs import FULL, small_random_graph, tc_program

pytestmark = pytest.mark.gpu


def no_rules(b, edges, move):
    R = b.rel_create(2, 1, 300)
    b.load_rows(R, edges, FULL)
    s = b.scc_create(True, 1)
    b.scc_add_relation(s, R, move)
    return R, s


@pytest.mark.parametrize("move", [True, False])
@pytest.mark.parametrize("batch", [1, 2, 10])
def test_alone(batch, move):
    import pra_amd
    edges = small_random_graph(7)
    o = O.Oracle(3)
    Ro, so = no_rules(o, edges, move)
    o.execute(batch)
    g = pra_amd.Context(nbuckets=3, batch_size=batch)
    try:
        Rg, sg = no_rules(g, edges, move)
        print(f"[no rules] batch={batch} move={move}", flush=True)
        g.execute()
        np.testing.assert_array_equal(g.rows(Rg), o.rows(Ro))
        assert g.history(sg) == o.history(so)
        assert g.iterations_run() == o.iterations_run()
    finally:
        g.close()


@pytest.mark.parametrize("step", [False, True])
def test_beside_instances_with_rules(step):
    import pra_amd
    graphs = [small_random_graph(i, 30 + i, 45) for i in range(4)]
    g = pra_amd.Context(nbuckets=3, batch_size=10)
    try:
        made = []
        for i, e in enumerate(graphs):
            g.set_group(i)
            made.append((no_rules(g, e, True) if i % 2 else tc_program(g, e)[::2]))
        print(f"[no rules] beside others, step={step}", flush=True)
        if step:
            while g.step():
                pass
        else:
            g.execute()
        for i, e in enumerate(graphs):
            o = O.Oracle(3)
            Ro, so = no_rules(o, e, True) if i % 2 else tc_program(o, e)[::2]
            o.execute(10)
            np.testing.assert_array_equal(g.rows(made[i][0]), o.rows(Ro))
            assert g.history(made[i][1]) == o.history(so)
    finally:
        g.close()
