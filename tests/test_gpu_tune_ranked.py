"""The choice between the claim table and ranked membership settles: the
samples of both are kept, also where an iteration's summary arrives before its
last launch has ended."""
import numpy as np
import pytest

from programs import grid_graph, grid_tc_size, tc_program

pytestmark = pytest.mark.gpu


def test_ranked_membership_settles():
    import pra_amd
    n = 100
    rows = []
    for k in range(2):
        print(f"[tune ranked] grid {n}, solve {k}", flush=True)
        c = pra_amd.Context(nbuckets=8, batch_size=1)
        try:
            T = tc_program(c, grid_graph(n, seed=n))[0]
            c.execute()
            rows.append(c.rows(T))
        finally:
            c.close()
    assert rows[0].shape[0] == grid_tc_size(n)
    np.testing.assert_array_equal(rows[0], rows[1])
    # its iterations have capacities of 2^16 to 2^19 candidates, dozens of each
    bands = {band: (choice, means) for _, knob, band, choice, means in pra_amd.autotune_report()
             if knob == "ranked_membership"}
    for band in (16, 17, 18):
        choice, means = bands[band]
        assert choice == int(means[1] <= means[0]) and len(means) == 2, bands
