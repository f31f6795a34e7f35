"""Whole iterations of a small output by one block (k_rank_loop) where it hands
over to the general iterations: candidate counts around 8,192 an iteration
(16,384 with four instances or more), deltas of more rows, rank spaces around 1,024 superblocks (2^25 bits: 5,792
values), more iterations than a launch makes (256), logs that outgrow their
room, several instances of which some stop, join thresholds.  Rows, ids
included, per-batch deltas, iterations and join pairs must equal the oracle's
and those of the general iterations alone."""
import os

import numpy as np
import pytest

import oracle as O
import pra_amd
from programs import distinct_u64, random_graph, tc_program, with_rowid

pytestmark = pytest.mark.gpu


def chains(n, extra, h, depth):
    """n sources into h chains of `depth` vertices each, and `extra` sources
    into the first chain only: about n * h + extra candidates an iteration"""
    ids = distinct_u64(n + extra + h * depth, n + extra + 7)
    c = [[ids[n + extra + i * depth + j] for j in range(depth)] for i in range(h)]
    e = [(ids[s], c[i][0]) for i in range(h) for s in range(n)] + [(ids[n + s], c[0][0]) for s in range(extra)]
    return with_rowid(e + [(c[i][j], c[i][j + 1]) for i in range(h) for j in range(depth - 1)])


def pieces(count):
    """count separate paths of three vertices"""
    ids = distinct_u64(3 * count, count)
    return with_rowid([(ids[3 * i + j], ids[3 * i + j + 1]) for i in range(count) for j in range(2)])


def path(n):
    ids = distinct_u64(n, n)
    return with_rowid([(ids[i], ids[i + 1]) for i in range(n - 1)])


CASES = [(f"chains{n}_{x}", chains(n, x, 4, 6)) for n in range(2042, 2046) for x in range(4)] + [
    (f"pieces{n}", pieces(n)) for n in (1, 1930, 1931)] + [
    (f"path{n}", path(n)) for n in (3, 257, 259, 600)] + [
    (f"random{n}", random_graph(n, int(1.3 * n), n + 1)) for n in (40, 1100, 2300)]


def gpu_context(k, batch, loop, threshold=None):
    os.environ["PRA_RANK_LOOP"] = "1" if loop else "0"
    try:
        g = pra_amd.Context(nbuckets=k, batch_size=batch)
    finally:
        del os.environ["PRA_RANK_LOOP"]
    if threshold is not None:
        g.set_join_threshold(threshold)
    return g


@pytest.mark.parametrize("k,batch", [(1, 1), (3, 10), (33, 2), (200, 1)])
@pytest.mark.parametrize("name,edges", CASES, ids=[c[0] for c in CASES])
def test_tc_equals_oracle(name, edges, k, batch):
    o = O.Oracle(k)
    To, _, fo, _ = tc_program(o, edges)
    o.execute(batch)
    for loop in (True, False):
        print(f"[rank loop] {name} k={k} batch={batch} loop={loop}", flush=True)
        g = gpu_context(k, batch, loop)
        try:
            g.set_profiling(True)
            Tg, _, fg, _ = tc_program(g, edges)
            g.execute()
            np.testing.assert_array_equal(g.rows(Tg), o.rows(To))
            assert g.history(fg) == o.history(fo)
            assert g.joined() == o.joined()
            assert g.iterations_run() == o.iterations_run()
            if not loop:
                assert g.kernel_stats()["rank_loop"]["launches"] == 0
            elif name in ("path600", "random1100") and batch == 1:
                assert g.kernel_stats()["rank_loop"]["launches"] > 0
        finally:
            g.close()


@pytest.mark.parametrize("threshold", [0, 50, 2000])
def test_thresholds(threshold):
    edges = random_graph(400, 560, 5)
    o = O.Oracle(3)
    o.set_join_threshold(threshold)
    To, _, fo, _ = tc_program(o, edges)
    o.execute(1)
    g = gpu_context(3, 1, True, threshold)
    try:
        Tg, _, fg, _ = tc_program(g, edges)
        g.execute()
        np.testing.assert_array_equal(g.rows(Tg), o.rows(To))
        assert g.history(fg) == o.history(fo)
    finally:
        g.close()


@pytest.mark.parametrize("k,batch", [(1, 3), (8, 1)])
def test_instances_beside_each_other(k, batch):
    graphs = [chains(n, x, 4, 6) for n in (4090, 4091, 4092) for x in range(4)] + [
        path(600), random_graph(900, 1170, 3), pieces(1900), random_graph(60, 80, 9), random_graph(2300, 2990, 4)]
    g = gpu_context(k, batch, True)
    try:
        made = []
        for i, e in enumerate(graphs):
            g.set_group(i)
            made.append(tc_program(g, e))
        g.execute()
        for i, e in enumerate(graphs):
            o = O.Oracle(k)
            To, _, fo, _ = tc_program(o, e)
            o.execute(batch)
            print(f"[rank loop] instance {i} k={k}", flush=True)
            np.testing.assert_array_equal(g.rows(made[i][0]), o.rows(To))
            assert g.history(made[i][2]) == o.history(fo)
            assert g.group_joined(i) == o.joined()
    finally:
        g.close()
