"""Served groups in schedule order: one to sixteen endpoint subsets of a graph
settled together (padded to a power of two), on graphs whose rows are
shorter and longer than a group's step, whose levels are narrower and wider
than a wave's vertices, and with vertices on a cycle; several graphs in one
launch.  Each query's costs equal the masked oracle's."""
import numpy as np
import pytest

import cpgamd
import pyoracle
from test_sfxt_schedule import SHAPES
from test_simt_emulator import bits_equal, emu  # noqa: F401  (fixture)


def with_lowest():
    """One source whose only path sums to the lowest 32-bit distance."""
    n, u, v, w = SHAPES["mean3"]()
    sink = np.setdiff1d(v, u)[0]
    return (n + 1, np.append(u, n).astype(np.int32), np.append(v, sink).astype(np.int32),
            np.append(w, np.float32(-214748.3648)))


def check(lib, shapes, queries, ks):
    rng = np.random.default_rng(queries)
    s = lib.Server(max_in_flight=64)
    try:
        jobs = []
        for name in shapes:
            n, u, v, w = SHAPES[name]()
            gid = s.add_graph(n, u, v, w)
            og = pyoracle.OracleGraph.from_edges(n, u, v, w)
            sinks = np.nonzero(np.bincount(u, minlength=n)[:n] == 0)[0]
            for i in range(queries):
                mask = None
                if i:
                    mask = np.zeros(n, np.uint8)
                    mask[rng.choice(sinks, max(1, len(sinks) // (1 + i % 4)), replace=False)] = 1
                k = ks[i % len(ks)]
                dist, succ, _, _ = og.sfxt(mask)
                jobs.append((s.submit(gid, k, mask), k, og.topk(dist, succ, k)[0]))
        while s.step() > 0:
            pass
        for q, k, want in jobs:
            assert bits_equal(want, s.get_slacks(q, k))
    finally:
        s.close()


def test_emulated_served_groups(emu):  # noqa: F811
    check(emu, ["mean3", "cycle"], 3, [5])


def test_emulated_lowest_distance_is_served(emu, monkeypatch):  # noqa: F811
    monkeypatch.setitem(SHAPES, "lowest", with_lowest)
    dist = pyoracle.OracleGraph.from_edges(*with_lowest()).sfxt()[0]
    assert dist[-1] == -2**31
    check(emu, ["lowest", "chain"], 3, [5, 40])


@pytest.mark.gpu
def test_gpu_lowest_distance_is_served(monkeypatch):
    monkeypatch.setitem(SHAPES, "lowest", with_lowest)
    check(cpgamd, ["lowest", "chain"], 3, [5, 40])


@pytest.mark.gpu
@pytest.mark.parametrize("queries", [1, 2, 3, 5, 16, 17])
@pytest.mark.parametrize("shapes", [["sparse", "chain", "cycle"], ["mean6", "mean12", "dense_hub", "mean3"]])
def test_gpu_served_groups(shapes, queries):
    check(cpgamd, shapes, queries, [1, 9, 200])
