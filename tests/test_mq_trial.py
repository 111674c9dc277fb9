"""First bounds of multi-query rounds: every query of a batch or a served
stream begins with a trial bound over its roots that is widened until K
paths lie under it, or goes unbounded when there are fewer.  K from one to
more than there are paths, K on either side of the root count, no reachable
root, equal costs everywhere, more paths than one LDS stage, and more
queries than the key pass counts in LDS; each result against the oracle
alone."""
import numpy as np
import pytest

import cpgamd
import pyoracle
from test_sfxt_schedule import layered
from test_simt_emulator import bits_equal, emu  # noqa: F401  (fixture)


def designs(big):
    out = []
    for i, (sizes, deg) in enumerate([((6, 9, 9, 4), 2), ((3, 20, 20, 5), 3), ((30, 12, 12, 12), 2)]):
        if big:
            sizes = tuple(7 * s for s in sizes)
        out.append(layered(sizes, deg, 40 + i))
    n, u, v, w = layered((8, 10, 10, 6), 2, 50)
    out.append((n, u, v, np.ones_like(w)))  # unit delays: ties
    out.append((2, np.array([0], np.int32), np.array([1], np.int32), np.array([0.25], np.float32)))
    return out


def want_costs(design, k, mask=None):
    og = pyoracle.OracleGraph.from_edges(*design)
    dist, succ, _, _ = og.sfxt(mask)
    return og.topk(dist, succ, k)[0]


def check_batch(lib, ks, big=False):
    ds = designs(big)
    b = lib.Batch()
    try:
        jobs = [(d, k) for k in ks for d in ds]
        for d, k in jobs:
            b.add(*d, k)
        for _ in range(2):  # the second run replays captured rounds and the schedule
            b.run()
            for q, (d, k) in enumerate(jobs):
                assert bits_equal(want_costs(d, k), b.get_slacks(q, k)), (q, k)
    finally:
        b.close()


def check_server(lib, ks, big=False):
    ds = designs(big)
    s = lib.Server()
    try:
        jobs = []
        for d in ds:
            gid = s.add_graph(*d)
            sinks = np.nonzero(np.bincount(d[1], minlength=d[0])[:d[0]] == 0)[0]
            for j, k in enumerate(ks):
                mask = None
                if j % 2:
                    mask = np.zeros(d[0], np.uint8)
                    mask[sinks[::3]] = 1
                jobs.append((d, k, mask, s.submit(gid, k, mask)))
        while s.step() > 0:
            pass
        for d, k, mask, q in jobs:
            assert bits_equal(want_costs(d, k, mask), s.get_slacks(q, k)), (k, mask is None)
    finally:
        s.close()


def tiny():
    """Fewer paths than any K asked of it; root walks of a few dozen edges."""
    return layered((2, 4, 4, 4, 4, 2), 2, 60)


def check_tiny_rounds(lib):
    """A query with few paths takes a round per prefix-tree level, not one per
    trial bound on top."""
    levels = 6
    with lib.Server() as s:
        gid = s.add_graph(*tiny())
        q = s.submit(gid, 1000)
        while s.step() > 0:
            pass
        assert bits_equal(want_costs(tiny(), 1000), s.get_slacks(q, 1000))
        assert s.stats()["rounds"] <= levels + 1
    with lib.Batch() as b:
        b.add(*tiny(), 1000)
        b.set_tuning(group=1)
        b.run()
        assert bits_equal(want_costs(tiny(), 1000), b.get_slacks(0, 1000))
        assert b.timings()["rounds"] <= levels + 1


def wide(roots):
    """Root walks of more than 65,536 edges, or of somewhat fewer (but many
    for one path)."""
    return layered((roots, 15, 15, 9), 9, 61)


def check_wide(lib, ks):
    for roots in (1000, 3000):
        d = wide(roots)
        edges = roots * 5 * len(d[1]) / d[0]
        assert (edges > 65536) == (roots == 3000)
        with lib.Batch() as b:
            for k in ks:
                b.add(*d, k)
            b.run()
            for q, k in enumerate(ks):
                assert bits_equal(want_costs(d, k), b.get_slacks(q, k)), (roots, k)
        with lib.Server() as s:
            gid = s.add_graph(*d)
            qs = [s.submit(gid, k) for k in ks]
            while s.step() > 0:
                pass
            for q, k in zip(qs, ks):
                assert bits_equal(want_costs(d, k), s.get_slacks(q, k)), (roots, k)


def test_emulated_tiny_queries_take_no_trials(emu):  # noqa: F811
    check_tiny_rounds(emu)


def test_emulated_bounds_on_either_side_of_the_line(emu):  # noqa: F811
    check_wide(emu, [1, 5000])


@pytest.mark.gpu
def test_gpu_tiny_queries_take_no_trials():
    check_tiny_rounds(cpgamd)


@pytest.mark.gpu
def test_gpu_bounds_on_either_side_of_the_line():
    check_wide(cpgamd, [1, 7, 300, 5000, 30000, 1000000])


def test_emulated_batch_first_bounds(emu):  # noqa: F811
    check_batch(emu, [1, 7, 300])


def test_emulated_server_first_bounds(emu):  # noqa: F811
    check_server(emu, [1, 40])


@pytest.mark.gpu
@pytest.mark.parametrize("big", [False, True])
def test_gpu_batch_first_bounds(big):
    check_batch(cpgamd, [0, 1, 2, 7, 30, 300, 5000, 100000], big)


@pytest.mark.gpu
@pytest.mark.parametrize("big", [False, True])
def test_gpu_server_first_bounds(big):
    check_server(cpgamd, [0, 1, 2, 7, 30, 300, 5000, 100000], big)


@pytest.mark.gpu
def test_gpu_batch_of_many_queries():
    """More queries than the key pass counts in LDS (1024)."""
    design = (3, np.array([0, 0], np.int32), np.array([1, 2], np.int32), np.array([0.5, 0.25], np.float32))
    b = cpgamd.Batch()
    try:
        for i in range(1030):
            b.add(*design, 1 + i % 3)
        b.run()
        for i in range(1030):
            assert bits_equal(want_costs(design, 1 + i % 3), b.get_slacks(i, 1 + i % 3))
    finally:
        b.close()
