"""Deviation lists by groups of lanes: fanouts just within, at and past what
a group keeps in registers (twice its lanes), lists that a wave and that a
block sorts, equal deltas (ties keep fanout order, which the costs and the
parents of a report rest on), unreachable heads under an endpoint subset.
Checked through whole queries against the oracle."""
import numpy as np
import pytest

import cpgamd
import pyoracle
from test_simt_emulator import bits_equal, emu  # noqa: F401  (fixture)


def hubs(degrees, base, width, seed):
    """Sources of the given out-degrees over `width` middle vertices, each of
    these with `base` fanouts to sinks; a third of the weights are equal."""
    rng = np.random.default_rng(seed)
    nh, ns = len(degrees), 12
    eu, ev = [], []
    for h, d in enumerate(degrees):
        eu += [h] * d
        ev += (nh + rng.choice(width, size=d, replace=False)).tolist()
    for m in range(width):
        for t in rng.choice(ns, size=base, replace=False):
            eu.append(nh + m)
            ev.append(nh + width + int(t))
    w = rng.uniform(0.05, 1.0, len(eu)).astype(np.float32)
    w[rng.random(len(w)) < 0.33] = 0.5
    return nh + width + ns, np.array(eu, np.int32), np.array(ev, np.int32), w


def check(lib, graph, k, masked):
    n, u, v, w = graph
    og = pyoracle.OracleGraph.from_edges(n, u, v, w)
    mask = None
    if masked:
        mask = np.zeros(n, np.uint8)
        mask[n - 12::2] = 1
    dist, succ, _, _ = og.sfxt(mask)
    want, _ = og.topk(dist, succ, k)
    g = lib.CpGen()
    try:
        g.load_edges(n, u, v, w)
        for _ in range(2):  # the level loop's successors, then the pass's own
            g.reset()
            g.report_paths(k, endpoint_mask=mask)
            assert bits_equal(want, g.get_slacks(k))
    finally:
        g.close()


def test_emulated_devs_lanes(emu):  # noqa: F811
    check(emu, hubs([1, 7, 8, 9, 17, 70], 1, 70, 1), 60, False)


EDGES = [1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 66, 127, 128, 129, 130, 300]


@pytest.mark.gpu
@pytest.mark.parametrize("base", [1, 2, 3, 5, 8, 11])  # 4.6 x mean steps through 4 to 64 lanes
@pytest.mark.parametrize("masked", [False, True])
def test_gpu_devs_lanes(base, masked):
    check(cpgamd, hubs(EDGES, base, 1500, base), 3000, masked)


@pytest.mark.gpu
def test_gpu_devs_lists_past_the_lds_sort():
    check(cpgamd, hubs([2047, 2049, 2050, 5000], 2, 6000, 3), 9000, False)
