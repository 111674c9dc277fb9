"""Chain walks by groups of lanes: two per parent on sparse graphs, four
elsewhere.  Vertices with no, one, a few, exactly a group's and many
deviations, bounds that cut a list at its start, inside a group and at its
end, equal deltas, and a chain longer than any row; every K prefix and both
walk passes (with and without a bound probe) against the oracle."""
import numpy as np
import pytest

import cpgamd
import pyoracle
from test_sfxt_schedule import layered
from test_simt_emulator import bits_equal, emu  # noqa: F401  (fixture)


def rows(fan, levels, width, seed, ties):
    """Every vertex of a level has `fan` fanouts in the next."""
    rng = np.random.default_rng(seed)
    eu, ev = [], []
    for lv in range(levels - 1):
        for a in range(width):
            for b in rng.choice(width, size=min(fan, width), replace=False):
                eu.append(lv * width + a)
                ev.append((lv + 1) * width + int(b))
    w = rng.uniform(0.05, 1.0, len(eu)).astype(np.float32)
    if ties:
        w = (np.round(w * 4) / 4 + 0.25).astype(np.float32)
    return levels * width, np.array(eu, np.int32), np.array(ev, np.int32), w


def check(lib, graph, ks, probes):
    og = pyoracle.OracleGraph.from_edges(*graph)
    dist, succ, _, _ = og.sfxt()
    g = lib.CpGen()
    try:
        g.load_edges(*graph)
        for k in ks:
            want, _ = og.topk(dist, succ, k)
            for probe in probes:
                g.reset()
                g.report_paths(k, bound_probe=probe)
                assert bits_equal(want, g.get_slacks(k)), (k, probe)
    finally:
        g.close()


def test_emulated_walk_lanes(emu):  # noqa: F811
    check(emu, rows(5, 6, 9, 1, False), [60], [1])
    check(emu, rows(2, 7, 6, 2, True), [25], [-1])


@pytest.mark.gpu
@pytest.mark.parametrize("fan", [1, 2, 3, 4, 5, 8, 9, 33])
@pytest.mark.parametrize("ties", [False, True])
def test_gpu_walk_lanes(fan, ties):
    check(cpgamd, rows(fan, 9, 40, fan, ties), [1, 3, 64, 1000, 20000], [1, -1])


@pytest.mark.gpu
def test_gpu_walk_long_chains():
    check(cpgamd, layered([25] * 400, 2, 3), [10, 5000], [1, -1])
