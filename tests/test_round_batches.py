"""Round batches that grow from a small first one, and bound trials that step
back from a full node store: graphs whose cheapest paths have very many
children (long fan-outs on deep chains), equal costs everywhere (no bound
lies between too few paths and too many), stores too small for a trial;
K around one whole batch (131,072).  Each against the oracle."""
import numpy as np
import pytest

import cpgamd
import pyoracle
from test_sfxt_schedule import layered
from test_simt_emulator import bits_equal, emu  # noqa: F401  (fixture)
from test_walk_lanes import rows


def check(lib, graph, ks, **opts):
    og = pyoracle.OracleGraph.from_edges(*graph)
    dist, succ, _, _ = og.sfxt()
    g = lib.CpGen()
    try:
        g.load_edges(*graph)
        for k in ks:
            want, _ = og.topk(dist, succ, k)
            g.reset()
            g.report_paths(k, **opts)
            assert bits_equal(want, g.get_slacks(k)), k
        return g.timings()
    finally:
        g.close()


def test_emulated_probe_steps_back(emu):  # noqa: F811
    check(emu, rows(6, 6, 12, 5, True), [40], bound_probe=1, max_nodes=400)


@pytest.mark.gpu
@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("fan,levels,width", [(20, 60, 40), (3, 200, 30), (33, 12, 64)])
def test_gpu_round_batches(fan, levels, width, ties):
    graph = rows(fan, levels, width, fan + levels, ties)
    for probe in (1, -1):
        check(cpgamd, graph, [1, 30000, 131072, 131073, 200000], bound_probe=probe)
    check(cpgamd, graph, [5000], batch=77)


@pytest.mark.gpu
@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("nodes", [3000, 20000, 200000])
def test_gpu_probe_in_a_small_store(nodes, ties):
    check(cpgamd, rows(12, 40, 60, 9, ties), [2000], bound_probe=1, max_nodes=nodes)


@pytest.mark.gpu
@pytest.mark.parametrize("probe", [1, -1])
def test_gpu_histogram_parts(probe):
    """Stores of one histogram block (8,192 paths) and just past it, of a few,
    and of more than there are partials for."""
    check(cpgamd, rows(6, 30, 300, 11, False), [2, 2000, 4000, 8000, 16000, 33000, 700000], bound_probe=probe)


@pytest.mark.gpu
def test_gpu_shallow_graph_takes_whole_batches():
    """Few children per parent: a round per level of the prefix tree, none of
    them small."""
    graph = layered([4000, 3000, 3000, 2000], 5, 90)
    assert check(cpgamd, graph, [131073, 200000, 300000])["rounds"] <= 4
