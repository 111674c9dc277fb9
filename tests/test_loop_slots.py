"""Level and scheduled loops in flight together share the device's block slots:
a loop beside others takes at most half of what they leave, one block where
they leave nothing, and all it asks for once they have ended.  The grid does
not change dist, succ, level or the costs."""
import ctypes
import threading

import numpy as np
import pytest

import cpgamd
import pyoracle
from test_sfxt_schedule import SHAPES, layered
from test_simt_emulator import bits_equal, emu  # noqa: F401  (fixture)
from test_zz_noalloc_widths import HostMemory
from test_zz_no_alloc import run_noalloc


@pytest.fixture
def slots(emu):  # noqa: F811
    hold = emu.lib().cpg_test_hold_slots
    hold.argtypes = [ctypes.c_int]
    yield hold
    hold(0)


def forest(g, method=0):
    g.reset()
    g.report_paths(0, sfxt_method=method)
    return g.timings()["sfxt_blocks"], [x.copy() for x in g.sfxt()]


@pytest.mark.parametrize("shape", ["mean3", "dense_hub"])
def test_emulated_loops_share_the_slots(emu, slots, shape):  # noqa: F811
    n, u, v, w = SHAPES[shape]()
    want = pyoracle.OracleGraph.from_edges(n, u, v, w).sfxt()[:3]
    with emu.CpGen() as g:
        g.load_edges(n, u, v, w)
        for method in (0, 0, 1, 3, 4, 5):  # level loop, scheduled loop, ...
            alone = forest(g, method)[0]
            seen = []
            for held in (8, 16, 1000000):
                slots(held)
                blocks, got = forest(g, method)
                slots(0)
                seen.append(blocks)
                for a, b in zip(want, got):
                    np.testing.assert_array_equal(a, b)
            assert alone >= seen[0] >= seen[1] >= seen[2] == 1, (method, alone, seen)
            assert forest(g, method)[0] == alone
            assert alone > 1 or method == 5  # few blocks fit one XCD of the emulated device


def test_emulated_noalloc_beside_other_loops(emu, slots):  # noqa: F811
    n, u, v, w = SHAPES["mean6"]()
    want = pyoracle.OracleGraph.from_edges(n, u, v, w).sfxt()
    mem = HostMemory()
    for held in (0, 16, 1000000):
        slots(held)
        levels, got = run_noalloc(mem, emu.lib(), n, u, v, w)
        assert levels == want[3]
        for a, b in zip(want, got):
            np.testing.assert_array_equal(a, b)


def test_emulated_server_beside_other_loops(emu, slots):  # noqa: F811
    names = ("mean3", "cycle", "mean6")
    for held in (0, 16, 1000000):
        slots(held)
        with emu.Server(initial_nodes=4000) as s:
            qs = [(name, s.submit(s.add_graph(*SHAPES[name]()), 5)) for name in names]
            while s.step() > 0:
                pass
            for name, q in qs:
                og = pyoracle.OracleGraph.from_edges(*SHAPES[name]())
                dist, succ, _, _ = og.sfxt()
                assert bits_equal(og.topk(dist, succ, 5)[0], s.get_slacks(q, 5))


@pytest.mark.gpu
def test_gpu_handles_on_threads():
    """Twelve handles on threads of their own, each with a graph wide enough
    for the largest grid."""
    n, u, v, w = layered([4000] * 12, 3, 80)
    want = pyoracle.OracleGraph.from_edges(n, u, v, w).sfxt()[:3]
    wrong = []

    def work(i):
        try:
            with cpgamd.CpGen() as g:
                g.load_edges(n, u, v, w)
                for _ in range(6):
                    for a, b in zip(want, forest(g)[1]):
                        np.testing.assert_array_equal(a, b)
        except Exception as e:
            wrong.append((i, e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(12)]
    print("case handles on threads", flush=True)
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
