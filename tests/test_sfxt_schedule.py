"""The SFXT in schedule order: the second and later runs on a resident graph
settle its vertices in the level order the first run left.  Every run has
to give the oracle's dist, succ and level, with and without an endpoint
subset, as loaded and relabelled, and the query's costs bit for bit.  The
cases sit at the edges of the schedule: each choice of lanes per vertex,
rows longer than a wave's step, levels narrower and wider than a wave's
vertices, vertices on a cycle, one level, no edges, and a graph replaced by
another in the same handle."""
import numpy as np
import pytest

import cpgamd
import pyoracle
from test_simt_emulator import bits_equal, emu  # noqa: F401  (fixture)


def layered(sizes, deg, seed, hub=0):
    """Levels of the given sizes (sources first), deg random fanouts per
    vertex one to three levels ahead, one vertex of hub extra fanouts."""
    rng = np.random.default_rng(seed)
    first = np.concatenate([[0], np.cumsum(sizes)])
    n, L = int(first[-1]), len(sizes)
    eu, ev = [], []
    for lv in range(L - 1):
        for a in range(first[lv], first[lv + 1]):
            d = rng.integers(1, 2 * deg) if deg > 1 else 1
            tl = np.minimum(lv + rng.integers(1, 4, size=d), L - 1)
            heads = {int(rng.integers(first[t], first[t + 1])) for t in tl}
            heads.add(int(rng.integers(first[lv + 1], first[lv + 2])))
            eu += [a] * len(heads)
            ev += sorted(heads)
    if hub:
        heads = rng.choice(np.arange(first[1], n), size=min(hub, n - first[1]), replace=False)
        eu += [0] * len(heads)
        ev += [int(x) for x in heads]
    ids = rng.permutation(n)
    u, v = ids[np.asarray(eu, np.int64)], ids[np.asarray(ev, np.int64)]
    w = rng.uniform(0.01, 1.0, len(u)).astype(np.float32)
    w[rng.random(len(w)) < 0.3] = 0.25  # equal candidates: the successor's tie rule
    return n, u.astype(np.int32), v.astype(np.int32), w


SHAPES = {
    "sparse": lambda: layered([9, 70, 130, 64, 1, 3, 65, 20], 1, 1),
    "mean3": lambda: layered([40] * 9, 3, 2),
    "mean6": lambda: layered([33, 100, 31, 32, 17], 6, 3),
    "mean12": lambda: layered([50, 60, 70, 20], 12, 4),
    "dense_hub": lambda: layered([20, 90, 90, 40], 24, 5, hub=200),
    "sparse_hub": lambda: layered([9, 70, 130, 64, 30], 1, 8, hub=60),
    "mean3_hub": lambda: layered([40] * 9, 3, 9, hub=90),
    "mean6_hub": lambda: layered([33, 100, 31, 32, 17], 6, 10, hub=120),
    "chain": lambda: (19, np.arange(18, dtype=np.int32), np.arange(1, 19, dtype=np.int32),
                      np.linspace(0.01, 0.9, 18, dtype=np.float32)),
    "one_edge": lambda: (2, np.array([1], np.int32), np.array([0], np.int32), np.array([0.5], np.float32)),
    "cycle": lambda: with_cycle(*layered([12, 30, 30, 9], 3, 6)),
    "no_edges": lambda: (5, np.zeros(0, np.int32), np.zeros(0, np.int32), np.zeros(0, np.float32)),
}


def with_cycle(n, u, v, w):
    """Three vertices on a cycle that reaches the graph, and one alone."""
    more = np.array([[n, n + 1], [n + 1, n + 2], [n + 2, n], [n, int(v[0])]], np.int32)
    return (n + 4, np.concatenate([u, more[:, 0]]), np.concatenate([v, more[:, 1]]),
            np.concatenate([w, np.full(4, 0.1, np.float32)]))


def check_runs(lib, n, u, v, w, reorder, k):
    og = pyoracle.OracleGraph.from_edges(n, u, v, w)
    sinks = np.nonzero(np.bincount(u, minlength=n)[:n] == 0)[0]
    some = np.zeros(n, np.uint8)
    some[sinks[::2]] = 1
    g = lib.CpGen()
    try:
        g.load_edges(n, u, v, w)
        if reorder:
            g.set_csr_reorder(1)
        for mask in (None, None, some, None, some):
            dist, succ, level, levels = og.sfxt(mask)
            g.reset()
            g.report_paths(k, endpoint_mask=mask)
            gd, gs, gl = g.sfxt()
            np.testing.assert_array_equal(gd, dist)
            np.testing.assert_array_equal(gs, succ)
            np.testing.assert_array_equal(gl, level)
            assert g.graph_diameter == levels
            want, _ = og.topk(dist, succ, k)
            assert bits_equal(want, g.get_slacks(k))
    finally:
        g.close()


@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_emulated_schedule_equals_oracle(emu, shape, reorder):  # noqa: F811
    check_runs(emu, *SHAPES[shape](), reorder, 0)


def test_emulated_schedule_follows_the_loaded_graph(emu):  # noqa: F811
    g = emu.CpGen()
    try:
        for shape in ("mean6", "chain", "mean3"):
            n, u, v, w = SHAPES[shape]()
            og = pyoracle.OracleGraph.from_edges(n, u, v, w)
            dist, succ, level, _ = og.sfxt()
            g.load_edges(n, u, v, w)
            for method in (0, 0, 2, 0, 3, 0):  # loops that leave no level order between
                g.reset()
                g.report_paths(0, sfxt_method=method)
                for got, want in zip(g.sfxt(), (dist, succ, level)):
                    np.testing.assert_array_equal(got, want)
    finally:
        g.close()


@pytest.mark.parametrize("nth", range(8))
def test_emulated_full_device_leaves_the_schedule_out(emu, nth):  # noqa: F811
    """One device allocation fails on the run that lays the schedule out, its
    own or a later one of the query (which grows its node store): the query
    is answered as without a schedule."""
    n, u, v, w = SHAPES["mean3"]()
    og = pyoracle.OracleGraph.from_edges(n, u, v, w)
    dist, succ, level, _ = og.sfxt()
    g = emu.CpGen()
    try:
        g.load_edges(n, u, v, w)
        g.report_paths(1)
        for k in (2000, 2000):
            g.reset()
            emu._lib.simt_fail_malloc(nth)
            try:
                g.report_paths(k)
            finally:
                emu._lib.simt_fail_malloc(-1)
            for got, want in zip(g.sfxt(), (dist, succ, level)):
                np.testing.assert_array_equal(got, want)
            want, _ = og.topk(dist, succ, k)
            assert bits_equal(want, g.get_slacks(k))
    finally:
        g.close()


@pytest.mark.parametrize("nth", range(10))
def test_emulated_full_device_in_discovery(emu, nth):  # noqa: F811
    """An allocation of a deviation discovery fails on a handle that holds a
    schedule: the schedule is given back and the call answered."""
    n, u, v, w = SHAPES["mean3"]()
    front = [np.arange(i, n, 7, dtype=np.int32) for i in range(3)]
    with emu.CpGen() as g:
        g.load_edges(n, u, v, w)
        want = g.bvss_discover(front)
    with emu.CpGen() as g:
        g.load_edges(n, u, v, w)
        for _ in range(2):
            g.reset()
            g.run_sfxt()
        emu._lib.simt_fail_malloc(nth)
        try:
            got = g.bvss_discover(front)
        finally:
            emu._lib.simt_fail_malloc(-1)
    for a, b in zip(want, got):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("nth", range(6))
def test_emulated_full_device_in_a_batch(emu, nth):  # noqa: F811
    """An allocation fails on the batch's run that holds a schedule of the
    union graph (larger rounds store more paths than the first run's, so its
    buffers grow)."""
    graphs = [SHAPES["mean12"](), SHAPES["mean3"]()]
    k = 3000
    with emu.Batch() as b:
        for g in graphs:
            b.add(*g, k)
        b.set_tuning(target_div=(32, 32, 32))
        b.run()
        want = [b.get_slacks(q, k).copy() for q in range(2)]
        stored = b.timings()["generated"]
        b.set_tuning(target_div=(1, 1, 1))
        emu._lib.simt_fail_malloc(nth)
        try:
            b.run()
        finally:
            emu._lib.simt_fail_malloc(-1)
        assert b.timings()["generated"] > stored
        for q in range(2):
            assert bits_equal(want[q], b.get_slacks(q, k))


@pytest.mark.parametrize("nth", range(0, 102, 6))
def test_emulated_full_device_in_a_server(emu, nth):  # noqa: F811
    """An allocation fails while a server with two resident graphs adds the
    second, starts or serves its queries (six numbers apart: a first query's
    buffers are reserved in groups): every query is answered."""
    graphs = [SHAPES["mean3"](), SHAPES["mean6"]()]
    jobs = []
    with emu.Server(max_in_flight=4, initial_nodes=4000) as s:
        s.add_graph(*graphs[0])
        emu._lib.simt_fail_malloc(nth)
        try:
            s.add_graph(*graphs[1])
            for i in range(3):
                jobs.append((i % 2, s.submit(i % 2, 4 + i)))
            while s.step() > 0:
                pass
        finally:
            emu._lib.simt_fail_malloc(-1)
        for gi, q in jobs:
            og = pyoracle.OracleGraph.from_edges(*graphs[gi])
            dist, succ, _, _ = og.sfxt()
            assert bits_equal(og.topk(dist, succ, 3 + q)[0], s.get_slacks(q, 3 + q))


def test_emulated_layout_is_not_tried_again(emu):  # noqa: F811
    """A device with no room for the schedule: the level loop stays until the
    graph is loaded again, without another attempt at each query."""
    def held(g):
        g.reset()
        g.report_paths(5, max_nodes=4000)
        return g.timings()["device_bytes"]

    n, u, v, w = SHAPES["mean3"]()
    with emu.CpGen() as g:
        g.load_edges(n, u, v, w)
        without = held(g)
        emu._lib.simt_fail_malloc(0)
        try:
            assert held(g) == without
        finally:
            emu._lib.simt_fail_malloc(-1)
        assert held(g) == without
        g.load_edges(n, u, v, w)
        assert held(g) == without
        assert held(g) > without


def budget_after(lib, n, u, v, w, change):
    """The graph of a handle that holds a schedule is loaded again, or
    relabelled: a budget of what a new handle holds for it is still enough,
    with as many node slots."""
    def load(g):
        g.load_edges(n, u, v, w)

    def forest(g):
        g.reset()
        g.run_sfxt()

    def ask(g, budget):
        g.reset()
        g.report_paths(20, mem_budget_bytes=budget, max_nodes=20000)
        return g.get_slacks(20).copy(), g.timings()

    steps = {"load": load, "reorder": lambda g: g.set_csr_reorder(1)}
    with lib.CpGen() as g:
        load(g)
        forest(g)
        steps[change](g)
        forest(g)
        want, ref = ask(g, 1 << 40)  # a budget: no schedule is held
    held = ref["device_bytes"]
    with lib.CpGen() as g:
        load(g)
        forest(g)
        forest(g)
        steps[change](g)
        forest(g)
        got, t = ask(g, held)
    assert bits_equal(want, got)
    assert t["device_bytes"] <= held and t["node_slots"] == ref["node_slots"]


@pytest.mark.parametrize("change", ["load", "reorder"])
def test_emulated_schedule_ends_with_its_graph(emu, change):  # noqa: F811
    budget_after(emu, *SHAPES["mean6"](), change)


@pytest.mark.gpu
@pytest.mark.parametrize("change", ["load", "reorder"])
def test_gpu_schedule_ends_with_its_graph(change):
    budget_after(cpgamd, *layered([300] * 150, 4, 8), change)


@pytest.mark.gpu
@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_gpu_schedule_equals_oracle(shape, reorder):
    check_runs(cpgamd, *SHAPES[shape](), reorder, 40)


@pytest.mark.gpu
def test_gpu_schedule_deep_and_wide():
    n, u, v, w = layered([300] * 150, 4, 7)
    check_runs(cpgamd, n, u, v, w, False, 500)


@pytest.mark.gpu
def test_gpu_budget_leaves_the_schedule_out():
    """A budget of what the first query held is enough for every later one."""
    n, u, v, w = layered([300] * 150, 4, 8)
    g = cpgamd.CpGen()
    try:
        g.load_edges(n, u, v, w)
        g.report_paths(100)
        want, held = g.get_slacks(100), g.timings()["device_bytes"]
        for budget in (0, held, 0, held):
            g.reset()
            g.report_paths(100, mem_budget_bytes=budget)
            assert bits_equal(want, g.get_slacks(100))
            assert not budget or g.timings()["device_bytes"] <= budget
    finally:
        g.close()
