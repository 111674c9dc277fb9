"""Deviation discovery's output order and its stages: triples leave a wave in
groups through LDS, or directly when one step finds more than the stage
holds, and are sorted on the device as 64-bit keys.  Checked against the
set definition (u in the frontier, an edge u -> v with v != succ[u]), in
all three modes, from no triple to many per wave step, over frontier counts
around a tile's 16, with exact, short and zero capacity."""
import ctypes

import numpy as np
import pytest

import cpgamd
from test_simt_emulator import emu  # noqa: F401  (fixture)


def bipartite(a, b, fan, seed):
    rng = np.random.default_rng(seed)
    u = np.repeat(np.arange(a), fan)
    v = a + np.concatenate([rng.choice(b, size=fan, replace=False) for _ in range(a)])
    return a + b, u.astype(np.int32), v.astype(np.int32), rng.uniform(0.1, 1.0, a * fan).astype(np.float32)


def discover(g, frontiers, mode, cap):
    ptr = np.concatenate([[0], np.cumsum([len(f) for f in frontiers])]).astype(np.int32)
    src = np.concatenate(list(frontiers) + [np.zeros(1, np.int32)]).astype(np.int32)
    out = [np.full(max(cap, 1), -7, np.int32) for _ in range(3)]
    p = [x.ctypes.data_as(ctypes.POINTER(ctypes.c_int)) for x in [ptr, src] + out]
    return g.L.cpg_bvss_discover(g.h, len(frontiers), p[0], p[1], mode, 2, p[2], p[3], p[4], cap), out


def check(lib, a, b, fan, nfront, size):
    n, u, v, w = bipartite(a, b, fan, a + fan)
    rng = np.random.default_rng(nfront)
    g = lib.CpGen()
    try:
        g.load_edges(n, u, v, w)
        g.bvss_build()
        succ = g.sfxt()[1]
        dev = v != succ[u]
        fronts = [np.unique(rng.integers(0, a, size=size)).astype(np.int32) for _ in range(nfront)]
        want = sorted((f, int(x), int(y)) for f, fr in enumerate(fronts) for x, y in zip(u[dev], v[dev]) if x in fr)
        for mode in (0, 1, 2):
            got, out = discover(g, fronts, mode, len(want))
            assert got == len(want)
            assert list(zip(*(o[:got].tolist() for o in out))) == want
            if want:
                assert discover(g, fronts, mode, len(want) - 1)[0] == -len(want) - 1000
                assert discover(g, fronts, mode, 0)[0] == -len(want) - 1000
    finally:
        g.close()


CASES = [(64, 70, 60, 1, 400), (130, 20, 3, 17, 40), (65, 9, 1, 3, 10), (5, 4, 2, 16, 3), (200, 300, 9, 2, 150)]


@pytest.mark.parametrize("case", CASES)
def test_emulated_triples_sorted(emu, case):  # noqa: F811
    check(emu, *case)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES + [(4096, 3000, 25, 8, 3000)])
def test_gpu_triples_sorted(case):
    check(cpgamd, *case)
