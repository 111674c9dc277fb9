"""Deviation discovery's output order and its stages: triples leave a wave in
groups through LDS, or directly when one step finds more than the stage
holds, and are sorted on the device as 64-bit keys.  Checked against the
set definition (u in the frontier, an edge u -> v with v != succ[u]), in
all three modes, from no triple to many per wave step, over frontier counts
around a tile's 16, with exact, short and zero capacity."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import cpgamd
from test_simt_emulator import SIMT, emu  # noqa: F401  (fixture)


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


def check_sort_line(lib):
    """Numbers of triples around the line between the host's sort and the
    device's (each source leaves all its edges but one)."""
    for a in (511, 512, 513):
        n, u, v, w = bipartite(a, 40, 4, a)
        with lib.CpGen() as g:
            g.load_edges(n, u, v, w)
            g.bvss_build()
            dev = v != g.sfxt()[1][u]
            got, out = discover(g, [np.arange(a)], 0, 4 * a)
            assert got == 3 * a == dev.sum()
            want = sorted(zip(u[dev].tolist(), v[dev].tolist()))
            assert list(zip(out[1][:got].tolist(), out[2][:got].tolist())) == want
            assert not out[0][:got].any()


def test_emulated_triples_at_the_sort_line(emu):  # noqa: F811
    check_sort_line(emu)


@pytest.mark.gpu
def test_gpu_triples_at_the_sort_line():
    check_sort_line(cpgamd)


@pytest.fixture
def parts(emu):  # noqa: F811
    """The emulator with keys of 18 bits, in place of the other one."""
    subprocess.run(["make", "-s", "-C", SIMT, "libcpgamd_simt_parts.so"], check=True)
    saved, cpgamd._lib = cpgamd._lib, cpgamd.load_library(os.path.join(SIMT, "libcpgamd_simt_parts.so"))
    yield cpgamd
    cpgamd._lib = saved


@pytest.mark.parametrize("case", [(64, 70, 60, 5, 400), (130, 20, 3, 17, 40), (65, 9, 1, 33, 10), (30, 100, 2, 8, 6)])
def test_emulated_triples_in_parts(parts, case):
    """More frontiers than one key holds."""
    check(parts, *case)


def test_emulated_parts_and_capacity(parts):
    """Parts that fill the caller's arrays, overrun them, or find nothing."""
    n, u, v, w = bipartite(80, 60, 3, 5)
    fronts = [np.arange(f, 80, 17, dtype=np.int32) if f % 3 else np.zeros(0, np.int32) for f in range(14)]
    with parts.CpGen() as g:
        g.load_edges(n, u, v, w)
        total, full = discover(g, fronts, 0, 4096)
        assert total > 60
        for cap in sorted({0, 1, 7, total // 2, total // 2 + 1, total - 1, total, total + 2}):
            got, out = discover(g, fronts, 0, cap)
            assert got == (total if cap >= total else -total - 1000)
            if cap >= total:
                for a, b in zip(full, out):
                    np.testing.assert_array_equal(a[:total], b[:total])
                    assert (b[total:] == -7).all()
        one = [x.ctypes.data_as(ctypes.POINTER(ctypes.c_int)) for x in
               (np.array([0, 5] + [10] * 8, np.int32), np.arange(10, dtype=np.int32))]
        assert g.L.cpg_bvss_discover(g.h, 9, one[0], one[1], 0, 4, None, None, None, 4096) > 0  # counts only
