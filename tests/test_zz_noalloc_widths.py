"""The no-allocation suffix forest changes its grid with the width of the
levels: graphs that stay narrow or wide, that change once, back and forth, and
more often than the loop follows, with the levels on either side of both
lines.  dist, succ and level equal the oracle's."""
import numpy as np
import pytest

import cpgamd
import pyoracle
from test_sfxt_schedule import layered
from test_simt_emulator import emu  # noqa: F401  (fixture)
from test_zz_no_alloc import Hip, run_noalloc


class HostMemory:
    """The emulator's device memory is the host's."""

    def __init__(self):
        self.live = {}

    def put(self, arr):
        arr = np.ascontiguousarray(arr).copy() if arr.size else np.zeros(1, arr.dtype)
        self.live[arr.ctypes.data] = arr
        return arr.ctypes.data

    def get(self, p, n, dtype=np.int32):
        return self.live[p][:n].copy()

    def free_all(self):
        self.live.clear()


WIDE, NARROW = [4100, 4100], [6, 900, 900, 6]
SINKS = 131072  # the least size that changes grids; level 0 does not count as wide
SHAPES = {  # sources first; the loop goes from the last level up
    "small": NARROW + WIDE + [SINKS - 10100],
    "narrow": [40, 2400, 2400, 2400, SINKS],
    "at_the_lines": [7, 1000, 1000, 999, 4000, 4000, 4001, 5, 5, SINKS],
    "wide": [3, 4100, 4100, 4100, 4100, SINKS],
    "wide_to_narrow": NARROW + WIDE + [SINKS],
    "narrow_to_wide": [2, 4500] + WIDE + NARROW + [SINKS],
    "both_ways": NARROW + WIDE + NARROW + WIDE + NARROW + [SINKS],
    "often": [4] + 5 * (WIDE + NARROW) + [SINKS],
}


def check(lib, mem, shape):
    n, u, v, w = layered(SHAPES[shape], 2, 70)
    dist, succ, level, levels = pyoracle.OracleGraph.from_edges(n, u, v, w).sfxt()
    try:
        for _ in range(2):
            got, outs = run_noalloc(mem, lib, n, u, v, w)
            assert got == levels
            for want, have in zip((dist, succ, level), outs):
                np.testing.assert_array_equal(have, want)
    finally:
        mem.free_all()


@pytest.mark.parametrize("shape", ["narrow", "at_the_lines", "both_ways", "often"])
def test_emulated_noalloc_widths(emu, shape):  # noqa: F811
    check(emu.lib(), HostMemory(), shape)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_gpu_noalloc_widths(shape):
    print(f"case noalloc widths {shape}", flush=True)
    check(cpgamd.lib(), Hip(), shape)
