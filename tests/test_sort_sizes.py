"""The device sort at its size limits: one key, the largest one-launch sort
(8,192 keys) and one more, whole and ragged tiles, and both tile sizes
(2,097,152 keys and one more), by way of the sorted deviation triples of a
graph with exactly that many; and costs of every byte pattern (ties, wide
and narrow ranges) by way of queries."""
import numpy as np
import pytest

import cpgamd
from test_bvss_order import discover
from test_round_batches import check
from test_simt_emulator import emu  # noqa: F401  (fixture)
from test_walk_lanes import rows


def check_count(lib, count):
    """`count` sources of two fanouts each: one deviation per source."""
    rng = np.random.default_rng(count)
    mid = max(2, min(count, 5000))
    u = np.repeat(np.arange(count), 2)
    first = rng.integers(0, mid, count)
    v = np.stack([first, (first + 1 + rng.integers(0, mid - 1, count)) % mid], 1).ravel() + count
    w = rng.uniform(0.1, 1.0, 2 * count).astype(np.float32)
    g = lib.CpGen()
    try:
        g.load_edges(count + mid, u.astype(np.int32), v.astype(np.int32), w)
        g.bvss_build()
        succ = g.sfxt()[1]
        keep = v != succ[u]
        assert keep.sum() == count
        got, out = discover(g, [np.arange(count)], 1, count)
        assert got == count
        np.testing.assert_array_equal(out[0], 0)
        np.testing.assert_array_equal(out[1], u[keep])
        np.testing.assert_array_equal(out[2], v[keep])
    finally:
        g.close()


@pytest.mark.parametrize("count", [1, 2, 257, 1025])
def test_emulated_sort_sizes(emu, count):  # noqa: F811
    check_count(emu, count)


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 2, 255, 1024, 1025, 8191, 8192, 8193, 9216, 262145, (1 << 21) - 1, 1 << 21,
                                   (1 << 21) + 1])
def test_gpu_sort_sizes(count):
    check_count(cpgamd, count)


@pytest.mark.gpu
@pytest.mark.parametrize("scale,offset", [(1.0, 0.0), (1e-3, 5.0), (300.0, 0.0), (0.0, 2.0)])
def test_gpu_sort_cost_ranges(scale, offset):
    n, u, v, w = rows(3, 12, 50, 13, False)
    check(cpgamd, (n, u, v, (w * np.float32(scale) + np.float32(offset)).astype(np.float32)),
          [1, 100, 8000, 9000, 60000])


@pytest.mark.gpu
def test_gpu_sort_negative_costs():
    n, u, v, w = rows(3, 12, 50, 14, False)
    check(cpgamd, (n, u, v, w - np.float32(0.4)), [1, 100, 9000])
