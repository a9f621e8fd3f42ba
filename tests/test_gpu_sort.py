"""The stable radix sort behind tile binning and per-pixel fragment lists.

Draws bin (tile, pair) items by sorting the tile keys with the pair index as
the value; the rasteriser then relies on each tile's pairs being in pair
(primitive) order, which is what a stable sort gives (the reference draws
primitives in ID order, pipeline/draw.c:84-165).  These tests sort host data
through the library's own sort scratch and compare with numpy's stable
argsort.  The sorts run back to back on that one scratch, so sums the sort
keeps between its passes must be back at zero for the next sort, and the
sizes cross every block layout: one block, the fused digit-offset passes up
to their 512-block limit, the scanned passes above it, and the long blocks
of more than 4 M items."""
import ctypes
import os

import numpy as np
import pytest

from scene_runner import REPO

LIB = os.path.join(REPO, "srp_amd", "libsrp_amd.so")

# (capacity, device count, key bits, key kind)
CASES = [
    (350_000, 350_000, 15, "tiles"),      # the 1080p mesh's pair count
    (1_000, 1_000, 15, "tiles"),          # one block
    (5_000, 3_001, 21, "uniform"),        # device count below the capacity, three passes
    (512 * 1024, 512 * 1024, 16, "few"),  # exactly the fused limit
    (440_000, 350_000, 15, "tiles"),      # capacity-sized grid, count from the device
    (600_000, 599_999, 12, "uniform"),    # scanned passes
    (5_000_000, 4_900_000, 15, "tiles"),  # long blocks
    (350_000, 350_000, 15, "tiles"),      # the first case again on the reused scratch
]


def _keys(rng, n, bits, kind):
    if kind == "uniform":
        return rng.integers(0, 1 << bits, size=n, dtype=np.uint32)
    if kind == "few":
        return rng.choice(np.array([3, 3, 200, 1 << 15, (1 << 16) - 1], np.uint32), size=n)
    # runs of neighbouring tiles, as consecutive triangles produce
    starts = rng.integers(0, (1 << bits) - 64, size=n // 8 + 1, dtype=np.uint32)
    return (np.repeat(starts, 8)[:n] + rng.integers(0, 3, size=n, dtype=np.uint32)) & ((1 << bits) - 1)


@pytest.mark.gpu
def test_radix_sort_matches_stable_argsort():
    lib = ctypes.CDLL(LIB, mode=ctypes.RTLD_LOCAL)
    lib.srp_lib_radix_sort.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_size_t,
                                       ctypes.c_int]
    rng = np.random.default_rng(20)
    for cap, count, bits, kind in CASES:
        print(f"[sort] cap={cap} count={count} bits={bits} keys={kind}", flush=True)
        keys = _keys(rng, cap, bits, kind)
        # bits above the sorted ones must ride along untouched
        keys |= rng.integers(0, 2, size=cap, dtype=np.uint32) << np.uint32(31)
        vals = np.arange(cap, dtype=np.uint32)
        k = keys.copy()
        v = vals.copy()
        lib.srp_lib_radix_sort(k.ctypes.data, v.ctypes.data, cap, count, bits)
        digit = keys[:count] & np.uint32((1 << (8 * ((bits + 7) // 8))) - 1)
        order = np.argsort(digit, kind="stable")
        assert np.array_equal(v[:count], vals[:count][order]), (cap, count, bits, kind)
        assert np.array_equal(k[:count], keys[:count][order]), (cap, count, bits, kind)


@pytest.mark.gpu
@pytest.mark.parametrize("cap,count,tiles,kind", [
    (1, 1, 1, "tiles"),             # no digit at all: one tile
    (64, 0, 300, "tiles"),          # nothing counted
    (64, 63, 2, "tiles"),
    (1_025, 1_024, 255, "tiles"),   # one full round of the block, one digit
    (5_000, 1_025, 257, "tiles"),   # a second round, two digits
    (16_384, 16_383, 3_600, "same"),
    (16_384, 16_384, 65_536, "uniform"),
    (16_384, 16_384, 32_400, "tiles"),
])
def test_one_launch_tile_sort(cap, count, tiles, kind):
    lib = ctypes.CDLL(LIB, mode=ctypes.RTLD_LOCAL)
    lib.srp_lib_tile_sort.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_size_t, ctypes.c_uint32,
                                      ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p]
    rng = np.random.default_rng(21)
    if kind == "same":
        keys = np.full(cap, tiles - 1, np.uint32)
    elif kind == "uniform":
        keys = rng.integers(0, tiles, size=cap, dtype=np.uint32)
    else:
        keys = np.minimum(np.repeat(rng.integers(0, tiles, size=cap // 4 + 1), 4)[:cap] + np.arange(cap) % 3,
                          tiles - 1).astype(np.uint32)
    order, start, end = (np.full(max(n, 1), 7, np.uint32) for n in (cap, tiles, tiles))
    lib.srp_lib_tile_sort(keys.ctypes.data, cap, count, tiles, order.ctypes.data, start.ctypes.data, end.ctypes.data)
    want = np.argsort(keys[:count], kind="stable")
    assert np.array_equal(order[:count], want)
    first = np.searchsorted(keys[:count][want], np.arange(tiles), "left")
    last = np.searchsorted(keys[:count][want], np.arange(tiles), "right")
    some = last > first
    assert np.array_equal(start, np.where(some, first, 0)) and np.array_equal(end, np.where(some, last, 0))


@pytest.mark.gpu
@pytest.mark.parametrize("cap,count,bits,kind", [
    (1 << 20, 1 << 20, 15, "tiles"),                 # the last size of the short rounds
    ((1 << 20) + 1, (1 << 20) + 1, 15, "tiles"),     # long rounds, the last one of a single item
    (1_200_000, 4_097, 9, "few"),                    # most blocks past the device count
    (9_000_000, 8_388_608, 16, "few"),               # blocks of two rounds, very uneven digits
    (9_000_000, 8_388_607, 21, "uniform"),
])
def test_long_sort_matches_stable_argsort(cap, count, bits, kind):
    lib = ctypes.CDLL(LIB, mode=ctypes.RTLD_LOCAL)
    lib.srp_lib_radix_sort.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_size_t,
                                       ctypes.c_int]
    keys = _keys(np.random.default_rng(22), cap, bits, kind)
    vals = np.arange(cap, dtype=np.uint32)[::-1].copy()
    k, v = keys.copy(), vals.copy()
    lib.srp_lib_radix_sort(k.ctypes.data, v.ctypes.data, cap, count, bits)
    order = np.argsort(keys[:count] & np.uint32((1 << (8 * ((bits + 7) // 8))) - 1), kind="stable")
    assert np.array_equal(v[:count], vals[:count][order])
    assert np.array_equal(k[:count], keys[:count][order])
