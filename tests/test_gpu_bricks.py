"""GPU check of the lookup bricks: probes of uploaded grids equal the oracle's tree lookups bit for bit, at
block faces, in and beside tiles of several values, around one lone leaf, across root tiles and the index
origin, and outside the leaf map."""
import ctypes as C

import numpy as np
import pytest

from oracle_lib import LOWER, TILE, download_grid, oracle, ptr, tables_from_leaves

pytestmark = pytest.mark.gpu


def _grid(kind):
    rng = np.random.default_rng(11)
    if kind == "one_leaf":
        origins = np.array([[16, 8, 24]])
    elif kind == "across_roots":
        origins = np.array([[x, y, z] for x in (-16, -8, 0) for y in (-8, 0) for z in (-8, 4088, 4096)])
    else:
        origins = 8 * np.array([[x, y, z] for x in range(5) for y in range(4) for z in range(6)
                                if rng.random() < 0.4 or (x, y, z) == (0, 0, 0)])
    values = rng.random((len(origins), 512)).astype(np.float32)
    hg = tables_from_leaves(origins, values, 1.0, [*origins.min(0), *(origins.max(0) + 8)])
    if kind == "tiles":
        hg.arrays["tiles"] = np.array([0.0, 0.25, 0.75], np.float32)
        hg.grid.tile_values = hg.arrays["tiles"].ctypes.data
        lower = hg.arrays["lower"][:LOWER]
        free = np.flatnonzero(lower == TILE)
        lower[free[: free.size // 2]] = TILE | 1  # a slab of one value, beside leaves and other tiles
        lower[free[free.size // 2 :: 3]] = TILE | 2
    return hg, origins


@pytest.mark.parametrize("kind", ["one_leaf", "across_roots", "tiles"])
def test_brick_lookups_match_the_tree(kind):
    from rtcamp8_amd import _abi
    from rtcamp8_amd._lib import call
    from rtcamp8_amd.device import DeviceBuffer

    hg, origins = _grid(kind)
    rng = np.random.default_rng(12)
    n = 30000
    # around the leaves' blocks (the margin of the leaf map and a block beyond it), a third at block faces
    pts = origins[rng.integers(0, len(origins), n)] + rng.uniform(-18.0, 26.0, (n, 3))
    pts[: n // 3, rng.integers(0, 3)] = np.round(pts[: n // 3, 0:1] / 8.0)[:, 0] * 8.0 - rng.choice([0.0, 0.5, 1.0], n // 3)
    pts = np.ascontiguousarray(pts, np.float32)
    dg = _abi.Grid()
    call("rtc8x_grid_upload", C.byref(hg.grid), C.byref(dg))
    try:
        d = [DeviceBuffer.from_array(pts), DeviceBuffer(12 * n), DeviceBuffer(12 * n), DeviceBuffer(4 * n)]
        call("rtc8x_grid_probe", C.byref(dg), n, *[C.c_void_p(b.ptr) for b in d], None)
        ijk, off, val = np.empty(3 * n, np.int32), np.empty(3 * n, np.uint32), np.empty(n, np.float32)
        oracle().oracle_grid_probe(C.byref(hg.grid), n, ptr(pts), ptr(ijk), ptr(off), ptr(val))
        assert np.array_equal(d[3].download(np.float32, n).view(np.uint32), val.view(np.uint32))
        if kind == "one_leaf":
            # tables copied by hand, the device grid's fields with them, encode as the library's own copy does
            ref = _abi.Grid()
            call("rtc8x_grid_download", C.byref(dg), C.byref(ref))
            copied, sizes = download_grid(dg), []
            for g in (copied.grid, ref):
                size = C.c_size_t(0)
                call("rtc8x_nanovdb_encode", C.byref(g), b"g", None, 0, C.byref(size))
                sizes.append(size.value)
            call("rtc8x_grid_free_host", C.byref(ref))
            assert sizes[0] == sizes[1] > 0
    finally:
        call("rtc8x_grid_destroy", C.byref(dg))
