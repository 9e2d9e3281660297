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


def _probe(grid, pts):
    from rtcamp8_amd._lib import call
    from rtcamp8_amd.device import DeviceBuffer

    n = len(pts)
    d = [DeviceBuffer.from_array(pts), DeviceBuffer(12 * n), DeviceBuffer(12 * n), DeviceBuffer(4 * n)]
    call("rtc8x_grid_probe", C.byref(grid), n, *[C.c_void_p(b.ptr) for b in d], None)
    return d[3].download(np.float32, n)


def _oracle_probe(grid, pts):
    n = len(pts)
    ijk, off, val = np.empty(3 * n, np.int32), np.empty(3 * n, np.uint32), np.empty(n, np.float32)
    oracle().oracle_grid_probe(C.byref(grid), n, ptr(pts), ptr(ijk), ptr(off), ptr(val))
    return val


@pytest.mark.parametrize("table", ["leaf_values", "tile_values"])
def test_lookups_follow_tables_put_into_a_copy(table):
    """A copy of a device grid with another table of values is looked up in that table, not in bricks that
    hold the former one's."""
    from rtcamp8_amd import _abi
    from rtcamp8_amd._lib import call
    from rtcamp8_amd.device import DeviceBuffer

    hg, origins = _grid("tiles")
    rng = np.random.default_rng(14)
    pts = np.ascontiguousarray(origins[rng.integers(0, len(origins), 4000)] + rng.uniform(-18.0, 26.0, (4000, 3)), np.float32)
    dg = _abi.Grid()
    call("rtc8x_grid_upload", C.byref(hg.grid), C.byref(dg))
    try:
        key = "values" if table == "leaf_values" else "tiles"
        other = np.ascontiguousarray(1.0 - hg.arrays[key].reshape(-1), np.float32)
        if key == "tiles":
            other[0] = hg.arrays[key][0]  # the background stays tile 0
        d = DeviceBuffer.from_array(np.append(other, np.float32(0.0)))  # one float of padding
        copy = _abi.Grid.from_buffer_copy(dg)
        setattr(copy, table, d.ptr)
        host = _abi.Grid.from_buffer_copy(hg.grid)
        setattr(host, table, other.ctypes.data)
        assert np.array_equal(_probe(copy, pts).view(np.uint32), _oracle_probe(host, pts).view(np.uint32))
        assert np.array_equal(_probe(dg, pts).view(np.uint32), _oracle_probe(hg.grid, pts).view(np.uint32))
    finally:
        call("rtc8x_grid_destroy", C.byref(dg))


def test_the_mask_fields_are_the_callers():
    """The library neither uses nor needs a device grid's host-only mask fields: with them cleared the grid is
    looked up as before and destroyed whole."""
    import torch

    from rtcamp8_amd import _abi
    from rtcamp8_amd._lib import call

    desc = _abi.FbmDesc()
    desc.resolution, desc.octaves, desc.seed = 128, 4, 5
    desc.base_frequency, desc.lacunarity, desc.gain, desc.contrast = 4.0, 2.0, 0.5, 1.0

    def cycle():
        dg = _abi.Grid()
        call("rtc8x_grid_build_fbm", C.byref(desc), C.byref(dg), None)
        assert not dg.leaf_masks and not dg.lower_masks and not dg.upper_masks
        assert dg.bricks and dg.brick_map
        dg.leaf_masks = dg.lower_masks = dg.upper_masks = None
        call("rtc8x_grid_destroy", C.byref(dg))

    cycle()
    free = torch.cuda.mem_get_info()[0]
    for _ in range(4):  # the bricks take 36 MB
        cycle()
    assert torch.cuda.mem_get_info()[0] >= free - (16 << 20)


@pytest.mark.parametrize("kind", ["one_leaf", "across_roots", "tiles"])
@pytest.mark.parametrize("leaf_map", [True, False])
def test_lookups_without_bricks_match_the_tree(kind, leaf_map):
    from rtcamp8_amd import _abi
    from rtcamp8_amd._lib import call

    hg, origins = _grid(kind)
    rng = np.random.default_rng(13)
    n = 20000
    pts = origins[rng.integers(0, len(origins), n)] + rng.uniform(-18.0, 26.0, (n, 3))
    pts[: n // 2] = np.round(pts[: n // 2] / 8.0) * 8.0 - rng.choice([0.0, 0.25, 0.5, 1.0, 7.5], (n // 2, 3))
    pts = np.ascontiguousarray(pts, np.float32)
    dg = _abi.Grid()
    call("rtc8x_grid_upload", C.byref(hg.grid), C.byref(dg))
    try:
        bare = _abi.Grid.from_buffer_copy(dg)
        bare.bricks = None
        if not leaf_map:
            bare.leaf_map = None
        assert np.array_equal(_probe(bare, pts).view(np.uint32), _oracle_probe(hg.grid, pts).view(np.uint32))
    finally:
        call("rtc8x_grid_destroy", C.byref(dg))


@pytest.mark.parametrize("tracking", [0, 1])
def test_frames_without_bricks(tracking):
    """Frames of the plain and the cache-rendering entry and training records: the same bits with and without."""
    from rtcamp8_amd import _abi
    from rtcamp8_amd import scene as sc
    from rtcamp8_amd._lib import call
    from rtcamp8_amd.nrc import NrcRenderer
    from rtcamp8_amd.tracer import PathTracer

    cfg = sc.CONFIGS["sparse512"].with_(width=75, height=41, tracking=tracking, sky_width=64, sky_height=32,
                                        fbm=sc.FbmConfig(resolution=128, seed=0x5EED0007, sparse=True,
                                                         active_leaf_fraction=0.25))
    s = sc.DeviceScene(cfg)
    npx = cfg.width * cfg.height
    got = []
    for bricks in (True, False):
        t, r = PathTracer(s), NrcRenderer(s, samples_per_launch=2)

        def params(owner):
            p = owner.params()
            if not bricks:
                p.grid.bricks = None
            return p

        for _ in range(2):
            t.trace(2, params(t))
        p = params(r)
        p.nrc.num_samples = 2
        call("rtc8x_trace", None, C.byref(p), _abi.ENTRY_PATH_TRACE_WITH_NRC, 2)
        out = [t.accum.download(np.uint64, 3 * npx), t.rng.download(np.uint64, npx), t.stats.download(np.uint64, 4),
               r.buffers.inference_terminals.download(np.uint32), r.buffers.per_frame_contribution.download(np.uint32)]
        p = params(r)
        call("rtc8x_nrc_prepare", None, C.byref(p), 1)
        call("rtc8x_trace", None, C.byref(p), _abi.ENTRY_GENERATE_TRAINING_DATA, 1)
        n = int(r.buffers.num_training_data.download(np.uint32, 2)[p.nrc.nrc_buffer_index])
        out += [np.array([n]), r.buffers.train_queries[0].download(np.uint32, 14 * min(n, 1000)), r.rng.download(np.uint64, npx)]
        got.append(out)
        t.close()
        r.close()
    s.close()
    assert got[0][5][0] > 0  # there were training records
    for a, b in zip(*got):
        assert np.array_equal(a, b)


def test_bricks_within_a_bound():
    """rtc8x_grid_build_bricks: none, none within too few bytes, all within enough, filled from the values that
    the tables hold by then; the same lookups throughout."""
    import torch

    from rtcamp8_amd import _abi
    from rtcamp8_amd._lib import call

    hg, origins = _grid("tiles")
    rng = np.random.default_rng(15)
    pts = np.ascontiguousarray(origins[rng.integers(0, len(origins), 5000)] + rng.uniform(-18.0, 26.0, (5000, 3)), np.float32)
    dg = _abi.Grid()
    call("rtc8x_grid_upload", C.byref(hg.grid), C.byref(dg))
    try:
        assert dg.bricks
        ref = _oracle_probe(hg.grid, pts).view(np.uint32)
        own = 9216 * len(origins)  # the leaves' own bricks, without those of the blocks beside them
        for most, have in ((0, False), (own, False), (16 * own, True), (0, False), (1 << 40, True)):
            call("rtc8x_grid_build_bricks", C.byref(dg), most)
            assert bool(dg.bricks) == have and bool(dg.brick_map) == have, most
            assert np.array_equal(_probe(dg, pts).view(np.uint32), ref), most
        values = np.ascontiguousarray(2.0 * hg.arrays["values"].reshape(-1), np.float32)
        call("rtc8x_memcpy_htod", C.c_void_p(dg.leaf_values), values.ctypes.data_as(C.c_void_p), values.nbytes)
        call("rtc8x_grid_build_bricks", C.byref(dg), 1 << 40)
        host = _abi.Grid.from_buffer_copy(hg.grid)
        host.leaf_values = values.ctypes.data
        assert np.array_equal(_probe(dg, pts).view(np.uint32), _oracle_probe(host, pts).view(np.uint32))
    finally:
        call("rtc8x_grid_destroy", C.byref(dg))
    desc = _abi.FbmDesc()
    desc.resolution, desc.octaves, desc.seed = 128, 4, 5
    desc.base_frequency, desc.lacunarity, desc.gain, desc.contrast = 4.0, 2.0, 0.5, 1.0
    call("rtc8x_grid_build_fbm", C.byref(desc), C.byref(dg), None)
    free = torch.cuda.mem_get_info()[0]
    call("rtc8x_grid_build_bricks", C.byref(dg), 0)
    assert torch.cuda.mem_get_info()[0] >= free + (30 << 20)  # 36 MB of bricks
    call("rtc8x_grid_destroy", C.byref(dg))
