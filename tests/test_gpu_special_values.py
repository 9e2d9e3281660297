"""GPU parity with the FP32 oracle, bit for bit, where a volume's voxels are not ordinary numbers: negative
infinities, the lowest float (a common mark for no data), NaN, negative densities; both trackers."""
import ctypes as C

import numpy as np
import pytest

from oracle_lib import nthreads, oracle, oracle_seed, ptr, tables_from_leaves

pytestmark = pytest.mark.gpu

SPECIAL = {"infinite": -np.inf, "lowest": np.finfo(np.float32).min, "large": -2.0 ** 100, "nan": np.nan, "negative": -3.0}


@pytest.mark.parametrize("tracking", [0, 1])
@pytest.mark.parametrize("kind", sorted(SPECIAL))
def test_volumes_with_special_voxels(kind, tracking):
    from rtcamp8_amd import _abi
    from rtcamp8_amd import scene as sc
    from rtcamp8_amd._lib import call
    from rtcamp8_amd.device import DeviceBuffer

    rng = np.random.default_rng(21)
    origins = np.array([[x, y, z] for x in range(0, 32, 8) for y in range(0, 32, 8) for z in range(0, 32, 8)])
    values = rng.random((len(origins), 512)).astype(np.float32)
    values[rng.random(values.shape) < 0.01] = np.float32(SPECIAL[kind])
    hg = tables_from_leaves(origins, values, 1.0 / 32.0, [0.0, 0.0, 0.0, 1.0, 1.0, 1.0])
    w, h, spp = 48, 32, 4
    cfg = sc.CONFIGS["dense128"].with_(width=w, height=h, tracking=tracking, env_kind="constant", density_coeff=4.0)
    scene = sc.DeviceScene(cfg)
    dg = _abi.Grid()
    call("rtc8x_grid_upload", C.byref(hg.grid), C.byref(dg))
    try:
        p = sc.fill_params(cfg, dg, scene.env, scene.camera)
        seeds = oracle_seed(w, h, cfg.rng_seed)
        d = {"rng": DeviceBuffer.from_array(seeds), "accum": DeviceBuffer.zeros(24 * w * h), "stats": DeviceBuffer.zeros(8 * 4),
             "verts": DeviceBuffer.zeros(4 * w * h)}
        p.rng_states, p.accum, p.stats, p.path_vertices = (d[k].ptr for k in ("rng", "accum", "stats", "verts"))
        call("rtc8x_trace", None, C.byref(p), _abi.ENTRY_PATH_TRACE, spp)
        got = [d["rng"].download(np.uint64), d["accum"].download(np.uint64), d["verts"].download(np.uint32),
               d["stats"].download(np.uint64)]
        from oracle_lib import download_grid

        host = download_grid(dg)
        p = sc.fill_params(cfg, host.grid, scene.env, scene.camera)
        accum, verts, stats = np.zeros(3 * w * h), np.zeros(w * h, np.uint32), np.zeros(_abi.STAT_COUNT, np.uint64)
        p.rng_states, p.accum, p.path_vertices, p.stats = ptr(seeds), ptr(accum), ptr(verts), ptr(stats)
        assert oracle().oracle_trace_f32(C.byref(p), _abi.ENTRY_PATH_TRACE, spp, 0, h, nthreads()) == 0
    finally:
        call("rtc8x_grid_destroy", C.byref(dg))
        scene.close()
    for a, b in zip(got, (seeds, accum.view(np.uint64), verts, stats[:4])):
        assert np.array_equal(a, b)
    assert accum.any()
