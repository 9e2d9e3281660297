"""GPU parity of the slot scheduler with the FP32 oracle, bit for bit, at the sizes where it changes its
ways: one pixel, fewer pixels than workgroups, ragged images dealt out to the workgroups, and more pixels
than all slots hold (the work counter, with and without a work order); both trackers, a region table small
and large, a majorant beyond the range of the fast division."""
import numpy as np
import pytest

from oracle_lib import trace_parity_case

pytestmark = pytest.mark.gpu


def _check(res, pixels, spp):
    assert res["rng_equal"] and res["vertices_equal"]
    assert np.array_equal(res["gpu_accum"].view(np.uint64), res["cpu_accum"].view(np.uint64))
    assert res["paths"] == pixels * spp
    assert res["lookups"] == int(res["cpu_stats"][2])


@pytest.mark.parametrize("tracking", [0, 1])
@pytest.mark.parametrize("width,height,spp", [(1, 1, 3), (9, 3, 2), (157, 83, 1)])
def test_few_pixels(width, height, spp, tracking):
    _check(trace_parity_case("dense128", width=width, height=height, spp=spp, tracking=tracking, fbm_resolution=64),
           width * height, spp)


@pytest.mark.parametrize("tracking,config", [(0, "sparse512"), (1, "sparse512"), (1, "dense128")])
def test_more_pixels_than_slots(tracking, config):
    """Two launches: the second takes the pixels in the work order of the first."""
    w, h = 701, 547
    res = trace_parity_case(config, width=w, height=h, spp=2, tracking=tracking, fbm_resolution=64, samples_per_launch=1,
                            env_kind="constant", max_path_length=24)
    _check(res, w * h, 2)


@pytest.mark.parametrize("region_cells", [1, 2])
def test_large_region_table(region_cells):
    """32,768 regions (the largest table) and 4,096 on the 256^3 cloud."""
    _check(trace_parity_case("sparse512", width=96, height=54, spp=2, tracking=1, fbm_resolution=256, env_kind="constant",
                             region_cells=region_cells), 96 * 54, 2)


@pytest.mark.parametrize("tracking", [0, 1])
def test_majorant_below_the_fast_divisions_range(tracking):
    _check(trace_parity_case("dense128", width=40, height=24, spp=2, tracking=tracking, fbm_resolution=64,
                             density_coeff=2.0 ** -42), 40 * 24, 2)


@pytest.mark.parametrize("tracking", [0, 1])
@pytest.mark.parametrize("width,height", [(362, 362), (364, 361), (14563, 9), (16384, 8)])
def test_at_the_line_of_few_paths(width, height, tracking):
    """Just below, above and at 512 pixels a workgroup on 256 CUs; and below it with rows that its tiles pad to
    more than the slots of the small variant."""
    _check(trace_parity_case("dense128", width=width, height=height, spp=1, tracking=tracking, fbm_resolution=64,
                             env_kind="constant", max_path_length=12), width * height, 1)


@pytest.mark.parametrize("tracking,config", [(0, "sparse512"), (1, "sparse512"), (0, "dense128")])
def test_several_samples_from_the_work_counter(tracking, config):
    """More pixels than slots, three samples a launch: the pixels' PCG streams run on from sample to sample while
    the slots take their next pixels from the counter; two launches, the second in work order."""
    w, h = 701, 547
    _check(trace_parity_case(config, width=w, height=h, spp=6, tracking=tracking, fbm_resolution=64, samples_per_launch=3,
                             env_kind="constant", max_path_length=24), w * h, 6)


@pytest.mark.parametrize("tracking", [0, 1])
def test_cache_rendering_from_the_work_counter(tracking):
    """PATH_TRACE_WITH_NRC with more pixels than slots and three samples a launch, without and with a work order:
    PCG states, terminals, contributions and the queries of live slots are the oracle's."""
    import ctypes as C

    from oracle_lib import oracle
    from rtcamp8_amd import _abi
    from rtcamp8_amd._lib import call
    from test_gpu_nrc import HostNrc, _host_params, _nrc_case

    w, h, k = 701, 547, 3
    cfg, ds, r = _nrc_case(width=w, height=h, tracking=tracking)
    n, nq = w * h, (w * h + 127) // 128 * 128
    b = r.buffers
    for ordered in (False, True):
        p = r.params()
        p.nrc.num_samples = k
        p.pixel_cost = r.cost.ptr
        if ordered:
            call("rtc8x_order_by_tile_cost", None, C.c_void_p(r.cost.ptr), w, h, C.c_void_p(r.order.ptr),
                 C.c_void_p(r.order_scratch.ptr))
            p.work_order = r.order.ptr
        rng = r.rng.download(np.uint64, n)
        before = HostNrc(b)
        call("rtc8x_trace", None, C.byref(p), _abi.ENTRY_PATH_TRACE_WITH_NRC, k)
        after = HostNrc(b)
        accum = np.zeros(3 * n)
        hp, keep = _host_params(cfg, ds, r, before, rng, accum)
        hp.nrc.num_samples = k
        assert oracle().oracle_trace_f32(C.byref(hp), _abi.ENTRY_PATH_TRACE_WITH_NRC, k, 0, 10 ** 6, 8) == 0
        assert np.array_equal(rng, r.rng.download(np.uint64, n))
        ta, tg = (x.a["inference_terminals"].reshape(-1, 4)[: k * n] for x in (before, after))
        assert np.array_equal(ta.view(np.uint32), tg.view(np.uint32))
        assert np.array_equal(before.a["per_frame_contribution"][: 3 * k * n].view(np.uint32),
                              after.a["per_frame_contribution"][: 3 * k * n].view(np.uint32))
        for s in range(k):
            live = (ta[s * n : (s + 1) * n, 3] & 1) == 1
            assert live.sum() > 1000
            qa, qg = (x.a["inference_queries"].reshape(-1, 14)[s * nq : s * nq + n][live] for x in (before, after))
            assert np.array_equal(qa.view(np.uint32), qg.view(np.uint32))
    r.close()
    ds.close()
