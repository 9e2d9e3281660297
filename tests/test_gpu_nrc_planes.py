"""GPU check of the hash-grid inference from staged planes: large batches give the bits that the same queries
give in batches below its threshold, at the threshold, at ragged sizes of one and of several tiles per
workgroup, after a training step (the planes follow the tables), and under a render mask."""
import ctypes as C

import numpy as np
import pytest

from rtcamp8_amd import _abi

pytestmark = pytest.mark.gpu

MIN, MIN_MASKED, PIECE = 3 * 256 * 256 + 256, 1 << 21, 100000


def _queries(n, seed):
    rng = np.random.default_rng(seed)
    q = np.zeros((n, 14), np.float32)
    q[:, 0:3] = rng.random((n, 3), dtype=np.float32) * 1.2 - 0.1  # beyond [0, 1] too
    q[::97, 0:3] = np.round(q[::97, 0:3])
    q[:, 3] = rng.random(n, dtype=np.float32) * np.pi
    q[:, 4] = rng.random(n, dtype=np.float32) * 2 * np.pi
    q[:, 5:7] = q[:, 3:5]
    q[:, 8:11] = 0.99
    return q


def _cache(precision, layers=2):
    from rtcamp8_amd.nrc import NeuralRadianceCache

    c = NeuralRadianceCache()
    c.initialize(num_hidden_layers=layers, precision=precision, encoding=1)
    w = np.random.default_rng(5).uniform(-0.3, 0.3, c.num_params()).astype(np.float32)
    c.set_weights(w)
    return c


def _in_pieces(c, dq, n):
    from rtcamp8_amd.device import DeviceBuffer

    out = DeviceBuffer(12 * n)
    for a in range(0, n, PIECE):
        c.infer(None, dq.ptr + 56 * a, min(PIECE, n - a), out.ptr + 12 * a)
    return out.download(np.uint32, 3 * n)


@pytest.mark.parametrize("precision", [_abi.NRC_FP16, _abi.NRC_BF16])
@pytest.mark.parametrize("n", [MIN, MIN + 1, 256 * 512 * 8 + 513, 1234567])
def test_large_batches_equal_small_ones(n, precision):
    from rtcamp8_amd.device import DeviceBuffer

    c = _cache(precision, layers=2 if n % 2 else 3)
    dq = DeviceBuffer.from_array(_queries(n, n))
    out = DeviceBuffer.zeros(12 * n + 64)
    for step in range(2):
        c.infer(None, dq.ptr, n, out.ptr)
        got = out.download(np.uint32, 3 * n + 16)
        assert np.array_equal(got[: 3 * n], _in_pieces(c, dq, n)), step
        assert not got[3 * n :].any()  # nothing behind the last query
        t = DeviceBuffer.from_array(np.random.default_rng(step).random((4096, 3)).astype(np.float32))
        c.train(None, dq.ptr, t.ptr, 4096)  # the second round sees other tables
    c.finalize()


@pytest.mark.parametrize("live", [0.0, 0.15, 1.0])
def test_masked_slots(live):
    """Live slots get what the whole batch gives them; the others keep what they held."""
    from rtcamp8_amd.device import DeviceBuffer
    from rtcamp8_amd.nrc import round_up

    w, h, k = 811, 647, 4
    npx = w * h
    stride = round_up(npx, 128)
    n = stride * k
    assert n >= MIN_MASKED
    c = _cache(_abi.NRC_FP16)
    dq = DeviceBuffer.from_array(_queries(n, 3))
    flags = np.random.default_rng(9).random((k, npx)) < live
    terms = np.zeros((k * npx, 4), np.uint32)
    terms[:, 3] = flags.reshape(-1) | 0x500
    dt = DeviceBuffer.from_array(terms)
    out = DeviceBuffer.from_array(np.full(3 * n, 7, np.uint32))
    p = _abi.FrameParams()
    p.image_width, p.image_height = w, h
    p.nrc.num_samples = k
    p.nrc.inference_queries, p.nrc.inferred_radiance, p.nrc.inference_terminals = dq.ptr, out.ptr, dt.ptr
    c.infer_render(None, p)
    got = out.download(np.uint32, 3 * n).reshape(k, stride, 3)
    ref = _in_pieces(c, dq, n).reshape(k, stride, 3)
    on = np.zeros((k, stride), bool)
    on[:, :npx] = flags
    assert np.array_equal(got[on], ref[on])
    assert (got[~on] == 7).all()
    c.finalize()


@pytest.mark.parametrize("precision", [_abi.NRC_FP16, _abi.NRC_BF16])
@pytest.mark.parametrize("live", ["one", "0.3 %", "a disc", "511 and 512"])
def test_tiles_of_few_queries(live, precision):
    """Tiles below and at the line under which corners are gathered from memory: the bits of the whole batch."""
    from rtcamp8_amd.device import DeviceBuffer
    from rtcamp8_amd.nrc import round_up

    w, h, k = 1024, 640, 4
    npx = w * h
    stride = round_up(npx, 128)
    n = stride * k
    assert n >= MIN_MASKED
    c = _cache(precision, layers=3)
    dq = DeviceBuffer.from_array(_queries(n, 4))
    flags = np.zeros((k, npx), bool)
    rng = np.random.default_rng(10)
    if live == "one":
        flags[2, npx - 1] = True
    elif live == "0.3 %":
        flags = rng.random((k, npx)) < 0.003
    elif live == "a disc":
        y, x = np.divmod(np.arange(npx), w)
        flags[:] = (x - 700) ** 2 + (y - 300) ** 2 < 90 ** 2
    else:  # whole blocks of 512 slots, and blocks with one slot less
        flags[0, : 512 * 256] = True
        flags[0, ::1024] = False
    terms = np.zeros((k * npx, 4), np.uint32)
    terms[:, 3] = flags.reshape(-1) | 0x300
    dt = DeviceBuffer.from_array(terms)
    out = DeviceBuffer.from_array(np.full(3 * n, 7, np.uint32))
    p = _abi.FrameParams()
    p.image_width, p.image_height = w, h
    p.nrc.num_samples = k
    p.nrc.inference_queries, p.nrc.inferred_radiance, p.nrc.inference_terminals = dq.ptr, out.ptr, dt.ptr
    c.infer_render(None, p)
    got = out.download(np.uint32, 3 * n).reshape(k, stride, 3)
    ref = _in_pieces(c, dq, n).reshape(k, stride, 3)
    on = np.zeros((k, stride), bool)
    on[:, :npx] = flags
    assert on.any() and np.array_equal(got[on], ref[on])
    assert (got[~on] == 7).all()
    c.finalize()


@pytest.mark.parametrize("n", [MIN - 1, MIN, MIN + 255])
def test_at_the_line(n):
    """The last batch of the direct kernel and the first ones of the planes."""
    from rtcamp8_amd.device import DeviceBuffer

    c = _cache(_abi.NRC_FP16, layers=8)
    dq = DeviceBuffer.from_array(_queries(n, n))
    out = DeviceBuffer.zeros(12 * n)
    c.infer(None, dq.ptr, n, out.ptr)
    assert np.array_equal(out.download(np.uint32, 3 * n), _in_pieces(c, dq, n))
    c.finalize()
