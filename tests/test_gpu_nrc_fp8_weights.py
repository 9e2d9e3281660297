"""GPU check of the FP8 inference that quantises the weights in its own workgroups: the bits of the launch that
reads the quantised copy, for the smallest and largest networks and batch sizes around the rule's line."""
import ctypes as C

import numpy as np
import pytest

from rtcamp8_amd import _abi

pytestmark = pytest.mark.gpu

LINE = 512 * 256  # queries of the largest launch that quantises for itself in every case


def _cache(encoding, layers, seed):
    from rtcamp8_amd.nrc import NeuralRadianceCache

    c = NeuralRadianceCache()
    c.initialize(num_hidden_layers=layers, precision=_abi.NRC_BF16_FP8, encoding=encoding)
    rng = np.random.default_rng(seed)
    w = rng.uniform(-0.3, 0.3, c.num_params()).astype(np.float32)
    w[:4096] *= 40.0  # layers of different scales
    if layers > 1:
        w[4096:8192] = 0.0
    c.set_weights(w)
    return c


def _queries(n):
    rng = np.random.default_rng(n)
    q = np.zeros((n, 14), np.float32)
    q[:, 0:3] = rng.random((n, 3), dtype=np.float32)
    q[:, 3:7] = rng.random((n, 4), dtype=np.float32) * 3.0
    q[:, 8:11] = 0.99
    return q


@pytest.mark.parametrize("layers", [1, 2, 5, 8])
@pytest.mark.parametrize("encoding", [0, 1])
@pytest.mark.parametrize("n", [LINE, LINE + 1, LINE + 64 * 1000 + 7])
def test_own_weights_equal_the_quantised_copy(n, encoding, layers):
    from rtcamp8_amd.device import DeviceBuffer
    from rtcamp8_amd.nrc import round_up

    c = _cache(encoding, layers, layers)
    stride = round_up(n, 128)
    q = np.zeros((stride, 14), np.float32)
    q[:n] = _queries(n)
    dq, out, pieces = DeviceBuffer.from_array(q), DeviceBuffer.zeros(12 * stride), DeviceBuffer.zeros(12 * stride)
    # one launch over every slot, masked (the quantised copy beyond the line)
    terms = np.zeros((n, 4), np.uint32)
    terms[:, 3] = 1
    dt = DeviceBuffer.from_array(terms)
    p = _abi.FrameParams()
    p.image_width, p.image_height = n, 1
    p.nrc.num_samples = 1
    p.nrc.inference_queries, p.nrc.inferred_radiance, p.nrc.inference_terminals = dq.ptr, out.ptr, dt.ptr
    c.infer_render(None, p)
    whole = out.download(np.uint32, 3 * n)
    # whole wavefronts of small launches (their own weights)
    for a in range(0, n, 64 * 500):
        c.infer(None, dq.ptr + 56 * a, min(64 * 500, n - a), pieces.ptr + 12 * a)
    assert np.array_equal(whole, pieces.download(np.uint32, 3 * n))
    # the unmasked launch of the same size
    c.infer(None, dq.ptr, n, pieces.ptr)
    assert np.array_equal(whole, pieces.download(np.uint32, 3 * n))
    c.finalize()
