"""The trackers' short logarithm and division against the functions they stand for, bit for bit: every number the
logarithm can be asked for, and the division over the ranges that its guard admits, both ends of each range,
mantissas at both ends, zeros, infinities and NaN among them."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _probe(op, a, b=None):
    from rtcamp8_amd._lib import call
    from rtcamp8_amd.device import DeviceBuffer

    da, out = DeviceBuffer.from_array(a), DeviceBuffer(4 * a.size)
    db = None if b is None else DeviceBuffer.from_array(b)
    call("rtc8x_math_probe", None, op, a.size, C.c_void_p(da.ptr), C.c_void_p(db.ptr if db else None), C.c_void_p(out.ptr))
    return out.download(np.uint32, a.size)


def test_the_logarithm_of_every_number_drawn():
    from oracle_lib import oracle

    u = (np.arange(1 << 23, dtype=np.float32) * np.float32(2.0 ** -23))
    got = _probe(0, u)
    assert np.array_equal(got, _probe(1, u))
    lib = oracle()
    lib.oracle_logf.restype, lib.oracle_logf.argtypes = C.c_float, [C.c_float]
    for k in [0, 1, 2, (1 << 23) - 1, *np.random.default_rng(1).integers(0, 1 << 23, 5000)]:
        assert got[k] == np.float32(-lib.oracle_logf(float(np.float32(1.0) - u[k]))).view(np.uint32), k


def _floats(rng, n, lo, hi):
    """Numbers in [2^lo, 2^hi): a quarter in the lowest and the highest binade, half of the mantissas near an end."""
    e = rng.integers(lo, hi, n)
    e[: n // 8], e[n // 8 : n // 4] = lo, hi - 1
    m = rng.integers(0, 1 << 23, n)
    near = rng.integers(0, 4, n)
    edge = rng.random(n) < 0.5
    m = np.where(edge, np.where(rng.random(n) < 0.5, near, (1 << 23) - 1 - near), m)
    return rng.permutation((((e + 127) << 23) | m).astype(np.uint32)).view(np.float32)


@pytest.mark.parametrize("op", [2, 3])
def test_the_division(op):
    rng = np.random.default_rng(40 + op)
    n = 1 << 24
    b = _floats(rng, n, -40, 40)
    b[:64] = 2.0 ** 40
    if op == 2:  # densities: any size from 2^-85 on, either sign, and what is no number
        a = _floats(rng, n, -85, 128) * rng.choice(np.array([-1.0, 1.0], np.float32), n)
        a[64 : n // 2] = _floats(rng, n // 2 - 64, -85, 41)
        a[::1001] = rng.choice(np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 3.4028235e38, -3.4028235e38, 2.0 ** 40], np.float32),
                               a[::1001].size)
    else:  # optical depths
        a = _floats(rng, n, -85, 4)
        a[::1001] = 0.0
        a[1::1001] = 16.0
    with np.errstate(all="ignore"):
        want = a / b
    got = _probe(op, np.ascontiguousarray(a), b).view(np.float32)
    assert got.dtype == want.dtype == np.float32
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    # a zero's sign aside (-0 gives +0): the trackers compare the quotient and subtract it from one
    got, want = got[~nan] + np.float32(0.0), want[~nan] + np.float32(0.0)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
