"""The kernels' arithmetic helpers that stand in for IEEE operations, against the host's.

* reciprocal: the quotient 1 / z, bit for bit, at every mantissa of the first and last
  binades that it may meet and of two between (a factor of two changes no mantissa), and
  where the quotient turns subnormal.
* bf16_rne: the nearest BF16 number, ties to even, as integer arithmetic on the bits gives
  it, at every upper half with the lower halves around the ties.
* pivot_inverse: within one unit in the last place of the FP64 quotient."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dm(kf):
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libdevicemath.so")
    L = C.CDLL(path)
    L.dm_reciprocals.argtypes = L.dm_bf16s.argtypes = [C.c_uint32, C.c_uint32, C.c_uint32, C.c_void_p]
    L.dm_pivots.argtypes = [C.c_void_p, C.c_uint32, C.c_void_p]
    return L


@pytest.mark.parametrize("exponent", [-20, -1, 0, 125, 126, 127])
def test_reciprocal(gpu, kf, dm, exponent):
    n, first = 1 << 23, (127 + exponent) << 23
    out = kf.DeviceBuffer(4 * n)
    assert dm.dm_reciprocals(first, 1, n, out.ptr) == 0
    kf.synchronize()
    z = np.arange(first, first + n, dtype=np.uint32).view(np.float32)
    want = np.float32(1.0) / z
    assert np.array_equal(out.download(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("low", [0x0000, 0x0001, 0x7fff, 0x8000, 0x8001, 0xffff])
def test_bf16(gpu, kf, dm, low):
    n = 1 << 16
    out = kf.DeviceBuffer(2 * n)
    assert dm.dm_bf16s(low, 1 << 16, n, out.ptr) == 0
    kf.synchronize()
    bits = (np.arange(n, dtype=np.uint64) << np.uint64(16)) | np.uint64(low)
    want = ((bits + np.uint64(0x7fff) + ((bits >> np.uint64(16)) & np.uint64(1))) >> np.uint64(16)).astype(np.uint16)
    number = ~np.isnan(bits.astype(np.uint32).view(np.float32))
    got = out.download(np.uint16)
    assert np.array_equal(got[number], want[number])


def test_pivot_inverse(gpu, kf, dm):
    rng = np.random.default_rng(5)
    n = 1 << 20
    m = 1.0 + rng.random(n)
    m[:4] = 1.0, np.nextafter(2.0, 0.0), np.nextafter(1.0, 2.0), 1.5
    d = np.ldexp(m, rng.integers(-300, 300, n))
    d[4:] *= rng.choice([-1.0, 1.0], n - 4)
    din, out = kf.upload(d), kf.DeviceBuffer(8 * n)
    assert dm.dm_pivots(din.ptr, n, out.ptr) == 0
    kf.synchronize()
    want = 1.0 / d
    assert np.all(np.abs(out.download(np.float64) - want) <= np.spacing(np.abs(want)))
