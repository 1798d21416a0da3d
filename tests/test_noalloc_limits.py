"""Image sizes that kf_icp_track_noalloc rejects, checked before anything touches a device:
786,432 pixels at level 0 and 262,144 at a coarser level are the largest that iterate."""
import ctypes as C

import pytest

from openfusion_amd import kinfu as kf
from tests.helpers import icp_params, intr


def _status(w, h, iters):
    k = intr(w, h, fx=0.9 * w, fy=0.9 * w)
    maps = kf.FrameMaps()  # no planes: an accepted size is turned down later, for these
    buf = (C.c_double * 64)()
    r = kf.lib().kf_icp_track_noalloc(C.byref(k), C.byref(icp_params(iters=iters)), C.byref(maps), C.byref(maps),
                                      C.addressof(buf), C.addressof(buf), None, None)
    return r, kf.lib().kf_last_error()


@pytest.mark.parametrize("w,h,iters,rejected", [
    (1024, 768, (3, 0, 0), False), (1025, 768, (3, 0, 0), True),
    (1024, 1024, (0, 3, 0), False), (1026, 1024, (0, 3, 0), True), (1500, 1000, (0, 3, 0), True),
    (1500, 1000, (0, 0, 3), False), (2052, 2048, (0, 0, 3), True),
])
def test_sizes(w, h, iters, rejected):
    r, msg = _status(w, h, iters)
    assert r != 0
    assert (b"too large for kf_icp_track_noalloc" in msg) == rejected
    if rejected:
        assert r == 1  # KF_ERR_INVALID_ARGUMENT
