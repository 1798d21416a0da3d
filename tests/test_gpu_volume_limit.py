"""The largest volume that kf_volume_create takes: 2048^3 FP32 voxels, 64 GiB, 2^32 16-byte
vectors to fill.  Created and reset, it reads free space (f = 1, w = 0) at its first voxels,
on both sides of the fill's 2^31st vector and at its last voxels."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_largest_volume_is_created_and_reset(kf, gpu):
    vol = kf.Volume(2048, 8.0, 0.05, 128.0, kf.KF_VOXEL_F32)
    assert vol.desc.n == 2048
    p, nb = C.c_void_p(), C.c_size_t()
    kf.check(kf.lib().kf_volume_data(vol.handle, C.byref(p), C.byref(nb)), "volume data")
    assert nb.value == 8 * 2048 ** 3
    free = np.tile(np.array([1.0, 0.0], np.float32), 8)
    for at in (0, nb.value // 2 - 64, nb.value // 2, nb.value - 64):
        assert np.array_equal(kf.download_ptr(p.value + at, np.float32, 16), free), at
        kf.upload_ptr(p.value + at, np.full(16, 0.5, np.float32))
    kf.check(kf.lib().kf_volume_reset(vol.handle, None), "reset")
    kf.synchronize()
    for at in (0, nb.value // 2 - 64, nb.value // 2, nb.value - 64):
        assert np.array_equal(kf.download_ptr(p.value + at, np.float32, 16), free), at
