"""kf_volume_export_tsdf into a buffer at a 16-byte boundary and off it, and volume
reset, at the smallest size, one whose last block is partial, and a full-block one."""
import ctypes as C

import numpy as np
import pytest

from tests.helpers import fill_volume

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [0, 1], ids=["f32", "f16"])
@pytest.mark.parametrize("n", [8, 24, 64])
def test_export_and_reset_edges(gpu, kf, n, fmt):
    rng = np.random.default_rng(n + fmt)
    f = rng.uniform(-1, 1, (n, n, n)).astype(np.float32)
    if fmt == kf.KF_VOXEL_F16:
        f = f.astype(np.float16).astype(np.float32)
    w = rng.integers(0, 3, (n, n, n)).astype(np.float32)
    vol = kf.Volume(n, 1.0, 0.05, 128.0, fmt)
    vol.upload_raw(fill_volume(vol.desc, f, w))
    ref = np.where(w > 0, f * np.float32(0.05), np.float32(0.05)).astype(np.float32).reshape(-1)
    for offset in (0, 1, 2, 3):  # floats past a 16-byte boundary
        out = kf.DeviceBuffer((n ** 3 + 8) * 4)
        out.upload(np.full(n ** 3 + 8, 7.0, np.float32))
        print(f"export n={n} fmt={fmt} offset={offset}", flush=True)
        kf.check(kf.lib().kf_volume_export_tsdf(vol.handle, C.c_void_p(out.ptr + 4 * offset), None), "export")
        kf.synchronize()
        got = out.download(np.float32)
        assert np.array_equal(got[offset:offset + n ** 3], ref)
        assert np.all(got[:offset] == 7.0) and np.all(got[offset + n ** 3:] == 7.0)
    kf.check(kf.lib().kf_volume_reset(vol.handle, None), "reset")
    kf.synchronize()
    f2, w2 = vol.tsdf_weight()
    assert np.all(f2 == 1.0) and np.all(w2 == 0.0)
