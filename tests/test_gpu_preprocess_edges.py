"""Preprocessing at sizes where a block's tile ends, every window size, and range weights
that do and do not reach zero inside the table, against the oracle bit for bit."""
import numpy as np
import pytest

from tests.helpers import intr, pre_params, same_bits

pytestmark = pytest.mark.gpu

PLANES = ("vx", "vy", "vz", "nx", "ny", "nz", "depth")


@pytest.mark.parametrize("w,h", [(16, 16), (17, 33), (33, 17), (65, 47), (130, 66)])
@pytest.mark.parametrize("radius", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("levels,sigma_r", [(3, 0.03), (2, 0.5), (1, 0.041)])
def test_preprocess_edges(gpu, kf, orc, w, h, radius, levels, sigma_r):
    rng = np.random.default_rng(w * h + radius)
    y, x = np.mgrid[0:h, 0:w]
    d = 900 + 9 * x + 14 * y + rng.integers(-12, 13, (h, w))
    d[rng.random((h, w)) < 0.06] = 0
    d[rng.random((h, w)) < 0.03] = 3000
    d[rng.random((h, w)) < 0.02] = 65535
    d[rng.random((h, w)) < 0.02] = 40
    d = d.astype(np.uint16)
    k = intr(w, h, 1.3 * w, 1.2 * w)
    p = pre_params(radius=radius, sigma_s=0.5 + radius, sigma_r=sigma_r)
    live, d_depth = kf.DeviceMaps(k, levels, True), kf.upload(d)
    kf.CameraHandler.updateCameraData(k, p, live, d_depth)
    kf.synchronize()
    o = orc.preprocess(k, p, d, levels)
    assert same_bits(live.raylen(), o.raylen())
    for lvl in range(levels):
        for nm in PLANES:
            assert same_bits(live.plane(lvl, nm), o.plane(lvl, nm)), (lvl, nm)
