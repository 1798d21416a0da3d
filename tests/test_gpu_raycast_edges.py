"""Raycasts where the march's shortcuts meet their edges, against the oracle bit for bit:
rays up and down every axis (components that are exactly zero among them), a camera inside
the volume, beside it and so far away that ends of rays round out of the trilinear domain,
a volume of one brick, few steps, and steps longer than a brick."""
import numpy as np
import pytest

from tests.helpers import fill_volume, intr, pose, ray_params, same_bits, vol_desc, voxel_centres

pytestmark = pytest.mark.gpu

PLANES = ("vx", "vy", "vz", "nx", "ny", "nz")
H = np.pi / 2
# name: rotation of the camera, distance behind the volume's centre along its axis, focal length
VIEWS = {
    "+z": ((0, 0, 0), 1.6, 60.0),
    "-z": ((np.pi, 0, 0), 1.6, 60.0),
    "+x": ((0, H, 0), 1.1, 40.0),
    "-x": ((0, -H, 0), 1.1, 40.0),
    "+y": ((-H, 0, 0), 1.6, 60.0),
    "-y": ((H, 0, 0), 1.6, 60.0),
    "diagonal": ((0.6, -2.3, 0.4), 1.5, 60.0),
    "inside": ((0.3, 0.5, -0.2), 0.35, 30.0),
    "past": ((0.3, 0.5, -0.2), -2.0, 60.0),
    "far": ((0, 0, 0), 2.0e3, 1.2e5),
    "farther": ((0, 0, 0), 1.0e4, 6.0e5),
    "far diagonal": ((0.6, -2.3, 0.4), 3.0e4, 2.0e6),
}


def _field(n, fmt):
    """A sphere, a slab of the floor and a thin plate inside a 1 m cube around (0.2, 0, 0)."""
    d = vol_desc(n, 1.0, max(0.04, 2.5 / n), fmt=fmt, origin=(-0.3, -0.5, -0.5))
    P = voxel_centres(d) - np.array([0.2, 0.0, 0.0])
    sd = np.linalg.norm(P - np.array([0.1, -0.05, 0.12]), axis=-1) - 0.17
    sd = np.minimum(sd, np.abs(P[..., 1] + 0.395) - 0.025)
    sd = np.minimum(sd, np.maximum(np.abs(P[..., 0] + 0.25) - 0.02, np.abs(P[..., 2]) - 0.2))
    return d, np.clip(sd / d.trunc_m, -1, 1).astype(np.float32)


@pytest.mark.parametrize("view", VIEWS)
@pytest.mark.parametrize("fmt", [0, 1], ids=["f32", "f16"])
@pytest.mark.parametrize("n", [8, 72])
def test_raycast_edges(gpu, kf, orc, n, fmt, view):
    d, f = _field(n, fmt)
    raw = fill_volume(d, f, 1.0)
    vol = kf.Volume(n, 1.0, d.trunc_m, 128.0, fmt, origin=(d.origin_m[0], d.origin_m[1], d.origin_m[2]))
    vol.upload_raw(raw)
    r, dist, fx = VIEWS[view]
    k = intr(97, 61, fx, fx, 48.0, 30.0)
    T = pose(*r)
    T[:3, 3] = np.array([0.2, 0.0, 0.0]) - dist * T[:3, 2]
    model, d_pose = kf.DeviceMaps(k, 3, False), kf.DevicePose(T)
    for far, near, most in ((0.8, 0.5, 2048), (0.8, 0.5, 5), (0.8, 0.5, 1), (6.0, 3.0, 2048), (0.05, 0.02, 2048)):
        p = ray_params(0.3, far, near, most)
        steps = kf.DeviceBuffer(8)
        steps.zero()
        kf.Raycaster(k, p).Raycast(vol, d_pose, model, steps=steps)
        kf.synchronize()
        om, osteps = orc.raycast(d, fmt, raw, k, p, T, 3)
        assert int(steps.download(np.uint64)[0]) == osteps, (far, most)
        for lvl in range(3):
            for nm in PLANES:
                assert same_bits(model.plane(lvl, nm), om.plane(lvl, nm)), (far, most, lvl, nm)
        if view not in ("past", "farther") and n == 72 and far == 0.8 and most == 2048:
            assert (~np.isnan(om.plane(0, "vz"))).sum() > 200


@pytest.mark.parametrize("w,h", [(319, 304), (313, 309)])
def test_raycast_block_maps(gpu, kf, orc, w, h):
    """380 and 400 blocks: the last image whose blocks cover 16x16 pixels, and an odd-sized
    one whose blocks' tiles are a quarter of the image apart; every pixel once."""
    d, f = _field(72, 1)
    raw = fill_volume(d, f, 1.0)
    vol = kf.Volume(72, 1.0, d.trunc_m, 128.0, 1, origin=(d.origin_m[0], d.origin_m[1], d.origin_m[2]))
    vol.upload_raw(raw)
    k, p = intr(w, h, 240.0, 240.0), ray_params()
    T = pose(0.6, -2.3, 0.4)
    T[:3, 3] = np.array([0.2, 0.0, 0.0]) - 1.2 * T[:3, 2]
    model, steps = kf.DeviceMaps(k, 3, False), kf.DeviceBuffer(8)
    steps.zero()
    kf.Raycaster(k, p).Raycast(vol, kf.DevicePose(T), model, steps=steps)
    kf.synchronize()
    om, osteps = orc.raycast(d, 1, raw, k, p, T, 3)
    assert int(steps.download(np.uint64)[0]) == osteps
    for lvl in range(3):
        for nm in PLANES:
            assert same_bits(model.plane(lvl, nm), om.plane(lvl, nm)), (lvl, nm)
