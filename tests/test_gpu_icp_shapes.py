"""Tracking steps at the image sizes where a step's pixels per block change and end: the
smallest image, the last and first size of each block shape, and one that needs a second
pass; counts against the oracle, poses against the same rows summed in FP64 (the oracle
rounds each product to FP32) and, bit for bit, against the single-launch form."""
import numpy as np
import pytest

from tests.helpers import icp_params, intr, pose

pytestmark = pytest.mark.gpu


def _maps(k, T, w2c):
    """Vertices and normals (H, W, 3) of the surface z = 2 + bumps seen from the camera T,
    in camera coordinates (w2c) or the world, a few pixels invalid."""
    y, x = np.mgrid[0:k.height, 0:k.width].astype(np.float64)
    d = np.stack([(x - k.cx) / k.fx, (y - k.cy) / k.fy, np.ones_like(x)], -1) @ T[:3, :3].T
    o = T[:3, 3]
    bump = lambda a, b: 0.12 * np.sin(3.1 * a) * np.cos(2.3 * b) + 0.05 * np.sin(7.0 * a + 4.0 * b)  # noqa: E731
    t = np.full_like(x, 2.0)
    for _ in range(30):
        p = o + t[..., None] * d
        t -= 0.8 * (p[..., 2] - 2.0 - bump(p[..., 0], p[..., 1])) / d[..., 2]
    p = o + t[..., None] * d
    a, b = p[..., 0], p[..., 1]
    gx = 0.12 * 3.1 * np.cos(3.1 * a) * np.cos(2.3 * b) + 0.35 * np.cos(7.0 * a + 4.0 * b)
    gy = -0.12 * 2.3 * np.sin(3.1 * a) * np.sin(2.3 * b) + 0.2 * np.cos(7.0 * a + 4.0 * b)
    n = np.stack([gx, gy, -np.ones_like(gx)], -1)
    n /= np.linalg.norm(n, axis=-1, keepdims=True)
    if w2c:
        p, n = (p - o) @ T[:3, :3], n @ T[:3, :3]
    bad = (x + 3 * y) % 37 == 0
    p[bad] = np.nan
    n[bad] = np.nan
    return p, n


def _track(k, live, model, iters, dist, deg):
    """The tracker's iterations: rows in FP32 as the kernels form them, sums and solve in FP64."""
    f = np.float32
    (d, nd), (s, m) = [[a.reshape(-1, 3).astype(f).T for a in mp] for mp in (live, model)]
    K = [f(v) for v in (k.fx, k.fy, k.cx, k.cy)]
    cos_gate = f(np.cos(deg * np.pi / 180.0))
    T = np.eye(4)

    def rot(R, v):
        return [(R[i, 0] * v[0] + R[i, 1] * v[1]) + R[i, 2] * v[2] for i in range(3)]

    for _ in range(iters):
        R, t = T[:3, :3], T[:3, 3]
        ti = [-((R[0, c] * t[0] + R[1, c] * t[1]) + R[2, c] * t[2]) for c in range(3)]
        Rf, Rif = R.astype(f), R.T.astype(f)
        with np.errstate(invalid="ignore"):
            c = [a + f(b) for a, b in zip(rot(Rif, s), ti)]
            iz = f(1) / c[2]
            u, v = ((K[i] * c[i] + K[2 + i] * c[2]) * iz for i in (0, 1))
            ru, rv = (np.where(a - np.floor(a) < f(0.5), np.floor(a), np.ceil(a)) for a in (u, v))
            ok = ~np.isnan(d[2]) & ~np.isnan(s[0]) & (c[2] > f(1e-6)) & (ru >= 0) & (ru < k.width) & (rv >= 0) & (rv < k.height)
            j = np.where(ok, rv, 0).astype(int) * k.width + np.where(ok, ru, 0).astype(int)
            dw = [a + f(b) for a, b in zip(rot(Rf, d[:, j]), t)]
            n = rot(Rf, nd[:, j])
            df = [a - b for a, b in zip(dw, s)]
            cs = (n[0] * m[0] + n[1] * m[1]) + n[2] * m[2]
            ok &= ~np.isnan(dw[0]) & (np.sqrt((df[0] * df[0] + df[1] * df[1]) + df[2] * df[2]) < f(dist))
            ok &= (cs > cos_gate) & (cs < f(1) + f(1e-6))
            A = np.stack([m[1] * dw[2] - m[2] * dw[1], m[2] * dw[0] - m[0] * dw[2], m[0] * dw[1] - m[1] * dw[0], *m])
            b = (m[0] * (s[0] - dw[0]) + m[1] * (s[1] - dw[1])) + m[2] * (s[2] - dw[2])
        A, b = A[:, ok].astype(np.float64), b[ok].astype(np.float64)
        x = np.linalg.solve(A @ A.T, A @ b)
        D = pose(-x[0], -x[1], -x[2], x[3:])
        T = D @ T
    return T, int(ok.sum())


@pytest.mark.parametrize("size", [(16, 16), (256, 256), (257, 256), (362, 363), (640, 512), (641, 512), (1280, 1230)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
def test_steps_at_shape_edges(gpu, kf, orc, size):
    W, H = size
    k = intr(W, H, fx=0.9 * W, fy=0.9 * W)
    T = pose(0.01, -0.015, 0.008, (0.012, -0.01, 0.02))
    live, model = kf.DeviceMaps(k, 1, True), kf.DeviceMaps(k, 1, False)
    hl, hm = orc.HostMaps(k, 1, True), orc.HostMaps(k, 1, False)
    host_maps = _maps(k, T, True), _maps(k, np.eye(4), False)
    for dev, host, (p, n) in ((live, hl, host_maps[0]), (model, hm, host_maps[1])):
        for c in range(3):
            for name, a in (("v", p), ("n", n)):
                plane = np.ascontiguousarray(a[..., c], np.float32)
                dev.set_plane(0, name + "xyz"[c], plane)
                host.set_plane(0, name + "xyz"[c], plane)
        if dev is live:
            z = np.nan_to_num(p[..., 2]).astype(np.float32)
            dev.set_plane(0, "depth", z)
            host.set_plane(0, "depth", z)
    T_ref, inliers = _track(k, *host_maps, 3, 0.1, 20.0)
    for comp in (1, 0):
        prm = icp_params(levels=1, iters=(3,), comp=comp)
        _, ost = orc.icp_track(k, prm, hl, hm, np.eye(4))
        res = []
        for single in (0, 1):
            print(f"icp {W}x{H} compensated={comp} single={single}", flush=True)
            icp = kf.ICP(k, icp_params(levels=1, iters=(3,), comp=comp, single=single))
            out = kf.DevicePose(np.eye(4))
            st = icp.Iterate_ICP(live, model, out)
            res.append((bytes(out.raw()), bytes(st)))
            assert st.status == 0 and st.iterations == 3
            assert st.candidates == ost.candidates
            if comp:  # plain mode's FP32-summed poses may put a pixel across a gate in later iterations
                assert st.inliers == ost.inliers == inliers and inliers > 0.5 * W * H
            # FP64 sums of the same rows in another order: 2^-53 relative each, times the
            # system's condition (< 1e5) and steps below 0.1; FP32 sums: 2e-4 relative
            assert np.max(np.abs(out.get() - T_ref)) < (1e-10 if comp else 1e-4)
        assert res[0] == res[1]
