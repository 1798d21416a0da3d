"""The single-launch form of tracking where a block makes several of a level's slots, and
several such calls at once: 320x240 takes 50 blocks, so four calls on streams of their own fit
the chip together.  Poses and statistics equal the multi-launch form's, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from tests.helpers import icp_params, intr, pose
from tests.test_gpu_icp_shapes import _maps

pytestmark = pytest.mark.gpu

CALLS, ROUNDS = 4, 8


def _device_maps(kf, k, levels):
    T = pose(0.01, -0.015, 0.008, (0.012, -0.01, 0.02))
    live, model = kf.DeviceMaps(k, levels, True), kf.DeviceMaps(k, levels, False)
    for l in range(levels):
        kl = intr(k.width >> l, k.height >> l, fx=k.fx / (1 << l), fy=k.fy / (1 << l))
        for dev, (p, n) in ((live, _maps(kl, T, True)), (model, _maps(kl, np.eye(4), False))):
            for c in range(3):
                dev.set_plane(l, "v" + "xyz"[c], np.ascontiguousarray(p[..., c], np.float32))
                dev.set_plane(l, "n" + "xyz"[c], np.ascontiguousarray(n[..., c], np.float32))
    return live, model


def _track(kf, icp, live, model, out, stream=None):
    kf.check(kf.lib().kf_icp_track(icp.handle, C.byref(live.maps), C.byref(model.maps), out.ptr, out.ptr,
                                   icp.stats.ptr, stream), "track")


def _result(kf, icp, out):
    return bytes(out.raw()), bytes(icp.stats.download(np.uint8, C.sizeof(kf.IcpStats)))


@pytest.mark.parametrize("size", [(93, 71), (200, 160), (320, 240), (443, 443), (444, 444)], ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("comp", [1, 0])
def test_single_launch_slots(gpu, kf, size, comp):
    k = intr(*size, fx=0.9 * size[0], fy=0.9 * size[0])
    live, model = _device_maps(kf, k, 3)
    res = []
    for single in (0, 1):
        icp, out = kf.ICP(k, icp_params(iters=(4, 3, 2), comp=comp, single=single)), kf.DevicePose(np.eye(4))
        _track(kf, icp, live, model, out)
        kf.synchronize()
        res.append(_result(kf, icp, out))
    st = kf.IcpStats.from_buffer_copy(res[0][1])
    assert st.status == 0 and st.iterations == 9
    assert res[0] == res[1]


def test_single_launch_calls_on_several_streams(gpu, kf):
    k = intr(320, 240, fx=288.0, fy=288.0)
    live, model = _device_maps(kf, k, 3)
    ref, out = kf.ICP(k, icp_params(single=0)), kf.DevicePose(np.eye(4))
    for _ in range(ROUNDS):
        _track(kf, ref, live, model, out)
    kf.synchronize()
    want = _result(kf, ref, out)
    streams, calls = [C.c_void_p() for _ in range(CALLS)], []
    for s in streams:
        kf.check(kf.lib().kf_stream_create(C.byref(s)), "stream")
        calls.append((kf.ICP(k, icp_params(single=1)), kf.DevicePose(np.eye(4)), s))
    kf.synchronize()
    for _ in range(ROUNDS):
        for icp, o, s in calls:
            _track(kf, icp, live, model, o, s)
    kf.synchronize()
    for icp, o, _ in calls:
        assert _result(kf, icp, o) == want
    for s in streams:
        kf.check(kf.lib().kf_stream_destroy(s), "stream")
