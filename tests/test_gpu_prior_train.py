"""The prior's training kernels against the FP64 oracle (BF16 operand rounding emulated)
at batches where their tilings end: one sample (layer 3's 300 pixels are no multiple of
a 16-pixel tile), odd batches, one where every wave takes several tiles, and the first
where layer 2's input gradient gets more blocks than its weight gradient."""
import numpy as np
import pytest

from oracle import prior_oracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 3, 37, 137])
def test_gradients_match_oracle_at_tile_edges(gpu, kf, B):
    rng = np.random.default_rng(100 + B)
    F = B + 1
    frames = rng.uniform(0.5, 3.5, size=(F, po.H0, po.W0)).astype(np.float32)
    frames[rng.random(frames.shape) < 0.1] = 0.0
    pairs = rng.integers(0, F, size=(B, 2)).astype(np.int32)
    prev = rng.normal(0, 0.5, size=(B, 6)).astype(np.float32)
    target = rng.normal(0, 0.5, size=(B, 6)).astype(np.float32)
    df, dp, dv, dt = [kf.upload(a) for a in (frames, pairs, prev, target)]
    prior = kf.Prior(max_batch=B)
    params = po.init_params(11).astype(np.float32)
    prior.set_params(params)
    dg, dl = kf.DeviceBuffer(prior.nparams * 4), kf.DeviceBuffer(4)
    print(f"prior gradients B={B}", flush=True)
    prior.gradients(df, dp, dv, dt, B, dg, dl)
    kf.synchronize()
    g = dg.download(np.float32).astype(np.float64)
    rloss, rg = po.gradients(params.astype(np.float64), frames, pairs, prev, target, bf=True)
    # FP32 sums of products that are exact in FP32 differ from FP64 ones by ~1e-7; what
    # remains are activations and gradients that round to the other BF16 neighbour
    # (2^-8 relative, in a small share of the elements): well under 5e-3 of a layer's norm
    assert abs(float(dl.download(np.float32)[0]) - rloss) < 1e-3 * rloss
    L, _ = po.layout()
    for li, (wo, ws, bo, bl) in enumerate(L):
        for lo, hi, what in ((wo, wo + ws[0] * ws[1], "W"), (bo, bo + bl, "b")):
            a, b = g[lo:hi], rg[lo:hi]
            rel = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-12)
            assert rel < 5e-3, (li, what, rel)
    # the same call again: the sums' orders are fixed
    prior.gradients(df, dp, dv, dt, B, dg, dl)
    kf.synchronize()
    assert np.array_equal(g, dg.download(np.float32).astype(np.float64))


def test_batched_inference_equals_single_samples(gpu, kf):
    """Batches of 1 and 3 run fused, 4 and 37 layer by layer: the same MFMA sequences, so
    the same bits per sample."""
    rng = np.random.default_rng(7)
    B = 37
    frames = rng.uniform(0.5, 3.5, size=(B + 1, po.H0, po.W0)).astype(np.float32)
    pairs = rng.integers(0, B + 1, size=(B, 2)).astype(np.int32)
    prev = rng.normal(0, 0.5, size=(B, 6)).astype(np.float32)
    df, dp, dv = [kf.upload(a) for a in (frames, pairs, prev)]
    prior = kf.Prior(max_batch=B)
    prior.set_params(po.init_params(3).astype(np.float32))
    dout = kf.DeviceBuffer(B * 24)

    def run(first, n):
        print(f"prior forward {first}..{first + n - 1}", flush=True)
        prior.forward(df, dp.ptr + first * 8, dv.ptr + first * 24, n, dout)
        kf.synchronize()
        return dout.download(np.float32, n * 6).reshape(n, 6).view(np.uint32)

    single = np.concatenate([run(i, 1) for i in range(B)])
    assert np.array_equal(run(0, B), single)
    assert np.array_equal(run(5, 4), single[5:9])
    assert np.array_equal(run(11, 3), single[11:14])
    ref, _ = po.forward(po.init_params(3), frames, pairs, prev, bf=True)
    out = single.view(np.float32)
    assert np.max(np.abs(out - ref)) < 2e-3 * np.abs(ref).max()
