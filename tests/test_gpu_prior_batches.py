"""The prior's batch sizes: inference on both sides of the line between its fused and its
layered form (five and six samples), gradients on one handle at batches that change."""
import numpy as np
import pytest

from oracle import prior_oracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 5, 6, 7])
def test_inference_where_the_form_changes(gpu, kf, n):
    rng = np.random.default_rng(70 + n)
    frames = rng.uniform(0.5, 3.5, size=(n + 1, po.H0, po.W0)).astype(np.float32)
    pairs = rng.integers(0, n + 1, size=(n, 2)).astype(np.int32)
    prev = rng.normal(0, 0.5, size=(n, 6)).astype(np.float32)
    df, dp, dv = [kf.upload(a) for a in (frames, pairs, prev)]
    prior = kf.Prior(max_batch=n)
    prior.set_params(po.init_params(3).astype(np.float32))
    dout = kf.DeviceBuffer(n * 24)

    def run(first, count):
        prior.forward(df, dp.ptr + first * 8, dv.ptr + first * 24, count, dout)
        kf.synchronize()
        return dout.download(np.uint32, count * 6).reshape(count, 6)

    single = np.concatenate([run(i, 1) for i in range(n)])  # one sample is always fused
    for _ in range(2):
        assert np.array_equal(run(0, n), single)


def test_gradients_on_one_handle_at_changing_batches(gpu, kf):
    """A handle keeps its partial planes from call to call, and how many of them a call makes
    depends on its batch: a smaller batch after a larger one gives what a fresh handle gives."""
    rng = np.random.default_rng(9)
    most = 137
    frames = rng.uniform(0.5, 3.5, size=(most + 1, po.H0, po.W0)).astype(np.float32)
    pairs = np.stack([np.arange(most), np.arange(most) + 1], -1).astype(np.int32)
    prev, target = rng.normal(0, 0.5, size=(2, most, 6)).astype(np.float32)
    df, dp, dv, dt = [kf.upload(a) for a in (frames, pairs, prev, target)]
    params = po.init_params(11).astype(np.float32)

    def handle(batch):
        prior = kf.Prior(max_batch=batch)
        prior.set_params(params)
        return prior

    def gradients(prior, n):
        print(f"prior gradients B={n}", flush=True)
        dg, dl = kf.DeviceBuffer(prior.nparams * 4), kf.DeviceBuffer(4)
        prior.gradients(df, dp, dv, dt, n, dg, dl)
        kf.synchronize()
        return dg.download(np.uint32), dl.download(np.uint32)

    kept = handle(most)
    for n in (most, 3, 37, 1, most):
        got, want = gradients(kept, n), gradients(handle(n), n)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), n
