"""The prior's batch sizes: inference on both sides of the line between its fused and its
layered form (five and six samples)."""
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
