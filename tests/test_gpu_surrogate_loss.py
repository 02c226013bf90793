"""GPU: the loss that a training call reports."""
import numpy as np
import pytest

from bellhopcuda_amd import surrogate

pytestmark = pytest.mark.gpu


def test_no_steps_return_the_last_loss():
    """The losses of even and odd steps lie in two halves of one buffer."""
    print("\n[gpu-case] network_no_steps", flush=True)
    rng = np.random.default_rng(1)
    m = surrogate.Mlp(members=2, max_batch=256, seed=5, n_out=32, front=1)
    try:
        x = rng.random((1024, 16), dtype=np.float32)
        y = rng.normal(size=(1024, 32)).astype(np.float32)
        m.set_dataset(x, y)
        for steps in (1, 2, 5):
            last = m.train(steps, 128, 1e-3, seed=steps)
            assert np.all(last > 0) and np.array_equal(m.train(0, 128), last)
        last = m.gradients(x[:64], y[:64])[1]
        assert np.array_equal(m.train(0, 128), last)
    finally:
        m.close()
