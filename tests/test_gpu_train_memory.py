"""Device memory that a network holds after training: no more than the room of a million
rows (112 bytes each) beyond a minibatch's, and what it held for its inference calls."""
import ctypes as C
import time

import numpy as np
import pytest

import xpbd_amd as X

pytestmark = pytest.mark.gpu
ROWS = 2_000_000
KEEP = (1 << 20) * 112


def _free(at_least=0):
    """Free device memory, some seconds later at most where memory that was freed is on its way back."""
    free, total = C.c_size_t(), C.c_size_t()
    for _ in range(50):
        # from the runtime that the library runs on
        assert X.lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        if free.value >= at_least:
            break
        time.sleep(0.1)
    return free.value


def test_training_gives_large_inputs_back():
    rng = np.random.default_rng(0)
    x = rng.standard_normal((ROWS, X.MLP_IN), dtype=np.float32)
    y = np.tanh(x[:, :3])
    net = X.Network((0.1 * rng.standard_normal(X.MLP_PARAMS)).astype(np.float32))
    net.set_scaling(np.zeros(X.MLP_IN), np.ones(X.MLP_IN), 1.0)
    net.train(x[:5000], y[:5000], batch=4096, epochs=1, lr=1e-4, seed=1)   # a minibatch's room is kept
    small = net.forward(x[:3000])
    before = _free()
    net.train(x, y, batch=4096, epochs=1, lr=1e-12, seed=1)
    assert _free(before - KEEP) >= before - KEEP
    # calls of every size, in the order that grows and shares the buffers, still agree
    a = net.forward(x[:3000])
    np.testing.assert_allclose(a, small, rtol=0, atol=1e-6)   # 488 steps of 1e-12
    big = net.forward(x[:400_000])
    np.testing.assert_array_equal(big[:3000], a)
    loss, _ = net.loss_grad(x[:30_000], y[:30_000])
    net.train(x[:100], y[:100], batch=64, epochs=1, lr=1e-12, seed=1)
    assert net.forward(x[:400_000]).shape == big.shape
    assert np.isfinite(loss)
    before = _free()
    net.train(x, y, batch=4096, epochs=1, lr=1e-12, seed=2)
    assert _free(before - KEEP) >= before - KEEP
