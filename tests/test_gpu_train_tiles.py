"""The training kernels at the edges of their tiles of 32 rows and of their runs of
rows (split from 256 rows on, longer past 4,096), against the oracle with the
same BF16 rounding of the products' operands.

A hidden value whose FP32 rounding differs by an ulp may round to another BF16
number (2^-9 relative) in a few of thousands of terms of a sum: 1e-2 in the norm
of a parameter block's gradient, as for the gradient's own test, is far above
that.  Adam divides by the gradient's size, so elements whose gradient is within
that error of zero may move the other way: 1% of a block's elements at most, 2 per
element of the unit step, which leaves the angle's cosine above 0.98."""
import numpy as np
import pytest

import mlp_oracle as M
import xpbd_amd as X

pytestmark = pytest.mark.gpu


def _data(n, seed):
    rng = np.random.default_rng(seed)
    p = np.concatenate([rng.normal(0, np.sqrt(1.0 / s[-1]) if len(s) > 1 else 0.1, s).ravel() for _, s in M.SIZES]).astype(np.float32)
    mean, std = rng.normal(size=M.N_IN).astype(np.float32), rng.uniform(0.5, 2, M.N_IN).astype(np.float32)
    x = (mean + std * rng.normal(size=(n, M.N_IN))).astype(np.float32)
    return p, x, rng.normal(size=(n, 3)).astype(np.float32), mean, std


def _blocks(g):
    at = np.cumsum([0] + [int(np.prod(s)) for _, s in M.SIZES])
    return {name: np.asarray(g[a:b], np.float64) for (name, _), a, b in zip(M.SIZES, at, at[1:])}


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 255, 256, 257, 1000, 4096, 4097, 8192, 8193, 20000])
def test_gradient(n):
    p, x, t, mean, std = _data(n, n)
    net = X.Network(p)
    net.set_scaling(mean, std, 0.7)
    loss, g = net.loss_grad(x, t)
    le, ge = M.loss_grad(p, x, t, mean, std, np.float32(0.7), emulate_bf16=True)
    assert abs(loss - le) <= 1e-3 * le
    for (name, a), b in zip(_blocks(g).items(), _blocks(ge).values()):
        err = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        print(f"n={n} {name}: {err:.2e}")
        assert err <= 1e-2
    again = net.loss_grad(x, t)
    assert again[0] == loss
    np.testing.assert_array_equal(again[1], g)
    # the gradient of a smaller call after a larger one has nothing of it left
    if n > 1:
        l1, g1 = net.loss_grad(x[:n // 2], t[:n // 2])
        other = X.Network(p)
        other.set_scaling(mean, std, 0.7)
        l2, g2 = other.loss_grad(x[:n // 2], t[:n // 2])
        assert l1 == l2
        np.testing.assert_array_equal(g1, g2)


@pytest.mark.parametrize("n", [32, 1000, 8200])
def test_full_batch_steps(n):
    p, x, t, mean, std = _data(n, n + 1)
    lr, steps = 1e-3, 4
    nets = [X.Network(p), X.Network(p)]
    for net in nets:
        net.set_scaling(mean, std, 1.3)
        net.train(x, t, batch=n, epochs=steps, lr=lr, seed=2)
    np.testing.assert_array_equal(nets[0].params(), nets[1].params())
    q, m, v = p.astype(np.float64), 0.0, 0.0
    for k in range(1, steps + 1):
        g = M.loss_grad(q.astype(np.float32), x, t, mean, std, np.float32(1.3), emulate_bf16=True)[1].astype(np.float64)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        q = q - lr * (m / (1 - 0.9 ** k)) / (np.sqrt(v / (1 - 0.999 ** k)) + 1e-8)
    for (name, a), b, c in zip(_blocks(nets[0].params()).items(), _blocks(q).values(), _blocks(p).values()):
        cos = (a - c) @ (b - c) / max(np.linalg.norm(a - c) * np.linalg.norm(b - c), 1e-30)
        print(f"n={n} {name}: cosine of the steps {cos:.5f}, length {np.linalg.norm(a - c) / np.linalg.norm(b - c):.4f}")
        assert cos >= 0.98
    # inference sees the trained weights
    y = nets[0].forward(x[:64])
    fresh = X.Network(nets[0].params())
    fresh.set_scaling(mean, std, 1.3)
    np.testing.assert_array_equal(y, fresh.forward(x[:64]))


@pytest.mark.parametrize("n,batch", [(100, 32), (2500, 1000), (5000, 4096)])
def test_minibatches_of_odd_sizes(n, batch):
    """A minibatch past the samples' end starts over; the loss falls as with a plain loop."""
    p, x, _, mean, std = _data(n, 3)
    t = np.tanh(((x - mean) / std) @ np.random.default_rng(4).normal(size=(M.N_IN, 3)) / 5).astype(np.float32)
    net = X.Network(p)
    net.set_scaling(mean, std, 1.0)
    before = net.loss_grad(x, t)[0]
    net.train(x, t, batch=batch, epochs=30, lr=2e-3, seed=1)
    after = net.loss_grad(x, t)[0]
    print(f"{n} rows by {batch}: loss {before:.4f} -> {after:.4f}")
    assert after < 0.5 * before
