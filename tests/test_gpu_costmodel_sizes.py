"""The cost model's matrix-core kernels against the float64 oracle where their tiles end: 16
samples a wavefront, 64 a chunk, 512 chunks before a workgroup takes a second one; minibatches
that leave a remainder. The tolerances are fp32 rounding over the longest chains: 2^-24 times
a few sums of 64 terms, 1e-5, and a factor of 10."""
import numpy as np
import pytest

from oracle import mlp as omlp

pytestmark = pytest.mark.gpu


def data(seed, n):
    rng = np.random.default_rng(seed)
    x = rng.uniform(0, 8, (n, 7)).astype(np.float32)
    return x, rng.uniform(0, 9, n).astype(np.float32)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 3071, 3073, 50000])
def test_forward_sizes(dqc, n):
    p = dqc.mlp_init(3)
    x, _ = data(n, n)
    ref = omlp.forward(p.astype(np.float64), x.astype(np.float64))
    assert np.max(np.abs(dqc.mlp_forward(p, x) - ref)) <= 1e-4 * max(1.0, float(np.max(np.abs(ref))))


@pytest.mark.parametrize("n", [1, 16, 17, 63, 64, 65, 129, 512 * 64, 512 * 64 + 1])
def test_gradient_sizes(dqc, n):
    p = dqc.mlp_init(4)
    p += np.float32(0.01)  # biases away from zero
    x, t = data(100 + n, n)
    g, loss = dqc.mlp_gradient(p, x, t)
    rloss, rg = omlp.loss_and_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64))
    assert abs(loss - rloss) <= 1e-4 * abs(rloss)
    o = 0
    for name, size in omlp.SIZES:
        a, b = g[o:o + size], rg[o:o + size]
        assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b) + 1e-6, name
        o += size


@pytest.mark.parametrize("n,batch", [(65, 64), (1000, 100), (130, 1000)])
def test_training_equals_steps_of_the_gradient(dqc, n, batch):
    """One epoch with no shuffle to matter (the batch holds everything, or the first Adam step is
    compared): after the first step every parameter moved by lr against its gradient's sign."""
    x, t = data(n, n)
    p0 = dqc.mlp_init(5)
    p0 += np.float32(0.01)
    if batch < n:
        a, _ = dqc.mlp_train(p0, x, t, epochs=1, batch=batch, lr=1e-3, seed=3)
        b, _ = dqc.mlp_train(p0, x, t, epochs=1, batch=batch, lr=1e-3, seed=3)
        assert np.array_equal(a, b) and np.all(np.isfinite(a))  # deterministic
        return
    g = omlp.loss_and_grad(p0.astype(np.float64), x.astype(np.float64), t.astype(np.float64))[1]
    p1, loss = dqc.mlp_train(p0, x, t, epochs=1, batch=batch, lr=1e-3, seed=3)
    clear = np.abs(g) > 1e-3 * np.max(np.abs(g))
    assert np.allclose((p1 - p0)[clear], -1e-3 * np.sign(g)[clear], rtol=1e-2)
    ref = omlp.loss_and_grad(p1.astype(np.float64), x.astype(np.float64), t.astype(np.float64))[0]
    assert abs(loss - ref) <= 1e-4 * ref
