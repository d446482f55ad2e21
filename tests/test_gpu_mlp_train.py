"""Training steps in one kernel (batches of up to 64 rows) against the same steps taken one by
one: the gradient from its own entry point and Adam in float32 on the host.  The kernel keeps
every product, sum and update in the same order, so the parameters are equal bit for bit.
Batches around the 16-row tile and the 32-row product step, both staging buffers more than
once (64 steps each), and the first batch size past the kernel's limit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _shuffled(rows, batch, epochs, seed):
    order, st = list(range(rows)), (seed + 0x9E3779B97F4A7C15) % 2 ** 64
    for _ in range(epochs):
        for i in range(rows - 1, 0, -1):
            st = (st * 6364136223846793005 + 1442695040888963407) % 2 ** 64
            j = (st >> 33) % (i + 1)
            order[i], order[j] = order[j], order[i]
        for b0 in range(0, rows - batch + 1, batch):
            yield order[b0:b0 + batch]


@pytest.mark.parametrize("rows,batch,epochs", [(70, 1, 3), (31, 15, 2), (48, 16, 2), (40, 17, 2), (100, 32, 2), (97, 48, 2),
                                               (64, 64, 2), (130, 64, 2), (131, 65, 2)])
def test_steps_equal_single_products(lee, rows, batch, epochs):
    rng = np.random.default_rng(rows * 100 + batch)
    x = rng.uniform(-1, 1, (rows, 4)).astype(np.float32)
    t = (0.5 + 0.4 * np.tanh(x @ rng.normal(size=(4, 8)))).astype(np.float32)
    f = np.float32
    one, b1, b2, eps, lr = f(1), f(0.9), f(0.999), f(1e-8), f(2e-3)
    a, b = lee.ground.Network(seed=4), lee.ground.Network(seed=4)
    mse = a.train(x, t, batch=batch, epochs=epochs, lr=2e-3, seed=7)
    w = b.params()
    m, v = np.zeros_like(w), np.zeros_like(w)
    for step, pick in enumerate(_shuffled(rows, batch, epochs, 7), 1):
        g, ref = b.gradient(x[pick], t[pick])
        c1, c2 = one - f(float(b1) ** step), one - f(float(b2) ** step)
        m = b1 * m + (one - b1) * g
        v = b2 * v + (one - b2) * g * g
        w = w - lr * (m / c1) / (np.sqrt(v / c2) + eps)
        b.set_params(w)
    got = a.params()
    print(f"[gpu train] rows={rows} batch={batch}: {step} steps, max diff {np.abs(got - w).max():.1e}", flush=True)
    a.close()
    b.close()
    assert mse == ref
    assert np.array_equal(got, w)
