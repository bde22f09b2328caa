"""One training step at the edges of its tiles, row chunks and splits, against the float64 oracle."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO
from watercube_amd.closure import ClosureNet, DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 1023, 1025, 16500])
def test_gradient_and_step(rows):
    """Gradients within 3e-2 of the oracle's per tensor: four layers, each with activations and deltas rounded
    to bf16 (2^-9), of which a single row averages nothing.  The step is Adam's first one from those gradients,
    to the roundings of its seven float32 operations and the parameter's own; the fused inference, which reads
    the transposed bf16 weights, then agrees with the training forward, which reads the others."""
    print(f"case rows={rows}", flush=True)
    rng = np.random.default_rng(rows)
    net = ClosureNet(max_batch=rows, seed=5)
    p = net.params()
    Lo = MO.layout()
    for k in ("b1", "b2", "b3"):
        p[Lo[k][0]:Lo[k][0] + 128] = rng.normal(0, 0.1, 128)
    p[Lo["b4"][0]:Lo["b4"][0] + 3] = rng.normal(0, 0.1, 3)
    net.set_params(p)
    x = np.zeros((rows, 208), np.float32)
    x[:, :195] = rng.normal(0, 1, (rows, 195))
    xb = (x.view(np.uint32) >> 16).astype(np.uint16)  # bf16, truncated
    t = np.zeros((rows, 4), np.float32)
    t[:, :3] = rng.normal(0, 1, (rows, 3))
    xd, td = DeviceArray(xb.shape, np.uint16).upload(xb), DeviceArray(t.shape, np.float32).upload(t)
    _, loss_ref, g_ref = MO.forward_backward(p.astype(np.float64), MO.bf16_bits_to_f64(xb), t[:, :3], bf16=True)
    g, loss = net.gradient(xd, td, rows)
    assert abs(loss - loss_ref) / loss_ref < 1e-2
    for k in ("w1", "b1", "w2", "b2", "w3", "b3", "w4", "b4"):
        a, b = (v[Lo[k][0]:Lo[k][0] + Lo[k][1]] for v in (g, g_ref))
        assert np.linalg.norm(a - b) < 3e-2 * np.linalg.norm(b), k
    again, _ = net.gradient(xd, td, rows)
    assert np.array_equal(g, again)  # sums are taken in a fixed order
    lr = 1e-3
    net.train_step(xd.ptr, td.ptr, rows, lr)
    g = g.astype(np.float64)
    big = np.abs(g) > 1e-15  # g * g stays a normal float32
    want = p - lr * g / (np.abs(g) + 1e-8)
    got = net.params()
    assert np.all(np.abs(got - want)[big] <= 2e-6 * lr + 2.0 ** -23 * np.abs(p[big]))
    assert np.array_equal(got[g == 0], p[g == 0])
    ya, yb = DeviceArray((rows, 4), np.float32), DeviceArray((rows, 4), np.float32)
    net.forward(xd, ya, rows)
    net.predict(xd, yb, rows)
    a, b = ya.download()[:, :3], yb.download()[:, :3]
    assert np.linalg.norm(a - b) < 2e-2 * np.linalg.norm(b)
