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


def test_several_steps_follow_their_gradients():
    """Six steps over 2,200 rows (nine partial sums a weight gradient): each step's parameters are, bit for bit,
    Adam's float32 update (seven operations, none contracted) by the gradient of the parameters before it, and that
    gradient is within 3e-2 of the oracle's per tensor, as in test_gradient_and_step.  Trajectories themselves are
    not compared: adding the partial sums in another order changes gradients by float32 roundings, now and then a
    bf16 weight rounds the other way, and parameters then part by up to about 1e-4 in a few steps."""
    import ctypes

    powf = ctypes.CDLL("libm.so.6").powf
    powf.restype, powf.argtypes = ctypes.c_float, [ctypes.c_float, ctypes.c_float]
    f = np.float32
    rows, lr, b1, b2, eps = 2200, f(1e-3), f(0.9), f(0.999), f(1e-8)
    rng = np.random.default_rng(3)
    net = ClosureNet(max_batch=rows, seed=8)
    p = net.params()
    m, v = np.zeros_like(p), np.zeros_like(p)
    Lo = MO.layout()
    for t in range(1, 7):
        print(f"case step {t}", flush=True)
        x = np.zeros((rows, 208), np.float32)
        x[:, :195] = rng.normal(0, 1, (rows, 195))
        xb = (x.view(np.uint32) >> 16).astype(np.uint16)
        y = np.zeros((rows, 4), np.float32)
        y[:, :3] = rng.normal(0, 1, (rows, 3))
        xd, yd = DeviceArray(xb.shape, np.uint16).upload(xb), DeviceArray(y.shape, np.float32).upload(y)
        g, _ = net.gradient(xd, yd, rows)
        _, _, ref = MO.forward_backward(p.astype(np.float64), MO.bf16_bits_to_f64(xb), y[:, :3], bf16=True)
        for k in ("w1", "b1", "w2", "b2", "w3", "b3", "w4", "b4"):
            a, b = (q[Lo[k][0]:Lo[k][0] + Lo[k][1]] for q in (g, ref))
            assert np.linalg.norm(a - b) < 3e-2 * np.linalg.norm(b), (t, k)
        net.train_step(xd.ptr, yd.ptr, rows, float(lr))
        m = b1 * m + (f(1) - b1) * g
        v = b2 * v + (f(1) - b2) * g * g
        c1, c2 = f(1) - f(powf(b1, t)), f(1) - f(powf(b2, t))
        p = p - lr * (m / c1) / (np.sqrt(v / c2) + eps)
        got = net.params()
        assert p.dtype == np.float32
        assert np.array_equal(got.view(np.uint32), p.view(np.uint32)), f"step {t}: {(got != p).sum()} parameters"
