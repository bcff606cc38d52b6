"""Training steps of the surrogate: the rows drawn by hash and the Adam update,
for batches of one tile, of one staged chunk of 512 columns and one tile more, and
of two chunks.  Gradient and loss of the drawn rows are those of sur.grad on the
same rows (compared with the restatement in test_gpu_surrogate_batch.py): the
kernel is the same and so are the operands.  The update is Adam in FP32: a handful
of roundings, each at most 2^-24 of what the terms of m would make without their
signs, those of the powers of beta in 1 - beta^t, and one of the parameter."""
import numpy as np
import pytest

from lare3d_amd import configs
from oracle import surrogate_ref as ref

pytestmark = pytest.mark.gpu
M64 = (1 << 64) - 1


@pytest.mark.parametrize("batch", [16, 512, 528, 1024])
def test_drawn_rows_and_update(batch):
    from lare3d_amd.device import Device
    from lare3d_amd.surrogate import Surrogate
    grid, params, f, dt = configs.harris_conduction(16, seed=1, s_target=5)
    dev = Device(grid, params, f)
    dev.boundary_conditions()
    dev.set_scalars(dt=dt)
    sur = Surrogate(dev)
    w = ref.init_params(5)
    sur.set_params(w)
    rows = sur.collect(700, 77)
    sur.fit_norm()
    X, y = sur.rows(rows)
    f32 = np.float32
    lr, b1, b2, eps = f32(1e-3), f32(0.9), f32(0.999), f32(1e-8)
    m, v, size = np.zeros_like(w), np.zeros_like(w), np.zeros_like(w)
    for step, seed in enumerate((9, 10, 2 ** 40 + 1), 1):
        print(f"\n[case] surrogate training batch={batch} seed={seed}", flush=True)
        h = ref.mix64(seed * 0x9E3779B97F4A7C15 & M64)
        r = [ref.mix64(h + b & M64) % rows for b in range(batch)]
        g, loss = sur.grad(X[r], y[r])
        hist = sur.train(1, batch=batch, lr=float(lr), seed=seed)
        assert abs(hist[0] - loss) <= 8 * 2.0 ** -24 * loss
        m = b1 * m + (f32(1) - b1) * g
        v = b2 * v + (f32(1) - b2) * g * g
        size = b1 * size + (f32(1) - b1) * np.abs(g)
        c1, c2 = f32(1) - f32(b1 ** f32(step)), f32(1) - f32(b2 ** f32(step))
        update = lr * (m / c1) / (np.sqrt(v / c2) + eps)
        got = sur.params()
        largest = lr * (size / c1) / (np.sqrt(v / c2) + eps)
        tol = (16 + 2 / c1 + 2 / c2) * 2.0 ** -24 * largest + 2.0 ** -23 * np.abs(w)
        assert np.all(np.abs(got - (w - update)) <= tol)
        assert np.abs(update).max() > 0.5 * lr
        w = got
    dev.close()
