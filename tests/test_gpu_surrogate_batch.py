"""Forward and gradient of the surrogate at the edges of the batch kernels: one
row, one column tile and one row more, a loss block of 256 columns and one
more, the 512 columns that a product stages at once and one tile more; against
the restatement with BF16 operands.  Its bounds are those of the batch test in
test_surrogate.py: BF16 operands rounded from FP32 sums in another order."""
import numpy as np
import pytest

from lare3d_amd import configs
from oracle import surrogate_ref as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 16, 17, 256, 257, 511, 513, 1040])
def test_forward_and_gradient(rows):
    from lare3d_amd.device import Device
    from lare3d_amd.surrogate import Surrogate
    grid, params, f, dt = configs.harris_conduction(8, seed=1)
    dev = Device(grid, params, f)
    sur = Surrogate(dev)
    rng = np.random.default_rng(rows)
    w = ref.init_params(5)
    w[ref.OFF_B1:ref.OFF_W2] = (0.1 * rng.standard_normal(ref.H)).astype(np.float32)
    sur.set_params(w)
    print(f"\n[case] surrogate batch rows={rows}", flush=True)
    X = rng.standard_normal((rows, ref.K)).astype(np.float32)
    X[:, ref.KREAL:] = 0.0
    t = rng.standard_normal(rows).astype(np.float32)
    y, yo = sur.forward(X), ref.forward(w, X, emulate_bf16=True)
    assert np.max(np.abs(y - yo)) <= 2e-3 * np.max(np.abs(yo))
    g, loss = sur.grad(X, t)
    go, losso = ref.backward(w, X, t, emulate_bf16=True)
    assert abs(loss - losso) <= 2e-3 * losso
    for a, b in ((ref.OFF_W1, ref.OFF_B1), (ref.OFF_B1, ref.OFF_W2), (ref.OFF_W2, ref.OFF_B2),
                 (ref.OFF_B2, ref.OFF_W3), (ref.OFF_W3, ref.OFF_B3), (ref.OFF_B3, ref.NPARAM)):
        assert np.linalg.norm(g[a:b] - go[a:b]) <= 2e-2 * np.linalg.norm(go[a:b])
    dev.close()
