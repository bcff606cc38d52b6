"""Upload and download: every element of every array comes back as it went
(rounded once to FP32 where the FP32 mode stores it so), for one launch, for
several chunks in one thread, and for several threads with a ragged last
chunk; and a second state on the same Device."""
import numpy as np
import pytest

from lare3d_amd import BC_USER, configs
from lare3d_amd.abi import PREC_FP32
from lare3d_amd.fields import NAMES, Fields
from lare3d_amd.grid import Grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(4, 5, 6), (33, 30, 35), (70, 61, 67)])
@pytest.mark.parametrize("precision", [0, PREC_FP32])
def test_round_trip(n, precision):
    from lare3d_amd.device import Device
    grid = Grid(*n, ((0.0, 1.0),) * 3, (BC_USER,) * 6)
    params = configs.default_params(precision=precision)
    rng = np.random.default_rng(5)
    states = []
    for _ in range(2):
        f = Fields(*n)
        for name in NAMES:
            a = getattr(f, name)
            a[...] = rng.standard_normal(a.shape)
        states.append(f)
    print(f"\n[case] transfer n={n} precision={precision}", flush=True)
    dev = Device(grid, params, states[0])
    for q, f in enumerate(states):
        if q:
            dev.upload(f)
        back = dev.fields()
        for name in NAMES:
            if name == "visc3":  # an input only
                continue
            want = getattr(f, name)
            if precision == PREC_FP32 and name not in ("bx", "by", "bz"):
                want = want.astype(np.float32).astype(np.float64)
            assert np.array_equal(getattr(back, name), want), name
    dev.close()
