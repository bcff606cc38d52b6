"""The one-launch boundary fill against the CPU restatement's pass per axis,
every element of every state array, on the smallest grid (n = 4, where the
layers of both sides are closest), odd unequal sizes and every kind of side.
The fill copies values, so equality is exact."""
import numpy as np
import pytest

from lare3d_amd import BC_OPEN, BC_PERIODIC, BC_USER, configs
from lare3d_amd.abi import PREC_FP32
from lare3d_amd.fields import Fields
from lare3d_amd.grid import Grid
from tests.util import STATE

pytestmark = pytest.mark.gpu

P, U, O = BC_PERIODIC, BC_USER, BC_OPEN


@pytest.mark.parametrize("n", [(4, 4, 4), (5, 4, 7), (67, 9, 4), (4, 31, 66)])
@pytest.mark.parametrize("bcs", [(P,) * 6, (U,) * 6, (U, U, P, P, U, U), (P, P, U, U, P, P), (O, U, P, P, U, O),
                                 (U, U, O, O, P, P), (O,) * 6])
@pytest.mark.parametrize("precision", [0, PREC_FP32])
def test_fill_every_kind_of_side(n, bcs, precision):
    from lare3d_amd.device import Device
    from oracle.oracle import Oracle
    if precision == PREC_FP32 and O in bcs:
        pytest.skip("BC_OPEN runs in the FP64 mode only")
    grid = Grid(*n, ((0.0, 1.0),) * 3, bcs)
    params = configs.default_params()
    f = Fields(*n)
    rng = np.random.default_rng(3)
    for name in STATE:
        a = getattr(f, name)
        # values that FP32 storage holds exactly
        a[...] = rng.integers(-1000, 1000, a.shape).astype(np.float64)
    orc = Oracle(grid, params, f)
    params.precision = precision
    dev = Device(grid, params, f)
    print(f"\n[case] fill n={n} bcs={bcs} precision={precision}", flush=True)
    dev.boundary_conditions()
    orc.boundary_conditions()
    fd, fo = dev.fields(), orc.fields()
    for name in STATE:
        assert np.array_equal(getattr(fd, name), getattr(fo, name)), name
    dev.close()
    orc.close()
