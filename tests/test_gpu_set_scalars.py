"""The heating totals set right after a step, whose last folds may still be on
their way to the pinned mirror of the totals: what is set is what is read, and what
the next step adds to."""
import ctypes as C

import pytest

from lare3d_amd import configs
from lare3d_amd.abi import LareScalars, check

pytestmark = pytest.mark.gpu


def test_totals_set_behind_a_step():
    from lare3d_amd.device import Device
    grid, params, f = configs.harris(64)
    print("\n[case] heating totals set behind a step", flush=True)
    dev = Device(grid, params, f)
    dev.boundary_conditions()
    dev.eta_calc()
    dev.step(1)
    s = dev.scalars()
    for q in range(2, 22):
        dev.step(q)
        s.total_visc_heating, s.total_ohmic_heating = 1000.0 * q, -1000.0 * q
        check(dev.lib, dev.lib.lare_dev_set_scalars(C.byref(s)), "set_scalars")
        got = LareScalars()
        check(dev.lib, dev.lib.lare_dev_get_scalars(C.byref(got)), "get_scalars")
        assert (got.total_visc_heating, got.total_ohmic_heating) == (1000.0 * q, -1000.0 * q)
    i = dev.step_info(22)
    assert 21000.0 < i.total_visc_heating < 21001.0 and -21000.0 < i.total_ohmic_heating < -20999.0
    dev.close()
