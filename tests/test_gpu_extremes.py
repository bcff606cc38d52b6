"""Infinities given to the diagnostics and quantities that leave the range of the
type, against the CPU restatement.  What is compared is whether a value is
infinite, so equality is exact."""
import numpy as np
import pytest

from lare3d_amd import configs
from tests.test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("field,value", [("bx", np.inf), ("by", -np.inf), ("bz", 1.7e308), ("rho", np.inf)])
def test_infinite_diagnostics(field, value):
    print(f"\n[case] diagnostics of {field} = {value}", flush=True)
    grid, params, f = configs.orszag_tang(12)
    getattr(f, field)[5, 6, 7] = value
    if field == "bz":  # finite, and so is the next face: their difference overflows
        f.bz[5, 6, 8] = -value
    from lare3d_amd.device import Device
    from oracle.oracle import Oracle
    orc = Oracle(grid, params, f)
    want, wdiv = orc.energy_account(), orc.divb()
    orc.close()
    assert np.isinf(wdiv) or field == "rho"
    dev = Device(grid, params, f)
    en, divb = dev.energy_account(with_divb=True)
    dev.close()
    for got in ((en, divb), _noalloc(grid, f)):
        assert [np.isinf(x) for x in got[0]] == [np.isinf(x) for x in want]
        assert not np.isnan(got[0]).any()
        assert np.isinf(got[1]) == np.isinf(wdiv)
