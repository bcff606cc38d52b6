"""The inverted temperature bracket of neutral_fraction reported by a whole step,
whose fault flag is read after the step's last fold and not at the end of the
stream: once for a faulty state, and not for the good one that follows."""
import pytest

from lare3d_amd import configs
from lare3d_amd.abi import DeviceError, EOS_ION, EOS_PI, F_TBOUNDS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eos", [EOS_PI, EOS_ION])
@pytest.mark.parametrize("cell", [(2, 2, 2), (20, 11, 30), (49, 40, 37)])
def test_step_reports_the_bracket_once(eos, cell):
    from lare3d_amd.device import Device
    cfg = configs.harris(48, ny=40, nz=36)
    configs.partially_ionised(cfg, eos, 1)
    grid, params, f = cfg
    good = f.energy.copy()
    print(f"\n[case] inverted bracket eos={eos} cell={cell}", flush=True)
    dev = Device(grid, params, f)
    for e in (None, 0.0, None):
        f.energy[...] = good
        if e is not None:
            f.energy[cell] = e
        dev.upload(f)
        dev.set_scalars(dt=0.0, time=0.0, first_set_dt=1, step=0)
        dev.boundary_conditions()
        dev.eta_calc()
        if e is None:
            assert dev.step(1)[0] > 0.0
        else:
            with pytest.raises(DeviceError) as err:
                dev.step(1)
            assert err.value.code == F_TBOUNDS, err.value
    dev.close()
