"""Steps of a grid whose sweeps are launches of their own, in the Strang orders
that end on y and on z (test_gpu_chunks.py: on x), against the CPU restatement:
every element of every state array.  The last sweep forms cv2 from the widths, the
others read it, in a kernel of its own for each axis."""
import numpy as np
import pytest

from lare3d_amd import configs
from tests.util import STATE

pytestmark = pytest.mark.gpu


def test_orders_that_end_on_y_and_z():
    from lare3d_amd.device import Device
    from oracle.oracle import Oracle
    # above 4096 blocks in every sweep, with few cells for the CPU
    grid, params, f = configs.harris(56, ny=260, nz=300)
    dev, orc = Device(grid, params, f), Oracle(grid, params, f)
    for d in (dev, orc):
        d.boundary_conditions()
        d.eta_calc()
    dev.profile(True)
    for step in (3, 5):  # x z y, y x z
        print(f"\n[case] sweeps apart 56x260x300 step={step}", flush=True)
        assert dev.step(step) == orc.step(step)
        names = dev.kernel_stats()
        assert "mom_remap" in names and "ct_sweep" in names and "mom_ct" not in names
        fd, fo = dev.fields(), orc.fields()
        for name in STATE:
            assert np.array_equal(getattr(fd, name), getattr(fo, name)), (step, name)
    dev.close()
    orc.close()
