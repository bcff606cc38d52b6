"""Full steps against the CPU restatement on grids for which the marching
kernels take chunks of 1, 2 and 4 points (chunks of 8: the 128^3 test of
test_gpu_parity.py), with sizes that leave a last chunk of one point:
every element of every state array, as in test_gpu_parity.py.  Resistive
with conduction, so that the RKL2 stages and the resistive tiles are in."""
import numpy as np
import pytest

from lare3d_amd import configs
from tests.util import STATE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,damping", [((4, 4, 4), None), ((9, 5, 12), 0.05), ((64, 59, 62), None), ((95, 97, 92), None)])
def test_steps_at_every_chunk(n, damping):
    from lare3d_amd.device import Device
    from oracle.oracle import Oracle
    grid, params, f = configs.harris(n[0], ny=n[1], nz=n[2], damping=damping)
    params.conduction = 1
    params.kappa_0 = 1.0e-2
    dev, orc = Device(grid, params, f), Oracle(grid, params, f)
    print(f"\n[case] chunked steps n={n}", flush=True)
    for d in (dev, orc):
        d.boundary_conditions()
        d.eta_calc()
    for step in (1, 2):
        assert dev.step(step) == orc.step(step)
        fd, fo = dev.fields(), orc.fields()
        for name in STATE:
            assert np.array_equal(getattr(fd, name), getattr(fo, name)), (step, name)
    dev.close()
    orc.close()
