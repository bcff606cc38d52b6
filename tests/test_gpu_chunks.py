"""Full steps against the CPU restatement on grids for which the marching
kernels take chunks of 3 points and of 6 to 8 (1, 2, 4 and 5: test_gpu_march.py),
with a short last chunk, and on one on which every sweep's momentum remap and CT
sweep are launches of their own: every element of every state array."""
import numpy as np
import pytest

from lare3d_amd import configs
from tests.util import STATE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(72, 71, 73), (107, 96, 100), (120, 97, 102)])
def test_steps_at_the_other_chunks(n):
    from lare3d_amd.device import Device
    from oracle.oracle import Oracle
    grid, params, f = configs.harris(n[0], ny=n[1], nz=n[2], stretch=(24.0, 10.0, 24.0))
    params.conduction = 1
    params.kappa_0 = 1.0e-2
    dev, orc = Device(grid, params, f), Oracle(grid, params, f)
    print(f"\n[case] chunked steps n={n}", flush=True)
    for d in (dev, orc):
        d.boundary_conditions()
        d.eta_calc()
    assert dev.step(1) == orc.step(1)
    fd, fo = dev.fields(), orc.fields()
    for name in STATE:
        assert np.array_equal(getattr(fd, name), getattr(fo, name)), name
    dev.close()
    orc.close()


def test_sweeps_of_large_grids():
    from lare3d_amd.device import Device
    from oracle.oracle import Oracle
    grid, params, f = configs.harris(192, ny=190, nz=190)
    dev, orc = Device(grid, params, f), Oracle(grid, params, f)
    print("\n[case] sweeps apart 192x190x190", flush=True)
    for d in (dev, orc):
        d.boundary_conditions()
        d.eta_calc()
    dev.profile(True)
    assert dev.step(1) == orc.step(1)
    names = dev.kernel_stats()
    assert "mom_remap" in names and "ct_sweep" in names and "mom_ct" not in names
    fd, fo = dev.fields(), orc.fields()
    for name in STATE:
        assert np.array_equal(getattr(fd, name), getattr(fo, name)), name
    dev.close()
    orc.close()
