"""energy_account against the CPU restatement on grids for which its march
takes chunks of 1, 2, 4 and 8 planes, the last one short.  The terms of each
sum are positive and the same on both sides, so the sums differ by their
order alone: by at most one rounding per term of the longer chain, the
restatement's over all nodes."""
import numpy as np
import pytest

from lare3d_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(4, 5, 6), (63, 64, 65), (88, 88, 65), (97, 88, 130)])
def test_energies_at_every_chunk(n):
    from lare3d_amd.device import Device
    from oracle.oracle import Oracle
    grid, params, f = configs.harris(n[0], ny=n[1], nz=n[2], stretch=(24.0, 10.0, 24.0))
    rng = np.random.default_rng(5)
    for v in (f.vx, f.vy, f.vz):
        v[...] = 2.0 * rng.random(v.shape) - 1.0
    print(f"\n[case] energies n={n}", flush=True)
    got = []
    for cls in (Device, Oracle):
        sim = cls(grid, params, f)
        sim.boundary_conditions()
        got.append(np.array(sim.energy_account()[:3]))
        sim.close()
    nodes = (n[0] + 1) * (n[1] + 1) * (n[2] + 1)
    assert np.all(np.abs(got[0] - got[1]) <= nodes * 2.0 ** -53 * np.abs(got[1]))
