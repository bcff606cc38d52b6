"""Steps that enter with negative energies in some cells, against the CPU
restatement: MAX(energy, 0), which the predictor and the corrector take on what
they read, without and with CAUCHY, beside the viscous heating, and after
FOURTHORDER substeps; every element of every state array."""
import numpy as np
import pytest

from lare3d_amd import BC_OPEN, BC_PERIODIC, configs
from lare3d_amd.grid import Grid
from tests.util import STATE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("problem,options", [
    ("vortex", {}),
    ("vortex", {"cauchy": 1}),
    ("vortex", {"visc1": 0.1, "visc2": 0.5, "rke": 1}),
    ("open", {}),
    ("sheet", {"fourth_order": 1}),
])
def test_negative_energies_on_entry(problem, options):
    from lare3d_amd.device import Device
    from oracle.oracle import Oracle
    if problem == "sheet":
        grid, params, f = configs.harris(20, ny=17, nz=23)
    else:
        grid, params, f = configs.orszag_tang(20)
    if problem == "open":
        grid = Grid(*grid.n, grid.extent, (BC_PERIODIC,) * 4 + (BC_OPEN,) * 2, grid.stretch, grid.widths)
    for key, value in options.items():
        setattr(params, key, value)
    f.bz[...] += 1.0  # the fast speed of a cell with negative pressure stays real
    cells = np.random.default_rng(7).random(f.energy.shape) < 0.05
    if problem == "open":  # the far field and the layers beside it stay as they are
        cells[:, :, :6] = cells[:, :, -6:] = False
    f.energy[cells] = -0.02
    dev, orc = Device(grid, params, f), Oracle(grid, params, f)
    for d in (dev, orc):
        d.boundary_conditions()
        d.eta_calc()
    for step in (1, 2, 3):
        print(f"\n[case] negative energies {problem} {options} step={step}", flush=True)
        assert dev.step(step) == orc.step(step)
        fd, fo = dev.fields(), orc.fields()
        assert np.isfinite(fo.interior("energy")).all()
        for name in STATE + ("visc_dep", "ohmic_dep"):
            assert np.array_equal(getattr(fd, name), getattr(fo, name)), (step, name)
    dev.close()
    orc.close()
