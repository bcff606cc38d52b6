"""Infinities given to the diagnostics and quantities that leave the range of the
type, against the CPU restatement.  What is compared is a time step, or
whether a value is finite, so equality is exact."""
import numpy as np
import pytest

from lare3d_amd import configs
from lare3d_amd.abi import DeviceError, PREC_FP32
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


def _pair(cfg):
    from lare3d_amd.device import Device
    from oracle.oracle import Oracle
    dev, orc = Device(*cfg), Oracle(*cfg)
    for d in (dev, orc):
        d.set_scalars(dt=1.0e-2)  # of the step before, which the edge viscosity looks at
        d.boundary_conditions()
        d.eta_calc()
    return dev, orc


def _thin_cell(b, visc):
    """Density 1e-300 in one cell, a field b on one of its faces alone."""
    grid, params, f = configs.orszag_tang(12)
    params.visc1, params.visc2 = visc
    f.rho[7, 7, 7] = 1e-300
    f.by[...] = f.bz[...] = 0.0
    f.bx[8, 7, 7] = b
    return grid, params, f


def test_infinite_speed_stops_the_step():
    # b^2 / rho = 4e308 in set_dt, 1e308 with the face average of the cell
    print("\n[case] infinite speed in set_dt", flush=True)
    dev, orc = _pair(_thin_cell(2.0e4, (0.0, 0.0)))
    assert orc.step(1)[0] == 0.0
    with pytest.raises(DeviceError, match="invalid dt 0"):
        dev.step(1)
    dev.close()
    orc.close()


def test_infinite_speed_of_a_cell_stays_on_its_nodes():
    # the cell's own speed is infinite: its edges to other nodes take theirs
    print("\n[case] infinite speed of a cell", flush=True)
    dev, orc = _pair(_thin_cell(1.0e5, (0.1, 0.5)))
    for d in (dev, orc):
        d.lagrangian_step()
    assert dev.scalars().dt == orc.scalars().dt
    for name in ("rho", "energy", "vx", "vy", "vz"):
        a, b = dev.fields().interior(name), orc.fields().interior(name)
        assert np.array_equal(np.isfinite(a), np.isfinite(b)), name
    dev.close()
    orc.close()


def test_viscous_heating_beyond_the_range():
    print("\n[case] viscous heating overflow", flush=True)
    grid, params, f = configs.orszag_tang(12)
    params.visc1, params.visc2 = 0.1, 0.5
    f.vx[6, 6, 6] = 1.0e104  # density x (velocity difference)^3 overflows, its square does not
    dev, orc = _pair((grid, params, f))
    for d in (dev, orc):
        d.lagrangian_step()
    for name in ("rho", "energy", "vx", "vy", "vz", "visc_dep"):
        a, b = dev.fields().interior(name), orc.fields().interior(name)
        assert np.array_equal(np.isfinite(a), np.isfinite(b)), name
    assert np.isinf(orc.fields().interior("energy")).any()
    dev.close()
    orc.close()


def test_ohmic_heating_beyond_the_range():
    print("\n[case] ohmic heating overflow", flush=True)
    grid, params, f = configs.harris(12)
    params.eta_background, params.eta0, params.visc1, params.visc2 = 1.0e7, 0.0, 0.0, 0.0
    # a thin cell without a field of its own, in the current of its neighbours'
    f.rho[6, 6, 6] = 1e-300
    f.bx[...] = 1.0e10
    f.bx[6:8, 6, 6] = f.by[6, 6:8, 6] = f.bz[6, 6, 6:8] = 0.0
    dev, orc = _pair((grid, params, f))
    for d in (dev, orc):
        d.lagrangian_step()
    assert dev.scalars().last_substeps == orc.scalars().last_substeps == 1
    lost = ~np.isfinite(orc.fields().interior("ohmic_dep"))
    assert lost.any()
    for name in ("ohmic_dep", "energy"):
        assert not np.isfinite(dev.fields().interior(name)[lost]).any(), name
    dev.close()
    orc.close()


@pytest.mark.parametrize("k", range(8, 16))
def test_negative_temperature_beside_the_step_limit(k):
    """One plane above the cell that sets the conduction step limit (229 stages;
    9 without it), a cell whose own limit is NaN."""
    print(f"\n[case] conduction step limit beside NaN, k={k}", flush=True)
    from lare3d_amd.device import Device
    grid, params, f, dt = configs.arcade_conduction(64, 64, 64, s_target=9)
    f.energy[20, 7, k] = 20.0 * f.energy.max()
    f.energy[20, 7, k + 1] = -1.0
    dev = Device(grid, params, f)
    dev.set_scalars(dt=dt)
    dev.boundary_conditions()
    dev.conduct_heat()
    assert dev.scalars().n_s_stages == 229
    dev.close()


@pytest.mark.parametrize("k", range(8, 16))
def test_nan_beside_the_largest_divergence(k):
    """One and two planes above the two cells with the largest |div B|, cells whose
    own is NaN."""
    print(f"\n[case] div B beside NaN, k={k}", flush=True)
    from lare3d_amd.device import Device
    grid, params, f = configs.orszag_tang(64)
    f.bx[20, 7, k] += 100.0
    want = []
    for nan in (False, True):
        if nan:
            f.bz[19:21, 7, k + 2] = np.nan
        dev = Device(grid, params, f)
        want.append(dev.divb())
        dev.close()
    assert want[0] == want[1] > 1.0


@pytest.mark.parametrize("e", [1.0e91, 1.0e100])
def test_limited_flux_beyond_the_range(e):
    """A conduction whose unlimited flux overflows in two cells: the flux limiter's
    factor is zero there."""
    print("\n[case] conduction flux overflow", flush=True)
    from lare3d_amd.device import Device
    from oracle.oracle import Oracle
    grid, params, f, dt = configs.harris_conduction(12, seed=1)
    params.heat_flux_limiter, params.flux_limiter = 1, 0.1
    f.energy[6:8, 6, 6] = e
    out = []
    for cls in (Device, Oracle):
        sim = cls(grid, params, f)
        sim.set_scalars(dt=0.01 * dt)
        sim.boundary_conditions()
        sim.conduct_heat()
        out.append((sim.scalars().n_s_stages, sim.fields().interior("energy")))
        sim.close()
    assert out[0][0] == out[1][0] == 3
    assert np.array_equal(out[0][1], out[1][1], equal_nan=True)


@pytest.mark.parametrize("field,value", [("bx", 1.0e155), ("rho", 1.0e-100)])
def test_flux_over_an_infinite_field(field, value):
    """B^2 beyond the range in two cells (no flux), and a density whose energy
    grows beyond it."""
    print(f"\n[case] conduction with {field} = {value}", flush=True)
    from lare3d_amd.device import Device
    from oracle.oracle import Oracle
    grid, params, f, dt = configs.harris_conduction(12, seed=1)
    getattr(f, field)[6:8, 6, 6] = value
    out = []
    for cls in (Device, Oracle):
        sim = cls(grid, params, f)
        sim.set_scalars(dt=1.0e-4 if field == "bx" else 1.0e-6)
        sim.boundary_conditions()
        sim.conduct_heat()
        out.append((sim.scalars().n_s_stages, sim.fields().interior("energy")))
        sim.close()
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1], equal_nan=True)


@pytest.mark.parametrize("precision,b", [(0, 1.7e308), (PREC_FP32, 1.0e39)])
def test_infinite_current_is_above_the_threshold(precision, b):
    """Currents beyond the range (the difference or its quotient) are above j_max:
    eta is eta_background + eta0 at their nodes, as the restatement has it."""
    print(f"\n[case] infinite current precision={precision}", flush=True)
    from lare3d_amd.device import Device
    from oracle.oracle import Oracle
    grid, params, f = configs.harris(12)
    params.eta_background, params.eta0 = 1.0 / 1024, 1.0 / 64  # values that FP32 holds
    params.j_max = 1.0e30
    f.bx[6, 6, 6] = b  # over the 2/3 of a cell in y
    orc = Oracle(grid, params, f)
    params.precision = precision
    dev = Device(grid, params, f)
    eta = []
    for sim in (dev, orc):
        sim.boundary_conditions()
        sim.eta_calc()
        eta.append(sim.fields().eta)
        sim.close()
    assert np.array_equal(eta[0], eta[1], equal_nan=True)
    assert (eta[1] > 1.0 / 64).any() and (eta[1] < 1.0 / 64).any()
