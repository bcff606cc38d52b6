"""energy_account against the CPU restatement on grids for which its march takes
chunks of 2 to 8 planes with a short last one.  The terms of each sum are the
same on both sides and positive, so the sums differ by their order alone: by at
most one rounding per term of the longer chain, the restatement's over all
nodes.  The chunk is worked out here by the rule of the library, so that a new
rule shows."""
import numpy as np
import pytest

from lare3d_amd import configs

pytestmark = pytest.mark.gpu


def _chunk(per_plane, points):
    """The c of 1..8 with the least max(3, blocks per CU) * (c + 1), the longer of
    two alike, on 256 CUs."""
    cost = [(max(3, -(-per_plane * -(-points // c) // 256)) * (c + 1), -c) for c in range(1, 9)]
    return -min(cost)[1]


@pytest.mark.parametrize("n,chunk,rest", [((63, 57, 68), 2, 1), ((63, 57, 102), 3, 1), ((120, 114, 40), 4, 1),
                                          ((128, 122, 48), 5, 4), ((120, 114, 72), 6, 1), ((120, 114, 78), 7, 2),
                                          ((120, 114, 92), 8, 5)])
def test_energies_with_a_short_last_chunk(n, chunk, rest):
    from lare3d_amd.device import Device
    from oracle.oracle import Oracle
    per_plane = -(-(n[0] + 1) * (n[1] + 1) // 256)
    assert _chunk(per_plane, n[2] + 1) == chunk and (n[2] + 1) % chunk == rest
    grid, params, f = configs.harris(n[0], ny=n[1], nz=n[2], stretch=(24.0, 10.0, 24.0))
    rng = np.random.default_rng(5)
    for v in (f.vx, f.vy, f.vz):
        v[...] = 2.0 * rng.random(v.shape) - 1.0
    print(f"\n[case] energies n={n} chunk={chunk}", flush=True)
    got = []
    for cls in (Device, Oracle):
        sim = cls(grid, params, f)
        sim.boundary_conditions()
        got.append(np.array(sim.energy_account()[:3]))
        sim.close()
    nodes = (n[0] + 1) * (n[1] + 1) * (n[2] + 1)
    assert np.all(np.abs(got[0] - got[1]) <= nodes * 2.0 ** -53 * np.abs(got[1]))
