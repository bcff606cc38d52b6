"""The metrics of the no-allocation energies at the edges of their transport:
one full launch of arguments, one value more, two full launches, and the
copies above that; the same bits as the library's energies."""
import pytest

from lare3d_amd import configs
from tests.test_zz_no_alloc import _library_energies, _noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [460, 461, 940, 941])
def test_metrics_in_arguments_and_copies(nx):
    print(f"\n[case] noalloc energies {nx}x4x4", flush=True)
    grid, fields, en_ref, divb_ref = _library_energies(configs.harris(nx, ny=4, nz=4, stretch=(24.0, 10.0, 24.0)), 1)
    en, divb = _noalloc(grid, fields)
    assert en == en_ref
    assert divb == divb_ref
