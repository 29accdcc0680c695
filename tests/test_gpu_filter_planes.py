"""The selective and the shock filter's march with one barrier per plane:
tiles that end inside a halo, columns shorter than a chunk of three planes,
bounded rows, periodic images and filled ghosts, against the oracle."""
import pytest

from musica2_newgrid_amd import cases
from tests._util import relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("filt", [1, 2])
@pytest.mark.parametrize("shape", [(32, 16, 11), (33, 17, 12), (38, 22, 13), (63, 31, 29), (70, 49, 11)])
@pytest.mark.parametrize("walls", [False, True])
def test_filters_match_oracle(walls, shape, filt):
    from musica2_newgrid_amd.solver import GpuSolver
    from oracle.oracle import Oracle
    nx, ny, nz = shape
    if walls:
        c = cases.duct(nx, ny, nz, filter=filt)
    else:
        c = cases.shock_tube(nx, ny, nz)
        c.filter = filt
    print(f"walls={walls} {shape} filter={filt}", flush=True)
    with GpuSolver(c) as s:
        s.step(2)
        U = s.get_state()
    ref = c.copy_state()
    Oracle(c).step(ref, 2)
    # round-off of 8 stages and 2 filters: as the other parity tests
    assert relerr(U, ref) < 1e-12
