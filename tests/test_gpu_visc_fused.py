"""The viscous terms in one kernel (blocks whose three axes wrap, long
k-chunks): partial tiles in i and j, a short last chunk, every geometry, the
shock filter's pressure and sensor from it, against the oracle."""
import pytest

from musica2_newgrid_amd import cases
from tests._util import relerr

pytestmark = pytest.mark.gpu


# the shortest chunks that take this path (5 planes, the last of 1), and longer ones
SHAPES = [(113, 75, 51), (133, 129, 57), (160, 144, 53), (130, 210, 43)]


@pytest.mark.parametrize("geo", ["cart", "c2", "c3"])
@pytest.mark.parametrize("shape", SHAPES)
def test_fused_viscous_terms_match_oracle(geo, shape):
    from musica2_newgrid_amd.solver import GpuSolver
    from oracle.oracle import Oracle
    nx, ny, nz = shape
    lengths = (0.01 * nx, 0.01 * ny, 0.01 * nz)
    if geo == "cart":
        c = cases.shock_tube(nx, ny, nz)
    else:
        make = cases.vortex_wavy if geo == "c3" else cases.vortex_wavy_c2
        c = make(nx, ny, nz, lengths=lengths, radius=0.1, re=200.0)
    print(f"{geo} {shape}", flush=True)
    with GpuSolver(c) as s:
        assert s.stage_config(2)[2] >= 5
        s.step(2)
        U = s.get_state()
    ref = c.copy_state()
    Oracle(c).step(ref, 2)
    # round-off of 8 stages: as the other parity tests
    assert relerr(U, ref) < 1e-12
