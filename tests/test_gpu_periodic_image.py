"""Axes that join themselves are read at the periodic image instead of in
exchanged ghosts: blocks as thin as the ghost layers, ragged tiles, one step
and several, against the oracle, and the ghosts that get_state returns."""
import numpy as np
import pytest

from musica2_newgrid_amd import _lib, cases
from musica2_newgrid_amd import grid as gr
from tests._util import relerr

G = gr.G
pytestmark = pytest.mark.gpu


def _case(geo, nx, ny, nz, filt):
    h = 0.01
    lengths = (nx * h, ny * h, nz * h)
    if geo == "c3":
        c = cases.vortex_wavy(nx, ny, nz, filter=filt, lengths=lengths, radius=0.25 * min(lengths[:2]), beta=1.0)
    elif geo == "c2":
        c = cases.vortex_wavy_c2(nx, ny, nz, filter=filt, lengths=lengths, radius=0.25 * min(lengths[:2]), beta=1.0)
    else:
        rng = np.random.default_rng(nx + 10 * ny + 100 * nz)
        f = [1.0 + 0.05 * rng.uniform(-1, 1, (nz, ny, nx)) for _ in range(5)]
        c = cases.cartesian_box(nx, ny, nz, lengths, (1.177 * f[0], 30 * f[1], 20 * f[2], 10 * f[3], 1e5 * f[4]),
                                iorder_visc=4, filter=filt, dt=5e-6)
        c.ducros = True
    return c


@pytest.mark.parametrize("geo", ["cart", "c2", "c3"])
@pytest.mark.parametrize("shape", [(5, 5, 5), (7, 70, 6), (69, 5, 19), (33, 17, 64)])
@pytest.mark.parametrize("filt", [1, 2])
def test_periodic_image_matches_oracle(geo, shape, filt):
    from musica2_newgrid_amd.solver import GpuSolver
    from oracle.oracle import Oracle
    c = _case(geo, *shape, filt)
    print(f"{geo} {shape} filter {filt}", flush=True)
    with GpuSolver(c) as s:
        s.step(1)
        s.step(4)
        U = s.get_state()
    ref = c.copy_state()
    Oracle(c).step(ref, 5)
    # round-off of 20 stages: as the other parity tests
    assert relerr(U, ref) < 1e-12
    for a in U:
        core = a[G:-G, G:-G, G:-G]
        for ax in range(3):
            n = core.shape[ax]
            lo = [slice(G, -G)] * 3
            hi = [slice(G, -G)] * 3
            lo[ax], hi[ax] = slice(0, G), slice(-G, None)
            assert np.array_equal(a[tuple(lo)], np.take(core, range(n - G, n), axis=ax))
            assert np.array_equal(a[tuple(hi)], np.take(core, range(G), axis=ax))


def test_partly_joined_block_table():
    """Two blocks joined along i, each onto itself along j and k, equal their parent bit by bit."""
    from musica2_newgrid_amd import multiblock as mb
    from musica2_newgrid_amd.solver import GpuSolver
    parent = _case("cart", 40, 13, 11, 2)
    ident = [((0, 1, 2), (1, 1, 1))] * 2
    blocks, bcs = mb.split_oriented(parent, 2, ident)
    print("two blocks along i against their parent", flush=True)
    for precision in (_lib.PREC_FP64, _lib.PREC_MIXED):
        with GpuSolver(bcs[0], precision=precision, topology=blocks, block_cases=bcs, stage_kernel="pipelined") as s:
            s.step(6)
            Us = mb.join_oriented(parent, s.get_states(), ident)
        with GpuSolver(parent, stage_kernel="pipelined") as s:
            s.step(6)
            U = s.get_state()
        if precision == _lib.PREC_FP64:
            for a, b in zip(Us, U):
                assert np.array_equal(gr.interior(a), gr.interior(b))
        else:
            assert relerr(Us, U) < 1e-5  # FP32 fluxes
