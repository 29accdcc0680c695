"""get_state through the pinned slots: an upload read back bit by bit, at sizes
of one piece, of a few pieces and of more pieces than slots, with the padding
between the arrays of a set inside a piece; and after a larger block of the
same handle has grown the slots."""
import numpy as np
import pytest

from musica2_newgrid_amd import cases
from musica2_newgrid_amd import grid as gr

G = gr.G
pytestmark = pytest.mark.gpu


def _box(nx, ny, nz):
    rng = np.random.default_rng(nx * 10007 + ny * 101 + nz)
    f = [1.0 + 0.1 * rng.uniform(-1, 1, (nz, ny, nx)) for _ in range(5)]
    return cases.cartesian_box(nx, ny, nz, (1.0, 1.0, 1.0), (f[0], f[1], f[2], f[3], 1e5 * f[4]))


# 0.14 MB, 0.7 MB (one piece), 1.1 MB (first with threads), 5, 33 and 80 MB (more pieces than slots)
@pytest.mark.parametrize("shape", [(5, 5, 5), (16, 16, 16), (21, 20, 19), (41, 40, 39), (90, 83, 79), (131, 115, 107)])
def test_state_comes_back_as_uploaded(shape):
    from musica2_newgrid_amd.solver import GpuSolver
    c = _box(*shape)
    print(f"fetch {shape}", flush=True)
    with GpuSolver(c) as s:
        for _ in range(2):
            for a, b in zip(s.get_state(), c.U):
                assert np.array_equal(a, b)


def test_slots_grow_with_the_largest_block():
    from musica2_newgrid_amd.solver import GpuSolver
    from musica2_newgrid_amd.multiblock import periodic_block
    shapes = [(16, 16, 16), (90, 83, 79), (21, 20, 19)]
    cs = [_box(*n) for n in shapes]
    table = [periodic_block(*n, b=b) for b, n in enumerate(shapes)]
    print("fetch of three blocks of one handle", flush=True)
    with GpuSolver(cs[0], topology=table, block_cases=cs) as s:
        for U, c in zip(s.get_states(), cs):
            for a, b in zip(U, c.U):
                assert np.array_equal(a, b)
