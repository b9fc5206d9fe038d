"""Device memory of a resident solver: its arrays and no more.  A solver holds
the five metrics, phi and rhs, nine Krylov vectors and, per level, eight arrays
(five metrics, three fields); the rows of a level halve only where the sides
allow it."""
import ctypes
from types import SimpleNamespace

import pytest

pytestmark = pytest.mark.gpu

mg = pytest.importorskip("mgpoisson2d_amd.capi")
from mgpoisson2d_amd import geometry as G  # noqa: E402


def free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert mg.lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


# an odd row count between Dirichlet sides has one level: 7 + 9 + 8 level arrays; with y-lines the rows are the columns
@pytest.mark.parametrize("nx,ny,lines", [(2048, 2049, mg.LINES_X), (2049, 2048, mg.LINES_Y)])
def test_one_level_takes_one_level(nx, ny, lines):
    geo = SimpleNamespace(nx=nx, ny=ny, dx=1.0 / nx, dy=1.0 / ny)
    bc = G.BoundaryConditions.uniform((1, 1, 1, 1))
    make = lambda: mg.Solver(geo, bc, mapping=mg.Mapping(mg.MAP_WARPED, 0.05, 1.0, 0.0, 0.0), lines=lines)  # noqa: E731
    make().close()  # what the first solver of a process allocates beside its arrays
    free = free_bytes()
    s = make()
    took = free - free_bytes()
    s.close()
    # a level array with its ghost ring and row padding (at most 64 elements a row); one array's worth for the small ones
    array = 8 * (max(nx, ny) + 64) * (max(nx, ny) + 2)
    assert took <= 25 * array, took / array
