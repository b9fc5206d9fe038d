"""The row solve of the x-line relaxation at the edges of its forms: rows of
fewer cells than a wave, chunk counts one off a power of two, and the last
rows of each chunk length (2, 4, 8, 16) and width."""
import numpy as np
import pytest

from cases import setup
from test_gpu_solver import zebra_reference

pytestmark = pytest.mark.gpu

mg = pytest.importorskip("mgpoisson2d_amd.capi")


@pytest.mark.parametrize("nx,ny", [(4, 4), (5, 6), (7, 5), (65, 4), (127, 4), (129, 5), (255, 4), (512, 4), (513, 4),
                                   (1027, 4), (1030, 5), (2055, 4), (2056, 4), (4111, 4)])
@pytest.mark.parametrize("types", [(1, 1, 0, 0), (0, 1, 1, 0)])
def test_row_solve_edges(nx, ny, types):
    geo, bc, phi, rhs = setup(nx, ny, 0.08, 2.0, types, seed=nx)
    got = mg.xline_relax(geo, bc, rhs, phi, 2)[1:-1, 1:-1]
    want = zebra_reference(geo, bc, rhs, phi, 2)
    # the row system's condition number is about 2 (dy / dx)^2 where the x couplings dominate
    tol = max(1e-10, 4 * np.finfo(float).eps * 2.0 * (geo.dy / geo.dx) ** 2)
    np.testing.assert_allclose(got, want, rtol=0, atol=tol * np.max(np.abs(want)))
