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


@pytest.mark.parametrize("ny", [4, 5, 6, 7, 9, 16])
@pytest.mark.parametrize("types", [(1, 1, 0, 0), (1, 1, 1, 1), (1, 0, 0, 1)])
@pytest.mark.parametrize("method", [mg.METHOD_KRYLOV_MG, mg.METHOD_KRYLOV_MG32])
def test_sweeps_of_few_rows(ny, types, method):
    """The boundary rows relax beside the other rows of their colour, on saved
    copies of the rows they reach; with few rows each row is a boundary row or
    next to one, and rows 2 and ny-3 may be the same or swap roles.  The solve
    must reach the direct solution, and the batch the same as the single
    solver."""
    import scipy.sparse.linalg as spl
    from cases import probed_matrix
    geo, bc, _, rhs = setup(40, ny, 0.08, 3.0, types, seed=ny)
    exact = spl.spsolve(probed_matrix(geo, bc).tocsc(), rhs.ravel()).reshape(geo.ny, geo.nx)
    s = mg.Solver(geo, bc, method=method)
    s.set_rhs(rhs)
    _, iters, oc = s.solve(1e-12, 100)
    assert oc == mg.CONVERGED and iters <= 30, iters
    np.testing.assert_allclose(s.get_phi()[1:-1, 1:-1], exact, rtol=0, atol=1e-10 * np.max(np.abs(exact)))
    b = mg.Batch([geo], [bc], method=method)
    b.set_rhs(0, rhs)
    its, oc = b.solve(1e-12, 100)
    assert oc[0] == mg.CONVERGED and its[0] <= 30
    np.testing.assert_allclose(b.get_phi(0), exact, rtol=0, atol=1e-10 * np.max(np.abs(exact)))


def test_many_rows_use_one_wave_each():
    """Past 512 rows in a launch, rows of 129 .. 512 cells take one wave each
    instead of 256 threads: 514 rows per colour here."""
    nx, ny = 300, 1030
    geo, bc, phi, rhs = setup(nx, ny, 0.05, 1.0, (1, 1, 0, 0), seed=2)
    got = mg.xline_relax(geo, bc, rhs, phi, 1)[1:-1, 1:-1]
    want = zebra_reference(geo, bc, rhs, phi, 1)
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-10 * np.max(np.abs(want)))


@pytest.mark.parametrize("nx", [1025, 2048, 2049, 4112, 8192, 8200])
def test_fp32_rows_of_each_width(nx):
    """FP32 cycles with few rows: 512 threads for 1025 .. 2048 cells, 256 up to
    4111, 1024 up to 8199 and 512 for the last few lengths.  x-lines are nearly
    a direct solve on this grid, so a wrong row solve shows as iterations."""
    import refcall as rc
    ny = 12
    geo, bc, _, rhs = setup(nx, ny, 0.0, 0.0, (1, 1, 0, 0), seed=nx)
    s = mg.Solver(geo, bc, method=mg.METHOD_KRYLOV_MG32, lines=mg.LINES_X)
    s.set_rhs(rhs)
    hist, iters, oc = s.solve(1e-9, 60)
    assert oc == mg.CONVERGED and iters <= 12, (iters, hist[-3:])
    r, _ = rc.oracle().residual(geo, bc, 1, rhs, s.get_phi())
    assert np.linalg.norm(r) <= 1.5e-9 * np.linalg.norm(rhs)


@pytest.mark.parametrize("nx,ny", [(4, 16), (63, 8), (64, 9), (65, 15), (66, 17), (128, 32), (129, 33), (130, 66)])
@pytest.mark.parametrize("types", [(1, 1, 0, 0), (1, 1, 1, 1), (0, 0, 1, 1)])
@pytest.mark.parametrize("method", [mg.METHOD_KRYLOV_MG, mg.METHOD_KRYLOV_MG32])
def test_operator_and_restriction_tiles(nx, ny, types, method):
    """The operator and the residual's restriction split a tile into interior
    cells and one side of the ring per wave: sizes one off the tile's 64
    columns and its 8, 16 and 32 rows.  The solvers' recurrences apply the
    operator tile by tile and the residual they end on is checked cell by
    cell, so the solution is the direct one only if no cell is left out or
    counted twice."""
    import scipy.sparse.linalg as spl
    from cases import probed_matrix
    geo, bc, _, rhs = setup(nx, ny, 0.08, 3.0, types, seed=ny)
    exact = spl.spsolve(probed_matrix(geo, bc).tocsc(), rhs.ravel()).reshape(geo.ny, geo.nx)
    s = mg.Solver(geo, bc, method=method)
    s.set_rhs(rhs)
    _, _, oc = s.solve(1e-12, 100)
    assert oc == mg.CONVERGED
    np.testing.assert_allclose(s.get_phi()[1:-1, 1:-1], exact, rtol=0, atol=1e-10 * np.max(np.abs(exact)))
    b = mg.Batch([geo], [bc], method=method)
    b.set_rhs(0, rhs)
    _, oc = b.solve(1e-12, 100)
    assert oc[0] == mg.CONVERGED
    np.testing.assert_allclose(b.get_phi(0), exact, rtol=0, atol=1e-10 * np.max(np.abs(exact)))


@pytest.mark.parametrize("nx,ny", [(4, 5), (255, 4), (256, 5), (257, 4), (511, 4), (513, 5)])
@pytest.mark.parametrize("method", [mg.METHOD_KRYLOV_MG, mg.METHOD_KRYLOV_MG32])
def test_iteration_passes_at_row_ends(nx, ny, method):
    """The iteration's last pass takes two cells a thread 256 apart and sums
    beside its updates; a launch's last workgroup adds the others' sums.  Two
    solves in a row start from the count the first left."""
    import scipy.sparse.linalg as spl
    from cases import probed_matrix
    geo, bc, _, rhs = setup(nx, ny, 0.08, 3.0, (1, 1, 0, 0), seed=nx)
    exact = spl.spsolve(probed_matrix(geo, bc).tocsc(), rhs.ravel()).reshape(geo.ny, geo.nx)
    s = mg.Solver(geo, bc, method=method)
    for _ in range(2):
        s.set_rhs(rhs)
        assert s.solve(1e-12, 100)[2] == mg.CONVERGED
        np.testing.assert_allclose(s.get_phi()[1:-1, 1:-1], exact, rtol=0, atol=1e-10 * np.max(np.abs(exact)))
