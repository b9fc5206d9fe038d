"""The ordered sums of the reference's cycles on the GPU, bit for bit against
the oracle where their forms change: the bottom solver in LDS with one wave
(up to 64 cells), in LDS with four, and in global memory (from about 30 x 30
cells), each ordering; and the ordered mean of the prolongation at the edges
of its tiles of 1024 cells."""
import numpy as np
import pytest

import refcall as rc
from cases import coarse_geo, setup
from mgpoisson2d_amd import geometry as G

pytestmark = pytest.mark.gpu

mg = pytest.importorskip("mgpoisson2d_amd.capi")

SIZES = [(4, 4), (8, 8), (13, 5), (29, 29), (31, 30), (53, 37)]


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("types", [(1, 1, 0, 0), (0, 0, 0, 0), (0, 1, 1, 0)])
@pytest.mark.parametrize("kind,order", [(0, rc.LEX), (1, rc.LEX), (1, rc.RB)])
def test_bottom_solver_forms(nx, ny, types, kind, order):
    geo, bc, phi, rhs = setup(nx, ny, 0.08, 1.0, types, seed=nx + ny)
    if kind == 1:
        bc = G.BoundaryConditions.uniform(types, mode=G.BCMODE_LAH)
    o = rc.oracle()
    inv = o.dc_invdiags(geo) if kind == 1 else o.invdiags(geo, bc, 1)
    its = 80 if nx * ny <= 64 else 6
    got = mg.solve_bicgstab2(kind, geo, bc, 1, inv, 1e-6, its, 5, 1, rhs, phi, ordering=order)
    want = o.bicgstab2(kind, geo, bc, 1, inv, 1e-6, its, 5, 1, rhs, phi, order=order)
    np.testing.assert_array_equal(got[1:-1, 1:-1], want[1:-1, 1:-1])


@pytest.mark.parametrize("nx,ny", [(4, 4), (8, 8), (12, 9)])
@pytest.mark.parametrize("types", [(1, 1, 0, 0), (0, 0, 0, 0)])
def test_bottom_solver_multi_colour(nx, ny, types):
    """One level only: the cycle is the smoother and the bottom solver."""
    geo, bc, phi, rhs = setup(nx, ny, 0.05, 1.0, types, seed=3 * nx + ny)
    got = mg.vcycle(0, geo, bc, 1, 0.0, 1, phi, rhs, maxdepth=0, zerophi=True, ordering=mg.ORDER_MC)
    want = rc.oracle().vcycle(0, geo, bc, 1, 0.0, 1, phi, rhs, maxdepth=0, zerophi=True, order=rc.MC)
    np.testing.assert_array_equal(got[0][1:-1, 1:-1], want[0][1:-1, 1:-1])


@pytest.mark.parametrize("nx,ny", [(8, 8), (32, 32), (64, 48), (62, 34), (66, 32), (256, 256)])
def test_ordered_mean(nx, ny):
    geo, _, _, _ = setup(nx, ny, 0.1, 2.0, (0, 0, 0, 0), seed=9)
    o = rc.oracle()
    cgeo = coarse_geo(o.restrict, geo)
    rng = np.random.default_rng(nx * ny)
    fine, crse = rng.standard_normal((ny + 2, nx + 2)), rng.standard_normal((cgeo.ny + 2, cgeo.nx + 2))
    got, _ = mg.prolong(geo, cgeo, (0, 0, 0, 0), (0,) * 4, 1, fine, crse)
    want, _ = o.prolong(geo, cgeo, (0, 0, 0, 0), (0,) * 4, 1, fine, crse)
    np.testing.assert_array_equal(got[1:-1, 1:-1], want[1:-1, 1:-1])


# lexicographic sweeps are one workgroup: the small sizes only
@pytest.mark.parametrize("n,order", [(32, rc.LEX), (64, rc.LEX), (32, rc.RB), (64, rc.RB), (96, rc.RB), (160, rc.RB)])
@pytest.mark.parametrize("types", [(1, 1, 0, 0), (1, 1, 1, 1), (0, 1, 1, 0), (0, 0, 0, 0), (2, 2, 1, 1)])
@pytest.mark.parametrize("numcycles,up", [(1, 2), (2, 1), (1, 0)])
def test_dc_cycle_transfers(n, types, order, numcycles, up):
    """The DC cycle's fused transfers (Neumann and Dirichlet sides, smoothing
    after the correction) and the separate ones (a periodic side, or none):
    two cycles against the oracle, bit for bit where no parallel sum enters."""
    geo, bc, phi, rhs = setup(n, n, 0.02, 0.3, types, seed=n)
    o = rc.oracle()
    args = dict(numcycles=numcycles, zerophi=True)
    got = mg.vcycle(1, geo, bc, 1, 0.0, 2, phi, rhs, smooth_up=up, ordering=order, **args)
    want = o.vcycle(1, geo, bc, 1, 0.0, 2, phi, rhs, sup=up, order=order, **args)
    assert (got[3], got[4]) == (want[3], want[4])
    np.testing.assert_array_equal(got[0][1:-1, 1:-1], want[0][1:-1, 1:-1])
