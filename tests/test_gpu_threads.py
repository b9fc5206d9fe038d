"""Distinct solvers from distinct threads: what a solve gives beside others in
other threads is what it gives alone, while threads allocate, copy, capture
their iterations and free in every order."""
import threading
from types import SimpleNamespace

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

mg = pytest.importorskip("mgpoisson2d_amd.capi")
from mgpoisson2d_amd import geometry as G  # noqa: E402

DDNN = G.BoundaryConditions.uniform((1, 1, 0, 0))


def shape(nx, ny):
    return SimpleNamespace(nx=nx, ny=ny, dx=1.0 / nx, dy=1.0 / ny)


def rhs(nx, ny):
    return np.random.default_rng(nx + ny).standard_normal((ny, nx))


def solve(nx, ny, amp=0.05, beta=2.0, **opts):
    s = mg.Solver(shape(nx, ny), DDNN, mapping=mg.Mapping(mg.MAP_WARPED, amp, beta, 0.0, 0.0), **opts)
    s.set_rhs(rhs(nx, ny))
    s.solve_fast(1e-9, 60)
    phi = s.get_phi()[1:-1, 1:-1].copy()
    s.close()
    return phi


def dropin(n):
    geo = G.mapped_geometry(n, n, 0.0, 0.0)
    return mg.vcycle(1, geo, DDNN, 1, 0.0, 3, np.zeros((n + 2, n + 2)), rhs(n, n), ordering=mg.ORDER_RB)[0][1:-1, 1:-1]


def batch(sizes):
    b = mg.Batch([shape(*q) for q in sizes], [DDNN] * len(sizes),
                 mappings=[mg.Mapping(mg.MAP_WARPED, 0.05, 2.0, 0.0, 0.0)] * len(sizes))
    for k, q in enumerate(sizes):
        b.set_rhs(k, rhs(*q))
    b.solve(1e-9, 60)
    phi = np.concatenate([b.get_phi(k).ravel() for k in range(len(sizes))])
    b.close()
    return phi


JOBS = [
    lambda: solve(64, 64),
    lambda: solve(300, 200, method=mg.METHOD_KRYLOV_MG32),
    lambda: solve(513, 257),
    lambda: solve(256, 64, krylov=mg.KRYLOV_FGMRES),
    lambda: solve(96, 96, 0.0, 0.0, method=mg.METHOD_DC_VCYCLE, ordering=mg.ORDER_RB),
    lambda: dropin(128),
    lambda: batch([(64, 48), (130, 33), (576, 32)]),
]


def test_solvers_in_threads():
    want = [job() for job in JOBS]
    for _ in range(6):
        got, errors = [None] * len(JOBS), []

        def run(k):
            try:
                got[k] = JOBS[k]()
            except Exception as e:  # noqa: BLE001 -- reported below, with its job
                errors.append((k, str(e)))

        threads = [threading.Thread(target=run, args=(k,)) for k in range(len(JOBS))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors
        for k in range(len(JOBS)):
            np.testing.assert_array_equal(got[k], want[k], err_msg=f"job {k}")
