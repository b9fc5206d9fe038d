"""Cases of work that users of this framework have it do, through its public entry points (mgpoisson2d_amd.capi).

Kinds of case:
  solve    a resident solver (KRYLOV_MG, or KRYLOV_MG32 with FP32 cycles) solves one mapped-grid problem to a tolerance;
  batch    mgp_batch solves many independent problems of uneven sizes together;
  cycles   the reference's deferred-correction (or plain) V-cycle on resident data, to a tolerance;
  project  the divergence cleaning of face fluxes with the reference's FMG driver or with KRYLOV_MG;
  dropin   the drop-in V-cycle call on host arrays, set-up and copies included, as a caller of the reference makes it.

The mapping is x = s + amp sin(2 pi s) sin(2 pi t), y = (exp(beta t) - 1)/(exp(beta) - 1) on the unit square; "types" are the
four sides' boundary conditions (xlo, xhi, ylo, yhi; D Dirichlet, N Neumann), homogeneous.  Right-hand sides are smooth source
terms with 1 % noise, -J (2 pi^2 sin(a x) cos(b y) + 1e-2 N(0, 1)).
"""
import ctypes
import math
from types import SimpleNamespace

import numpy as np
import torch

from mgpoisson2d_amd import capi
from mgpoisson2d_amd import geometry as G

TYPE = {"N": G.BCTYPE_NEUM, "D": G.BCTYPE_DIRI}
METHOD = {"fp64": capi.METHOD_KRYLOV_MG, "fp32": capi.METHOD_KRYLOV_MG32}
MAXITERS = 400


def listed():
    return [
        # the smallest grid a user solves: launches and latency are all of it (the smoke test's problem)
        {"name": "solve 64x64 fp64", "kind": "solve", "nx": 64, "ny": 64, "amp": 0.1, "beta": 5.0, "types": "DDNN", "cycle": "fp64", "tol": 1e-10},
        # odd sizes and mixed sides, as in the operator tests' odd case: ragged rows, and row counts that do not halve
        {"name": "solve 333x257 fp64", "kind": "solve", "nx": 333, "ny": 257, "amp": 0.05, "beta": 4.0, "types": "DNND", "cycle": "fp64", "tol": 1e-10},
        # an ordinary single problem
        {"name": "solve 512x512 fp64", "kind": "solve", "nx": 512, "ny": 512, "amp": 0.1, "beta": 5.0, "types": "DDNN", "cycle": "fp64", "tol": 1e-10},
        # an ordinary problem with FP32 cycles, all sides Dirichlet
        {"name": "solve 1024x768 fp32", "kind": "solve", "nx": 1024, "ny": 768, "amp": 0.1, "beta": 4.0, "types": "DDDD", "cycle": "fp32", "tol": 1e-10},
        # the large single solve of the benchmark (to 1e-9: the FP64 operator's rounding there is near 2e-10)
        {"name": "solve 2048x2048 fp64", "kind": "solve", "nx": 2048, "ny": 2048, "amp": 0.1, "beta": 5.0, "types": "DDNN", "cycle": "fp64", "tol": 1e-9},
        # rows longer than a 256-thread line solve, with the flexible GMRES outer iteration, as for the benchmark's 8192-cell rows
        {"name": "solve 8192x512 fp32 fgmres", "kind": "solve", "nx": 8192, "ny": 512, "amp": 0.05, "beta": 3.0, "types": "DDNN", "cycle": "fp32", "tol": 1e-9, "krylov": "fgmres"},
        # the benchmark's headline: many uneven problems at once, FP32 cycles (sizes 32..1024 as in its mix)
        {"name": "batch 256 fp32", "kind": "batch", "n": 256, "lo": 32, "hi": 1024, "cycle": "fp32", "tol": 1e-10},
        # a small ensemble in FP64 of odd and even sizes
        {"name": "batch 24 fp64 odd", "kind": "batch", "n": 24, "lo": 33, "hi": 400, "cycle": "fp64", "tol": 1e-10, "odd": True},
        # divergence cleaning with the fast solver on a stretched grid: fluxes up, solve, corrected in place
        {"name": "project krylov 500x300", "kind": "project", "nx": 500, "ny": 300, "amp": 0.1, "beta": 4.0, "driver": "krylov"},
        # the reference's deferred-correction driver on a large grid, red-black smoother
        {"name": "dc cycles 1024x1024", "kind": "cycles", "nx": 1024, "ny": 1024, "amp": 0.0, "beta": 0.0, "types": "DDNN", "driver": "dc", "tol": 1e-9},
        # the reference's projection step: fmg with all-Neumann sides, smoothing 8/8/8, 10 cycles
        {"name": "project fmg 256x256", "kind": "project", "nx": 256, "ny": 256, "amp": 0.05, "beta": 1.0, "driver": "fmg"},
        # a caller of the reference: one call on host arrays, everything in it
        {"name": "dropin dc vcycle 256x256", "kind": "dropin", "nx": 256, "ny": 256, "amp": 0.0, "beta": 0.0, "types": "DDDD", "cycles": 10},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _halving(rng, lo, hi):
    """A size that halves down to 8..15 cells: the reference's drivers coarsen 2 x 2 as far as the size halves."""
    return int(rng.choice([m << k for m in range(8, 16) for k in range(9) if lo <= m << k <= hi]))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "batch", "cycles", "project", "dropin"])
    if kind == "solve":
        types = rng.choice(["DDNN", "DDND", "DNND", "DDDD"])
        nx, ny = _log_int(rng, 32, 2048), _log_int(rng, 32, 2048)
        if types == "DDDD":  # rows coarsen by halving only: a user takes a size that does
            ny = 16 * max(2, ny // 16)
        case = {"nx": nx, "ny": ny, "amp": round(rng.uniform(0.0, 0.1), 3), "beta": round(rng.uniform(0.0, 4.0), 3), "types": types,
                "cycle": rng.choice(["fp64", "fp32"]), "tol": 1e-9 if max(nx, ny) > 1024 else 1e-10}
        if rng.random() < 0.2:
            case["krylov"] = "fgmres"
    elif kind == "batch":
        case = {"n": _log_int(rng, 8, 160), "lo": rng.choice([32, 33, 64]), "hi": _log_int(rng, 128, 1024), "cycle": rng.choice(["fp64", "fp32"]), "tol": 1e-10}
        if rng.random() < 0.5:
            case["odd"] = True
    elif kind == "cycles":  # the reference's drivers converge on gentle maps only
        n = _halving(rng, 32, 1024)
        case = {"nx": n, "ny": n, "amp": 0.0, "beta": 0.0, "types": rng.choice(["DDNN", "DDDD"]), "driver": "dc", "tol": 1e-9}
    elif kind == "project":
        if rng.random() < 0.5:
            n = _halving(rng, 32, 384)
            case = {"nx": n, "ny": n, "amp": round(rng.uniform(0.0, 0.05), 3), "beta": round(rng.uniform(0.0, 1.0), 3), "driver": "fmg"}
        else:
            case = {"nx": _log_int(rng, 32, 1024), "ny": _log_int(rng, 32, 1024), "amp": round(rng.uniform(0.0, 0.1), 3), "beta": round(rng.uniform(0.0, 4.0), 3), "driver": "krylov"}
    else:
        n = _halving(rng, 32, 768)
        case = {"nx": n, "ny": n, "amp": 0.0, "beta": 0.0, "types": rng.choice(["DDNN", "DDDD"]), "cycles": rng.randint(3, 12)}
    case["kind"] = kind
    return case


# ---- problems ------------------------------------------------------------------------------------------------------------------


def _bc(types):
    return G.BoundaryConditions.uniform(tuple(TYPE[t] for t in types))


def _shape(nx, ny):
    return SimpleNamespace(nx=nx, ny=ny, dx=1.0 / nx, dy=1.0 / ny)


def _map(amp, beta):
    return capi.Mapping(capi.MAP_WARPED, amp, beta, 0.0, 0.0)


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


def _rhs(nx, ny, amp, beta, gen):
    """-J (2 pi^2 sin(a x) cos(b y) + 1e-2 N(0, 1)) at the cell centres, a and b within 20 % of pi; float64 on the GPU."""
    dev = _device()
    a, b = (math.pi * (0.8 + 0.4 * torch.rand(2, generator=gen, device=dev, dtype=torch.float64))).tolist()
    s = (torch.arange(nx, device=dev, dtype=torch.float64) + 0.5) / nx
    t = ((torch.arange(ny, device=dev, dtype=torch.float64) + 0.5) / ny)[:, None]
    x = s + amp * torch.sin(2 * math.pi * s) * torch.sin(2 * math.pi * t)
    y = torch.expm1(beta * t) / math.expm1(beta) if beta else t
    J = (1.0 + amp * 2 * math.pi * torch.cos(2 * math.pi * s) * torch.sin(2 * math.pi * t)) * (beta * torch.exp(beta * t) / math.expm1(beta) if beta else 1.0)
    noise = torch.randn(ny, nx, generator=gen, device=dev, dtype=torch.float64)
    return -J * (2 * math.pi ** 2 * torch.sin(a * x) * torch.cos(b * y) + 1e-2 * noise)


def _sizes(case):
    """The problems of a batch: sizes log-uniform in [lo, hi] (multiples of 16 unless "odd"), mappings with
    beta up to 5 and amp up to 0.1, all-Dirichlet or Dirichlet xi / Neumann eta sides.  Of the case alone, not of the seed."""
    rng = np.random.default_rng(1000 * case["n"] + case["lo"] + 7 * case["hi"])
    probs = []
    for _ in range(case["n"]):
        nx, ny = (int(round(math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]))))) for _ in range(2))
        types = "DDDD" if rng.uniform() < 0.5 else "DDNN"
        if not case.get("odd"):
            nx, ny = 16 * max(2, round(nx / 16)), 16 * max(2, round(ny / 16))
        elif types == "DDDD":  # rows coarsen by halving only: a user takes a size that does
            ny = 16 * max(2, round(ny / 16))
        probs.append((nx, ny, float(rng.uniform(0.0, 0.1)), float(rng.uniform(0.0, 5.0)), types))
    return probs


def _flux(nx, ny, gen):
    """Smooth face fluxes with random amplitudes and no net outflow (the all-Neumann solve needs that)."""
    dev = _device()
    dx, dy = 1.0 / nx, 1.0 / ny
    c = (0.5 + torch.rand(4, generator=gen, device=dev, dtype=torch.float64)).tolist()
    ar = lambda n: torch.arange(n, device=dev, dtype=torch.float64)  # noqa: E731
    xn, yc, xc, yn = ar(nx + 1) * dx, ((ar(ny) + 0.5) * dy)[:, None], (ar(nx) + 0.5) * dx, (ar(ny + 1) * dy)[:, None]
    xf = c[0] * torch.sin(3 * xn) * torch.cos(2 * yc) + 0.3 * c[1] * torch.cos(5 * yc) * xn ** 2
    yf = c[2] * torch.cos(4 * xc) * torch.sin(yn) - 0.2 * c[3] * yn * torch.sin(2 * xc)
    net = (xf[:, -1] - xf[:, 0]).sum() * dy + (yf[-1] - yf[0]).sum() * dx
    return (xf - net * xn).cpu().numpy(), yf.cpu().numpy()


class _Field:
    """A resident field of a solver as an object that torch reads in place; it keeps the solver alive."""

    def __init__(self, solver, which, w, h):
        ptr, pitch = ctypes.POINTER(ctypes.c_double)(), ctypes.c_int(0)
        if capi.lib.mgp_solver_field(solver._h, which, ctypes.byref(ptr), ctypes.byref(pitch)) != capi.MGP_OK:
            raise RuntimeError("mgp_solver_field")
        self.solver = solver
        first = ctypes.cast(ptr, ctypes.c_void_p).value + 8 * (pitch.value + 32)
        self.__cuda_array_interface__ = {"shape": (h, w), "strides": (8 * pitch.value, 8), "typestr": "<f8", "data": (first, False), "version": 2}


def _view(solver, which, w, h):
    return torch.as_tensor(_Field(solver, which, w, h), device="cuda")


# ---- the measured passes -------------------------------------------------------------------------------------------------------


def prepare(case, seed):
    gen, kind = _generator(seed), case["kind"]
    if kind in ("solve", "cycles"):
        nx, ny, amp, beta = case["nx"], case["ny"], case["amp"], case["beta"]
        if kind == "solve":
            krylov = capi.KRYLOV_FGMRES if case.get("krylov") == "fgmres" else capi.KRYLOV_AUTO
            s = capi.Solver(_shape(nx, ny), _bc(case["types"]), method=METHOD[case["cycle"]], mapping=_map(amp, beta), krylov=krylov)
        else:
            s = capi.Solver(_shape(nx, ny), _bc(case["types"]), method=capi.METHOD_DC_VCYCLE, ordering=capi.ORDER_RB, mapping=_map(amp, beta))
        s.set_rhs(_rhs(nx, ny, amp, beta, gen).cpu().numpy())
        return {"case": case, "solver": s}
    if kind == "batch":
        probs = _sizes(case)
        b = capi.Batch([_shape(p[0], p[1]) for p in probs], [_bc(p[4]) for p in probs], mappings=[_map(p[2], p[3]) for p in probs], method=METHOD[case["cycle"]])
        b.set_tuning(capi.load_tuning())
        for k, p in enumerate(probs):
            b.set_rhs(k, _rhs(*p[:4], gen).cpu().numpy())
        phi = np.empty(sum(p[0] * p[1] for p in probs))
        phi.fill(0.0)
        at = np.cumsum([0] + [p[0] * p[1] for p in probs])
        return {"case": case, "batch": b, "phi": phi, "into": [phi[at[k]:].ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for k in range(len(probs))]}
    if kind == "project":
        nx, ny = case["nx"], case["ny"]
        xf, yf = _flux(nx, ny, gen)
        bc = G.BoundaryConditions((G.BCTYPE_NEUM,) * 4, (G.BCMODE_NONUNIFORM,) * 4, tuple(np.ascontiguousarray(a) for a in (xf[:, 0], xf[:, -1], yf[0], yf[-1])))
        if case["driver"] == "fmg":
            s = capi.Solver(_shape(nx, ny), bc, method=capi.METHOD_FMG, ordering=capi.ORDER_MC, smooth_down=8, smooth_up=8, smooth_bottom=8, mapping=_map(case["amp"], case["beta"]))
        else:
            s = capi.Solver(_shape(nx, ny), bc, method=capi.METHOD_KRYLOV_MG, mapping=_map(case["amp"], case["beta"]))
        return {"case": case, "solver": s, "flux": (xf, yf)}
    nx, ny = case["nx"], case["ny"]
    return {"case": case, "geo": G.mapped_geometry(nx, ny, case["amp"], case["beta"]), "bc": _bc(case["types"]),
            "rhs": _rhs(nx, ny, case["amp"], case["beta"], gen).cpu().numpy(), "phi": G.new_phi(nx, ny)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("solve", "cycles"):
        s = state["solver"]
        iters, outcome = s.solve_fast(case["tol"], MAXITERS)
        if outcome != capi.CONVERGED:
            raise RuntimeError("not converged: outcome %d after %d iterations" % (outcome, iters))
        return _view(s, 0, case["nx"], case["ny"])
    if kind == "batch":
        b = state["batch"]
        iters, outcomes = b.solve(case["tol"], MAXITERS)
        if (outcomes != capi.CONVERGED).any():
            raise RuntimeError("%d problems not converged" % (outcomes != capi.CONVERGED).sum())
        for k, to in enumerate(state["into"]):
            if capi.lib.mgp_batch_get_phi(b._h, ctypes.c_int(k), to) != capi.MGP_OK:
                raise RuntimeError("mgp_batch_get_phi")
        return state["phi"]
    if kind == "project":
        s = state["solver"]
        s.set_flux(*state["flux"])
        if case["driver"] == "fmg":
            s.project(1e-30, 10)  # the reference's workflow: 10 cycles, whatever the residual
        elif s.project(1e-10, MAXITERS)[3] != capi.CONVERGED:
            raise RuntimeError("projection not converged")
        nx, ny = case["nx"], case["ny"]
        return {"xflux": _view(s, 2, nx + 1, ny), "yflux": _view(s, 3, nx, ny + 1)}
    phi, _, relres, _, _ = capi.vcycle(1, state["geo"], state["bc"], 1, 1e-30, case["cycles"], state["phi"], state["rhs"], zerophi=True, ordering=capi.ORDER_RB)
    return {"phi": phi[1:-1, 1:-1], "relres": relres}


def work(case):
    """Of one pass: right-hand sides (or fluxes) and face metrics read once, solutions (or fluxes) written once, in FP64; one
    evaluation of the 9-point operator (41 operations a cell), without which no solution is known to be one."""
    kind = case["kind"]
    if kind == "batch":
        probs = [p[:2] for p in _sizes(case)]
    else:
        probs = [(case["nx"], case["ny"])]
    size, flops = 0, 0
    for nx, ny in probs:
        metrics = 2 * (nx + 1) * ny + 2 * nx * (ny + 1)
        fields = (nx + 1) * ny * 2 + nx * (ny + 1) * 2 if kind == "project" else 2 * nx * ny
        size += 8 * (metrics + fields + (nx * ny if kind in ("cycles", "dropin") else 0))
        flops += 41 * nx * ny
    return {"bytes": size, "flops": flops}


# ---- the same in 64 bits, by a direct solve in plain torch ----------------------------------------------------------------------


def _metrics(nx, ny, amp, beta, dev):
    """J g^11 and J g^12 on the x faces (ny, nx + 1), J g^21 and J g^22 on the y faces (ny + 1, nx)."""
    def at(s, t):
        w = 2 * math.pi
        xs = 1 + amp * w * torch.cos(w * s) * torch.sin(w * t)
        xt = amp * w * torch.sin(w * s) * torch.cos(w * t)
        yt = (beta * torch.exp(beta * t) / math.expm1(beta) if beta else torch.ones_like(t)) + 0 * s
        J = xs * yt
        return (xt * xt + yt * yt) / J, -(xs * xt) / J, xs * xs / J

    ar = lambda n: torch.arange(n, device=dev, dtype=torch.float64)  # noqa: E731
    sc, tc, sn, tn = (ar(nx) + 0.5) / nx, ((ar(ny) + 0.5) / ny)[:, None], ar(nx + 1) / nx, (ar(ny + 1) / ny)[:, None]
    g11, g12, _ = at(sn, tc)
    _, g21, g22 = at(sc, tn)
    return g11, g12, g21, g22


def _extrapolate(p, dim):
    """One more value on either side along dim, quadratically from three."""
    n = p.shape[dim]
    a = lambda k: p.narrow(dim, k, 1)  # noqa: E731
    return torch.cat([3 * (a(0) - a(1)) + a(2), p, 3 * (a(n - 1) - a(n - 2)) + a(n - 3)], dim)


def _ghosts(p, dim, lo, hi):
    """Homogeneous Dirichlet ghosts of third order (a Neumann side's are not used)."""
    n = p.shape[dim]
    a = lambda k: p.narrow(dim, k, 1)  # noqa: E731
    g = lambda k0, k1, k2: -3 * a(k0) + a(k1) - a(k2) / 5  # noqa: E731
    return torch.cat([g(0, 1, 2) if lo == "D" else 0 * a(0), p, g(n - 1, n - 2, n - 3) if hi == "D" else 0 * a(0)], dim)


def _gradient(p, met, types, nx, ny):
    """J grad p on the faces, for p of shape (..., ny, nx), with the operator's closures at the sides."""
    g11, g12, g21, g22 = met
    ex, ey = _extrapolate(p, -1), _extrapolate(p, -2)
    gx, gy = _ghosts(p, -1, types[0], types[1]), _ghosts(p, -2, types[2], types[3])
    # extrapolated values around the grid; a corner is the mean of its extrapolations along x and along y, each from two
    # extrapolated values and a ghost
    q = _extrapolate(ex, -2)
    for j, j1, j2 in ((0, 1, 2), (-1, -2, -3)):
        for i, i1, i2 in ((0, 1, 2), (-1, -2, -3)):
            q[..., j, i] = 0.5 * (3 * (ey[..., j, i] - ey[..., j, i1]) + gy[..., j, i2] + 3 * (ex[..., j, i] - ex[..., j1, i]) + gx[..., j2, i])
    dy = q[..., 2:, :] - q[..., :-2, :]          # (ny, nx + 2)
    dx = q[..., :, 2:] - q[..., :, :-2]          # (ny + 2, nx)
    xf = g11 * (gx[..., 1:] - gx[..., :-1]) * nx + 0.25 * g12 * (dy[..., 1:] + dy[..., :-1]) * ny
    yf = g22 * (gy[..., 1:, :] - gy[..., :-1, :]) * ny + 0.25 * g21 * (dx[..., 1:, :] + dx[..., :-1, :]) * nx
    for side, f in zip(types, (xf[..., 0], xf[..., -1], yf[..., 0, :], yf[..., -1, :])):
        if side == "N":
            f.zero_()
    return xf, yf


def _divergence(xf, yf, nx, ny):
    return (xf[..., 1:] - xf[..., :-1]) * nx + (yf[..., 1:, :] - yf[..., :-1, :]) * ny


class _Direct:
    """The operator's matrix, block tridiagonal in blocks of two lines (the last may have three), factored by blocks."""

    def __init__(self, nx, ny, amp, beta, types):
        self.nx, self.ny, self.types, self.dev = nx, ny, types, _device()
        self.met = _metrics(nx, ny, amp, beta, self.dev)
        self.pinned = types == "NNNN"  # known up to a constant: the last cell's value is set to 0
        self.turn = nx > ny            # lines along the shorter side
        n, lines = (ny, nx) if self.turn else (nx, ny)
        coef = torch.zeros(lines, n, 5, 5, device=self.dev, dtype=torch.float64)  # of the value at (line + a - 2, i + b - 2)
        ar = torch.arange
        for a in range(5):
            for b in range(5):
                p = torch.zeros(ny, nx, device=self.dev, dtype=torch.float64)
                p[a::5, b::5] = 1.0
                v = self.apply(p)
                v = v.T if self.turn else v
                la, lb = (b, a) if self.turn else (a, b)
                oj = (la - ar(lines, device=self.dev) + 2) % 5
                oi = (lb - ar(n, device=self.dev) + 2) % 5
                coef[ar(lines, device=self.dev)[:, None], ar(n, device=self.dev)[None], oj[:, None], oi[None]] = v
        if self.pinned:
            coef[-1, -1] = 0.0
            coef[-1, -1, 2, 2] = 1.0
        cuts = list(range(0, lines - 1, 2))
        self.blocks = [(j, cuts[k + 1] if k + 1 < len(cuts) else lines) for k, j in enumerate(cuts)]
        self.n = n
        pick = lambda r, c: self._block(coef, r, c)  # noqa: E731
        self.lu, self.up, self.low = [], [], []
        for k, r in enumerate(self.blocks):
            D = pick(r, r)
            if k:
                self.low.append(pick(r, self.blocks[k - 1]))
                D = D - self.low[-1] @ self.up[-1]
            self.lu.append(torch.linalg.lu_factor(D))
            if k + 1 < len(self.blocks):
                self.up.append(torch.linalg.lu_solve(*self.lu[-1], pick(r, self.blocks[k + 1])))

    def _block(self, coef, r, c):
        n, ar = self.n, torch.arange(self.n, device=self.dev)
        M = torch.zeros((r[1] - r[0]) * n, (c[1] - c[0]) * n, device=self.dev, dtype=torch.float64)
        for j in range(*r):
            for q in range(*c):
                if abs(q - j) > 2:
                    continue
                for b in range(-2, 3):
                    i = ar[max(0, -b):n - max(0, b)]
                    M[(j - r[0]) * n + i, (q - c[0]) * n + i + b] = coef[j, i, q - j + 2, b + 2]
        return M

    def apply(self, p):
        return _divergence(*_gradient(p, self.met, self.types, self.nx, self.ny), self.nx, self.ny)

    def _once(self, f):
        f = f.T if self.turn else f
        f = f.reshape(-1).clone()
        if self.pinned:
            f[-1] = 0.0
        parts, n = [], self.n
        for k, r in enumerate(self.blocks):
            g = f[r[0] * n:r[1] * n, None]
            if k:
                g = g - self.low[k - 1] @ parts[-1]
            parts.append(torch.linalg.lu_solve(*self.lu[k], g))
        for k in range(len(self.blocks) - 2, -1, -1):
            parts[k] = parts[k] - self.up[k] @ parts[k + 1]
        p = torch.cat(parts).reshape(-1, n)
        return p.T if self.turn else p

    def solve(self, f):
        p = self._once(f)
        for _ in range(2):
            p = p + self._once(f - self.apply(p))
        return p.contiguous()


def _direct_cost(nx, ny):
    n, lines = min(nx, ny), max(nx, ny)
    return lines / 2 * (2.0 * n) ** 3


def exact(case, seed):
    gen, kind, limit = _generator(seed), case["kind"], 3e11
    if kind == "batch":  # one array of all solutions: too many problems to solve directly
        return None
    nx, ny, amp, beta = case["nx"], case["ny"], case["amp"], case["beta"]
    if kind == "dropin" or _direct_cost(nx, ny) > limit:  # some cycles of an iteration; or too large
        return None
    if kind == "project":
        if case["driver"] == "fmg":  # 10 cycles of an iteration
            return None
        xf, yf = (torch.as_tensor(a, device=_device()) for a in _flux(nx, ny, gen))
        d = _Direct(nx, ny, amp, beta, "NNNN")
        gx, gy = _gradient(d.solve(_divergence(xf, yf, nx, ny)), d.met, "NNNN", nx, ny)
        return {"xflux": xf - gx, "yflux": yf - gy}
    return _Direct(nx, ny, amp, beta, case["types"]).solve(_rhs(nx, ny, amp, beta, gen))
