"""The framework's performance cases: what a program built on it spends its time in.

Each case is one call, or the few calls of one solver step, through the public Python API of
prism_amd, on data that a user's program would have in hand: a mesh, fields, an equation, a
solver.  The sizes are those of this repository's workloads (prism_amd/cases.py), tests and
benchmark, and generic odd ones.  `listed()` names the cases, `draw()` gives more of the same
ranges, `prepare()` builds a case's state from a seed, `run()` makes one pass from the same
start each time, `exact()` gives the answer in plain numpy where a separable operator, a dense
solve or a closed form has one (the other cases need the whole discretisation on a jittered
or tetrahedral mesh, which plain numpy does not restate here).

Krylov tolerances are 1e-13 (3e-14 for the bare pressure systems, whose smooth modes magnify
a residual 1e4 times): a solve's answer is then the linear system's solution to below 1e-9,
whatever path the iteration takes.
"""
import functools
import math

import numpy as np

import prism_amd as P
from prism_amd import cases as problems
from prism_amd import output
from prism_amd.turbulence import IncompressibleKEpsilon

TOL = 1e-13
MAX_KRYLOV = 20000
EPS = 2.220446049250313e-16
SIDES = problems.SIDES


def listed():
    return [
        # The smallest call: ISolver::step on a user's own small sparse matrix, host arrays in
        # and out (the reference's solver test is a 10 x 10 system).  Launches and latency.
        dict(name="csr_step_200", kind="csr", n=200, row=7, precision="fp64", precond="none"),
        # The same on a larger matrix with scattered columns, Jacobi preconditioned, FP32 + refinement.
        dict(name="csr_step_3001_jacobi_fp32", kind="csr", n=3001, row=12, precision="fp32", precond="jacobi"),
        # 2-D Poisson with Green-Gauss gradients and a tensor coefficient, one cell thick: the
        # reference's Poisson example at the size of this repository's first workload.
        dict(name="poisson_128x128", kind="poisson", nx=128, ny=128, precision="fp64"),
        # Steady advection-diffusion on a jittered hexahedral mesh, MUSCL, FP64: the second workload.
        dict(name="advection_muscl_64", kind="advection", nx=64, ny=64, nz=64, jitter=0.2, tets=False,
             scheme="MUSCL", precision="fp64", precond="none"),
        # The same equation on a small ragged tetrahedral mesh, Jacobi preconditioned, FP32 + refinement.
        dict(name="advection_tets_17x13x11_fp32", kind="advection", nx=17, ny=13, nz=11, jitter=0.15, tets=True,
             scheme="LinearUpwind", precision="fp32", precond="jacobi"),
        # The convection-dominated setting that asks for the symmetric Gauss-Seidel preconditioner.
        dict(name="advection_sgs_48", kind="advection", nx=48, ny=48, nz=48, jitter=0.2, tets=False,
             scheme="MINMOD", precision="fp64", precond="sgs"),
        # The pressure-correction solve of the 128^3 cavity (all-Neumann, reference cell) in
        # FP32 + refinement: the largest system, what most of a SIMPLE iteration goes into.
        dict(name="pressure_128_fp32", kind="pressure", nx=128, ny=128, nz=128, precision="fp32"),
        # The same solve in FP64 (the default precision), on an odd box.
        dict(name="pressure_97x83x71", kind="pressure", nx=97, ny=83, nz=71, precision="fp64"),
        # One whole SIMPLE outer iteration of the lid-driven cavity: three momentum solves,
        # Rhie-Chow, pressure correction with two non-orthogonal correctors, field updates.
        dict(name="simple_cavity_48", kind="simple", nx=48, ny=48, nz=48, scheme="MUSCL", precision="fp64"),
        # One whole PISO time step on tetrahedra: the transient workload at a moderate size.
        dict(name="piso_tets_24_fp32", kind="piso", nx=24, ny=24, nz=24, tets=True, precision="fp32"),
        # One k-epsilon time step: velocity gradients, model fields, both transport equations.
        dict(name="kepsilon_48", kind="kepsilon", nx=48, ny=48, nz=48, jitter=0.15, tets=False),
        # The discrete adjoint's gradient with respect to a source and a diffusivity field.
        dict(name="adjoint_64", kind="adjoint", nx=64, ny=64, nz=64, jitter=0.2, corrector="none"),
    ]


def draw(rng):
    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    def box(a, b):  # three extents about one size drawn over its logarithm
        n = math.exp(rng.uniform(math.log(a), math.log(b)))
        return dict(zip(("nx", "ny", "nz"), (max(4, int(round(n * rng.uniform(0.7, 1.3)))) for _ in range(3))))

    precision = rng.choice(["fp64", "fp32"])
    kind = rng.choice(["csr", "poisson", "advection", "advection", "pressure", "pressure", "simple", "piso",
                       "kepsilon", "adjoint"])
    if kind == "csr":
        return dict(kind=kind, n=log(10, 4000), row=rng.randint(3, 15), precision=precision,
                    precond=rng.choice(["none", "jacobi"]))
    if kind == "poisson":
        return dict(kind=kind, nx=log(16, 160), ny=log(16, 160), precision=precision)
    if kind == "advection":
        precond = rng.choice(["none", "none", "jacobi", "sgs"])
        tets = rng.random() < 0.4
        return dict(kind=kind, **box(6, 26 if tets else 60), jitter=rng.choice([0.0, 0.1, 0.2]), tets=tets,
                    scheme=rng.choice(["Upwind", "LinearUpwind", "MINMOD", "MUSCL", "SMART"]), precision=precision,
                    precond=precond)
    if kind == "pressure":
        return dict(kind=kind, **box(8, 80), precision=precision)
    if kind == "simple":
        return dict(kind=kind, **box(8, 40), scheme=rng.choice(["Upwind", "LinearUpwind", "MINMOD", "MUSCL"]),
                    precision=precision)
    if kind == "piso":
        tets = rng.random() < 0.7
        return dict(kind=kind, **box(6, 20 if tets else 34), tets=tets, precision=precision)
    if kind == "kepsilon":
        tets = rng.random() < 0.4
        return dict(kind=kind, **box(6, 24 if tets else 44), jitter=rng.choice([0.0, 0.15]), tets=tets)
    return dict(kind=kind, **box(6, 50), jitter=rng.choice([0.0, 0.2]), corrector=rng.choice(["none", "over-relaxed"]))


# ------------------------------------------------------------------------ substrate ----
@functools.lru_cache(maxsize=1)
def _backend():
    return P.Backend.hip(0)


@functools.lru_cache(maxsize=3)
def _box(nx, ny, nz, jitter, tets, length):
    return P.box(nx, ny, nz, x=(0.0, length), y=(0.0, length), z=(0.0, length), jitter=jitter, seed=1, tets=tets)


# A program keeps its mesh for as long as it solves on it: so do the states of one case.
@functools.lru_cache(maxsize=3)
def _mesh(kind, nx, ny, nz, jitter=0.0, tets=False):
    if kind == "poisson":
        data = P.box(nx, ny, 1, z=(0.0, 1.0 / nx))
        bcs = {s: {"T": ("fixed", 0.0), "f": ("fixed", 0.0)} for s in SIDES[:4]}
        bcs.update({s: {"T": "empty", "f": "empty"} for s in SIDES[4:]})
        return P.Mesh(_backend(), data, bcs, [("T", "scalar", "greenGauss"), ("f", "scalar", None)])
    data = _box(nx, ny, nz, jitter, tets, 2 * math.pi if kind == "piso" else 1.0)
    if kind == "advection":
        bcs = {s: {"T": ("zero-gradient", None), "U": ("fixed", (0.0, 0.0, 0.0))} for s in SIDES}
        bcs["left"]["T"] = ("fixed", 1.0)
        fields = [("T", "scalar", None), ("U", "velocity", None)]
    elif kind == "adjoint":
        bcs = {s: {"T": ("zero-gradient", None), "U": ("fixed", (0.0, 0.0, 0.0)), "s": ("zero-gradient", None),
                   "kappa": ("zero-gradient", None)} for s in SIDES}
        bcs["left"]["T"] = ("fixed", 1.0)
        fields = [("T", "scalar", None)]
    elif kind == "pressure":
        bcs = {s: {"P": ("zero-gradient", None), "U": ("no-slip", (0.0, 0.0, 0.0))} for s in SIDES}
        fields = [("P", "pressure", None), ("U", "velocity", None)]
    elif kind == "simple":
        bcs = {s: {"U": ("no-slip", (0.0, 0.0, 0.0)), "P": ("zero-gradient", None)} for s in SIDES}
        bcs["top"]["U"] = ("fixed", (1.0, 0.0, 0.0))
        fields = [("U", "velocity", None), ("P", "pressure", None)]
    elif kind == "piso":
        bcs = {s: {"U": ("symmetry", None), "P": ("zero-gradient", None)} for s in SIDES}
        fields = [("U", "velocity", None), ("P", "pressure", None)]
    else:  # kepsilon: a box channel, sheared inflow at the left, outflow at the right
        bcs = {s: {"U": ("fixed", (0.0, 0.0, 0.0)), "k": "zero-gradient", "epsilon": "zero-gradient",
                   "nu": "zero-gradient"} for s in SIDES}
        bcs["left"].update({"U": ("fixed", (1.0, 0.0, 0.0)), "k": ("fixed", 0.01), "epsilon": ("fixed", 1e-3)})
        bcs["right"].update({"U": "outlet"})
        fields = [("U", "vector"), ("k", "scalar"), ("epsilon", "scalar"), ("nu", "scalar")]
    return P.Mesh(_backend(), data, bcs, fields)


def _solver(case):
    tol = 3e-14 if case["kind"] == "pressure" else TOL
    return P.solver.BiCGSTAB(tol=tol, precision=case["precision"], precond=case.get("precond"), max_iters=MAX_KRYLOV)


def _smooth(rng, x, y, z, modes=3, scale=math.pi):
    """A seeded smooth function of the points: a few cosines with decaying amplitudes."""
    v = np.zeros_like(x)
    for _ in range(2 * modes):
        k = rng.integers(1, modes + 1, 3)
        ph = rng.uniform(0.0, 2 * math.pi, 3)
        v += rng.standard_normal() / k.sum() * (np.cos(scale * k[0] * x + ph[0]) * np.cos(scale * k[1] * y + ph[1])
                                                * np.cos(scale * k[2] * z + ph[2]))
    return v


def _fluxes(mesh, fn):
    """Face fluxes fn(x_f) . S_f on the interior faces, zero on the boundary."""
    g = mesh.geometry()
    f, S = g["face_center"], g["face_area"]
    u = fn(f[:, 0], f[:, 1], f[:, 2])
    flux = (u[:, 0] * S[:, 0] + u[:, 1] * S[:, 1]) + u[:, 2] * S[:, 2]
    flux[g["neighbor"] < 0] = 0.0
    return flux


def _set_vector(U, comps):
    for c, v in zip((U.x, U.y, U.z), comps):
        c.values = v


# ---------------------------------------------------------------------- bare matrix ----
def _csr_inputs(case, seed):
    """A strictly diagonally dominant nonsymmetric matrix with `row` scattered off-diagonals a
    row at most, and a right-hand side."""
    n, rng = case["n"], np.random.default_rng(seed)
    cols = rng.integers(0, n, (n, case["row"]))
    vals = rng.uniform(-1.0, 0.3, (n, case["row"]))
    M = np.zeros((n, n))
    np.add.at(M, (np.repeat(np.arange(n), case["row"]), cols.ravel()), vals.ravel())
    np.fill_diagonal(M, 0.0)
    np.fill_diagonal(M, (1.05 + 0.2 * rng.random(n)) * np.abs(M).sum(axis=1) + 0.1)
    return M, rng.standard_normal(n), np.zeros(n)


def _prepare_csr(case, seed):
    M, b, x0 = _csr_inputs(case, seed)
    row, col = np.nonzero(M)
    indptr = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=case["n"]))])
    return dict(A=P.Matrix(_backend(), indptr, col, M[row, col]), b=b, x0=x0, solver=_solver(case))


def _run_csr(s):
    return s["solver"].step(s["A"], s["x0"], s["b"])


# -------------------------------------------------------------------------- Poisson ----
def _link(s, d):
    """The over-relaxed coefficient of two cells a distance d apart across a face of kappa times
    area s on an orthogonal mesh, with the guards the scheme is defined with (s / d without)."""
    return s * s / (s + EPS) * d / (d * d + EPS)


def _poisson_functions(seed):
    rng = np.random.default_rng(seed)
    a, k = rng.uniform(0.5, 1.5, 4), rng.integers(1, 4, 4)
    ph = rng.uniform(0.0, 1.0, 4)

    def wall(x, y):
        return a[0] * np.sin(math.pi * (k[0] * x + ph[0])) * np.cos(math.pi * (k[1] * y + ph[1]))

    def source(x, y):
        return 2 * math.pi ** 2 * a[1] * np.sin(math.pi * (k[2] * x + ph[2])) * np.cos(math.pi * (k[3] * y + ph[3]))

    return wall, source


def _prepare_poisson(case, seed):
    mesh = _mesh("poisson", case["nx"], case["ny"], 1)
    wall, source = _poisson_functions(seed)
    g = mesh.geometry()
    T = mesh.scalar("T", 0.0)
    T.set_face_values(wall(g["face_center"][:, 0], g["face_center"][:, 1]))
    f = mesh.scalar("f", values=source(g["cell_center"][:, 0], g["cell_center"][:, 1]))
    eqn = P.Transport(P.diffusion.Corrected(mesh.tensor("kappa", np.eye(3)), T), P.source.ConstantScalar(f))
    return dict(T=T, eqn=eqn, solver=_solver(case))


def _run_solve(s):
    s["T"].fill(0.0)
    s["solver"].solve(s["eqn"])
    return s["T"].values


def _exact_poisson(case, seed):
    nx, ny = case["nx"], case["ny"]
    hx, hy, hz = 1.0 / nx, 1.0 / ny, 1.0 / nx
    wall, source = _poisson_functions(seed)
    cx, cy = _link(hy * hz, hx), _link(hx * hz, hy)
    X, Y = (np.arange(nx) + 0.5) * hx, (np.arange(ny) + 0.5) * hy
    b = source(X[:, None], Y[None, :]) * (hx * hy * hz)
    b[0, :] += 2 * cx * wall(0.0, Y)
    b[-1, :] += 2 * cx * wall(1.0, Y)
    b[:, 0] += 2 * cy * wall(X, 0.0)
    b[:, -1] += 2 * cy * wall(X, 1.0)

    def line(n, c):  # Dirichlet walls half a cell away
        L = np.diag(np.full(n, 2.0 * c)) - np.diag(np.full(n - 1, c), 1) - np.diag(np.full(n - 1, c), -1)
        L[0, 0] = L[-1, -1] = 3.0 * c
        return np.linalg.eigh(L)

    (lx, Qx), (ly, Qy) = line(nx, cx), line(ny, cy)
    x = Qx @ ((Qx.T @ b @ Qy) / (lx[:, None] + ly[None, :])) @ Qy.T
    return np.ascontiguousarray(x.T).reshape(-1)  # cells are numbered x-fastest


# ------------------------------------------------------------------------ advection ----
def _prepare_advection(case, seed):
    mesh = _mesh("advection", case["nx"], case["ny"], case["nz"], case["jitter"], case["tets"])
    rng = np.random.default_rng(seed)
    U = problems.prescribed_velocity(mesh)
    T = mesh.scalar("T", 0.0)
    kappa = mesh.scalar("kappa", values=2e-3 * np.exp(0.3 * rng.standard_normal(mesh.n_cells)))
    eqn = P.Transport(getattr(P.convection, case["scheme"])(U, T), P.diffusion.Corrected(kappa, T))
    return dict(T=T, eqn=eqn, solver=_solver(case), keep=(U, kappa))


# ------------------------------------------------------------------------- pressure ----
def _pressure_fluxes(case, seed):
    """Random fluxes through the interior faces normal to x, y and z, as a SIMPLE iterate's mass
    imbalance: arrays over (face position along the normal, the other two cell indices)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((nx - 1, ny, nz)) / (ny * nz), rng.standard_normal((nx, ny - 1, nz)) / (nx * nz),
            rng.standard_normal((nx, ny, nz - 1)) / (nx * ny))


@functools.lru_cache(maxsize=2)
def _pressure_faces(nx, ny, nz):
    """Per normal direction: the interior faces' indices and their positions in _pressure_fluxes."""
    g = _mesh("pressure", nx, ny, nz).geometry()
    inner = np.nonzero(g["neighbor"] >= 0)[0]
    o = g["owner"][inner]
    step = g["neighbor"][inner] - o
    i, j, k = o % nx, (o // nx) % ny, o // (nx * ny)
    out = []
    for s in (1, nx, nx * ny):  # the neighbour has the larger number: owner's position is the face's
        m = step == s
        out.append((inner[m], i[m], j[m], k[m]))
    return out


def _prepare_pressure(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    mesh = _mesh("pressure", nx, ny, nz)
    D = mesh.tensor("D", 1.0 / (6 * 0.01) / nx ** 2)
    flux = np.zeros(mesh.n_faces)
    for (f, i, j, k), values in zip(_pressure_faces(nx, ny, nz), _pressure_fluxes(case, seed)):
        flux[f] = values[i, j, k]
    mdot = mesh.vector("U", (0.0, 0.0, 0.0))
    mdot.set_face_fluxes(flux)
    pp = mesh.pressure("P", 0.0)
    eqn = P.Transport(P.diffusion.Corrected(D, pp), P.source.Divergence(mdot, "-"))
    return dict(p=pp, eqn=eqn, solver=_solver(case), keep=(D, mdot))


def _run_pressure(s):
    s["p"].fill(0.0)
    s["solver"].solve(s["eqn"], n_iter=5, eps=1e-7, ref_cell=0)
    return s["p"].values


def _exact_pressure(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    d = 1.0 / (6 * 0.01) / nx ** 2
    fx, fy, fz = _pressure_fluxes(case, seed)
    b = np.zeros((nx, ny, nz))  # minus the sum of the outward fluxes
    for f, lo, hi in ((fx, np.s_[:-1, :, :], np.s_[1:, :, :]), (fy, np.s_[:, :-1, :], np.s_[:, 1:, :]),
                      (fz, np.s_[:, :, :-1], np.s_[:, :, 1:])):
        b[lo] -= f
        b[hi] += f

    def line(n, c):  # zero gradient at both ends
        L = np.diag(np.full(n, 2.0 * c)) - np.diag(np.full(n - 1, c), 1) - np.diag(np.full(n - 1, c), -1)
        L[0, 0] = L[-1, -1] = c
        return np.linalg.eigh(L)

    (lx, Qx), (ly, Qy), (lz, Qz) = (line(nx, _link(d / (ny * nz), 1.0 / nx)), line(ny, _link(d / (nx * nz), 1.0 / ny)),
                                    line(nz, _link(d / (nx * ny), 1.0 / nz)))
    lam = lx[:, None, None] + ly[None, :, None] + lz[None, None, :]
    lam[0, 0, 0] = 1.0
    t = np.tensordot(Qx.T, b, (1, 0))
    t = np.tensordot(t, Qy, (1, 0)).transpose(0, 2, 1)
    t = (t @ Qz) / lam
    t[0, 0, 0] = 0.0  # the constant, set below by the reference cell
    t = np.tensordot(Qx, t, (1, 0))
    t = np.tensordot(t, Qy.T, (1, 0)).transpose(0, 2, 1)
    t = t @ Qz.T
    return np.ascontiguousarray((t - t[0, 0, 0]).transpose(2, 1, 0)).reshape(-1)


# ---------------------------------------------------------------------------- SIMPLE ----
def _prepare_simple(case, seed):
    mesh = _mesh("simple", case["nx"], case["ny"], case["nz"])
    rng = np.random.default_rng(seed)
    a = rng.uniform(0.5, 1.0, 2)

    def vortex(x, y, z):  # divergence-free, no flow through the walls
        s, c = np.sin(math.pi * x) * np.sin(math.pi * y), np.sin(2 * math.pi * z)
        return np.stack([a[0] * s * np.sin(math.pi * x) * np.cos(math.pi * y) * (1 + a[1] * c),
                         -a[0] * s * np.cos(math.pi * x) * np.sin(math.pi * y) * (1 + a[1] * c), 0.0 * x], axis=1)

    x, y, z = mesh.geometry()["cell_center"].T
    u0 = vortex(x, y, z) + 1e-3 * rng.standard_normal((mesh.n_cells, 3))
    U = mesh.vector("U", values=u0)
    p = mesh.pressure("P", 0.0)
    nu = mesh.scalar("nu", 0.01)
    mdot = U.clone()
    conv = getattr(P.convection, case["scheme"])
    eqns = [P.Transport(conv(mdot, c), P.diffusion.Corrected(nu, c), P.source.Gradient(p, k, "-"))
            for k, c in enumerate((U.x, U.y, U.z))]
    ctl = P.algo.SIMPLEControls(_backend(), momentum_tol=TOL, pressure_tol=TOL, max_krylov_iters=MAX_KRYLOV,
                                pressure_precision=1 if case["precision"] == "fp32" else 0)
    return dict(U=U, p=p, mdot=mdot, eqns=eqns, algo=P.algo.IncompressibleSIMPLE(ctl), keep=nu, history=False,
                u0=[np.ascontiguousarray(u0[:, k]) for k in range(3)], p0=0.1 * _smooth(rng, x, y, z),
                flux0=_fluxes(mesh, vortex))


def _prepare_piso(case, seed):
    mesh = _mesh("piso", case["nx"], case["ny"], case["nz"], 0.0, case["tets"])
    rng = np.random.default_rng(seed)
    a = rng.uniform(0.5, 1.0)

    def vortex(x, y, z):
        return np.stack([a * np.sin(x) * np.cos(y) * np.cos(z), -a * np.cos(x) * np.sin(y) * np.cos(z), 0.0 * x], axis=1)

    x, y, z = mesh.geometry()["cell_center"].T
    u0 = vortex(x, y, z) + problems.solenoidal_noise(x, y, z, 1e-2, seed)
    U = mesh.vector("U", values=u0)
    p = mesh.pressure("P", 0.0)
    nu = mesh.scalar("nu", 1e-3)
    mdot = U.clone()
    flux0 = _fluxes(mesh, vortex)
    mdot.set_face_fluxes(flux0)
    dt = problems.courant_dt(mdot, 0.5)
    for c in (U.x, U.y, U.z):
        c.set_history_size(1)
    eqns = [P.Transport(P.temporal.BackwardEuler(c, dt), P.convection.LinearUpwind(mdot, c),
                        P.diffusion.Corrected(nu, c), P.source.Gradient(p, k, "-"))
            for k, c in enumerate((U.x, U.y, U.z))]
    ctl = P.algo.PISOControls(_backend(), outer_iterations=1, pressure_correction_steps=2,
                              simple=dict(momentum_tol=TOL, pressure_tol=TOL, max_krylov_iters=MAX_KRYLOV,
                                          pressure_precision=1 if case["precision"] == "fp32" else 0))
    return dict(U=U, p=p, mdot=mdot, eqns=eqns, algo=P.algo.PISO(ctl), keep=nu, history=True,
                u0=[np.ascontiguousarray(u0[:, k]) for k in range(3)], p0=0.05 * _smooth(rng, x, y, z, 2, 0.5),
                flux0=flux0)


def _run_flow(s):
    U, p, mdot = s["U"], s["p"], s["mdot"]
    _set_vector(U, s["u0"])
    p.values = s["p0"]
    mdot.set_face_fluxes(s["flux0"])
    if s["history"]:
        for c in (U.x, U.y, U.z):
            c.update_prev_time_steps()
    s["algo"].step(s["eqns"], U, mdot, p)
    return dict(u=U.x.values, v=U.y.values, w=U.z.values, p=p.values, mdot=mdot.face_fluxes())


# ------------------------------------------------------------------------- k-epsilon ----
def _prepare_kepsilon(case, seed):
    mesh = _mesh("kepsilon", case["nx"], case["ny"], case["nz"], case["jitter"], case["tets"])
    rng = np.random.default_rng(seed)
    x, y, z = mesh.geometry()["cell_center"].T
    u0 = [0.5 + y + 0.05 * _smooth(rng, x, y, z), 0.1 * np.sin(math.pi * x) + 0.05 * _smooth(rng, x, y, z),
          0.05 * _smooth(rng, x, y, z)]
    U = mesh.vector("U", values=np.stack(u0, axis=1))
    nu = mesh.scalar("nu", 1e-3)
    model = IncompressibleKEpsilon(U, U, nu, dt=0.02)
    n = mesh.n_cells
    return dict(U=U, u0=u0, model=model, keep=nu, solver=P.solver.BiCGSTAB(tol=TOL, max_iters=MAX_KRYLOV),
                k=[rng.uniform(0.009, 0.011, n) for _ in range(2)], e=[rng.uniform(9e-4, 1.1e-3, n) for _ in range(2)])


def _run_kepsilon(s):
    model = s["model"]
    k, e = model.k(), model.epsilon()
    _set_vector(s["U"], s["u0"])
    for level in range(2):  # the two previous time levels
        k.values, e.values = s["k"][level], s["e"][level]
        k.update_prev_time_steps()
        e.update_prev_time_steps()
    for eqn in model.equations():
        s["solver"].solve(eqn)
    return dict(k=k.values, epsilon=e.values, nu_t=model.turbulent_viscosity().values, pk=model.production().values,
                k_points=output.cell_to_point(k), u_points=output.cell_to_point(s["U"]))


# --------------------------------------------------------------------------- adjoint ----
def _prepare_adjoint(case, seed):
    mesh = _mesh("adjoint", case["nx"], case["ny"], case["nz"], case["jitter"])
    rng = np.random.default_rng(seed)
    n = mesh.n_cells
    x, y, z = mesh.geometry()["cell_center"].T
    U = problems.prescribed_velocity(mesh)
    T = mesh.scalar("T", values=1.0 + 0.3 * _smooth(rng, x, y, z))
    kappa = mesh.scalar("kappa", values=np.exp(np.log(1e-2) + 0.5 * rng.standard_normal(n)))
    src = mesh.scalar("s", values=rng.uniform(0.0, 1.0, n))
    diff = (P.diffusion.NonCorrected(kappa, T) if case["corrector"] == "none"
            else P.diffusion.Corrected(kappa, T, corrector=case["corrector"]))
    eqn = P.Transport(P.convection.Upwind(U, T), diff, P.source.ConstantScalar(src))
    return dict(eqn=eqn, source=src, kappa=kappa, keep=(T, U), solver=P.solver.BiCGSTAB(tol=TOL, max_iters=MAX_KRYLOV))


def _run_adjoint(s):
    J, ds, dk, _ = P.adjoint.gradient(s["eqn"], s["source"], s["kappa"], solver=s["solver"])
    return dict(J=J, ds=ds, dkappa=dk)


# ----------------------------------------------------------------------- entry points ----
_PREPARE = dict(csr=_prepare_csr, poisson=_prepare_poisson, advection=_prepare_advection, pressure=_prepare_pressure,
                simple=_prepare_simple, piso=_prepare_piso, kepsilon=_prepare_kepsilon, adjoint=_prepare_adjoint)
_RUN = dict(csr=_run_csr, poisson=_run_solve, advection=_run_solve, pressure=_run_pressure, simple=_run_flow,
            piso=_run_flow, kepsilon=_run_kepsilon, adjoint=_run_adjoint)


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    s["kind"] = case["kind"]
    return s


def run(state):
    return _RUN[state["kind"]](state)


def exact(case, seed):
    if case["kind"] == "csr":
        M, b, _ = _csr_inputs(case, seed)
        return np.linalg.solve(M, b)
    if case["kind"] == "poisson":
        return _exact_poisson(case, seed)
    if case["kind"] == "pressure":
        return _exact_pressure(case, seed)
    return None


def work(case):
    """Bytes and operations of one pass.  A Krylov solve: the iterations that unpreconditioned
    BiCGSTAB takes to 1e-13 on such a system (a multiple of the cells along an edge; a few
    dozen on a diagonally dominant matrix), each with two passes over the matrix and sixteen
    vectors.  An equation's assembly: the geometry of every face and cell, the fields and the
    matrix once."""
    kind = case["kind"]
    w = 4 if case.get("precision") == "fp32" else 8
    if kind == "csr":
        n, nnz = case["n"], case["n"] * (case["row"] + 1)
        solves, iters, equations = 1, 40, 0
    else:
        nz = case.get("nz", 1)
        tets = case.get("tets", False)
        n = case["nx"] * case["ny"] * nz * (6 if tets else 1)
        nnz = n * (5 if tets or nz == 1 else 7)
        edge = max(case["nx"], case["ny"], nz)
        per_edge = {"poisson": 3.0, "pressure": 6.0, "advection": 15.0, "simple": 8.0, "piso": 14.0, "kepsilon": 0.5,
                    "adjoint": 15.0}[kind]
        iters = per_edge * edge * (0.4 if case.get("precond") == "sgs" else 1.0)
        solves = {"piso": 2, "kepsilon": 2}.get(kind, 1)
        equations = {"simple": 6, "piso": 12, "kepsilon": 2}.get(kind, 1)
    index = 0 if kind in ("poisson", "pressure") else 2 if case.get("tets") or kind == "csr" else 0
    faces = (nnz - n) // 2
    solve_bytes = iters * (2 * (w + index) * nnz + 16 * w * n)
    solve_flops = iters * (4 * nnz + 20 * n)
    assembly_bytes = 64 * faces + 80 * n + 8 * nnz
    assembly_flops = 120 * faces + 40 * n
    return {"bytes": solves * solve_bytes + equations * assembly_bytes + 32 * n,
            "flops": solves * solve_flops + equations * assembly_flops}
