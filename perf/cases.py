"""The work that users of this framework have it do, as cases to time.

Each case is a dict of plain values; `prepare` makes what a program holds
before the call (mesh on the device, solver object, initial fields), `run` is
one pass through the public entry points, and `exact` gives the result of the
linear-solve cases in plain torch at 64 bits.  Kinds of case:

  simple     steady laminar SIMPLE from a given start (run! on a Steady model)
  piso       transient laminar PISO steps (run! on a Transient model)
  komega     steady k-omega SIMPLE
  cavities   many 2D cavities stepped together on one batch mesh
  steps      a few k-omega step cases stepped together on one batch mesh
  serve      k-omega requests submitted to the serving engine and fetched
  pressure   one pressure equation: assembly, boundaries, DILU, CG
  transport  one scalar transport equation: assembly, boundaries, relaxation,
             preconditioner, BiCGSTAB

A run case starts every pass from its own initial fields (set, iterate, read
back), so passes do the same work.  The settings (schemes, boundary
conditions, tolerances, relaxation) are those of bench.py and the tests.
"""
from __future__ import annotations

import functools
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent


def _package():
    """The package; its folder's name holds a dot, so it is loaded by path."""
    if "xcal_amd" not in sys.modules:
        pkg = ROOT / "xcalibre.jl_amd"
        spec = importlib.util.spec_from_file_location(
            "xcal_amd", pkg / "__init__.py", submodule_search_locations=[str(pkg)])
        sys.modules["xcal_amd"] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules["xcal_amd"])
    return sys.modules["xcal_amd"]


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the reference's own CPU configuration, a 40x40 lid-driven cavity:
        # the smallest run a user makes, where launches and latency count
        dict(name="cavity_40", kind="simple", mesh="cavity", nx=40, ny=0, nz=0, order="natural",
             precision="fp64", precon="DILU", iterations=10),
        # a 3D box below the sizes where the large-mesh forms begin, odd in
        # every direction, as a mesher numbers it
        dict(name="box_37x41x29", kind="simple", mesh="box", nx=37, ny=41, nz=29, order="natural",
             precision="fp64", precon="DILU", iterations=4),
        # a mid-sized unstructured (renumbered) box with the mixed-precision
        # pressure solve
        dict(name="box_61x47x53_ir", kind="simple", mesh="box", nx=61, ny=47, nz=53,
             order="random", precision="fp32-ir", precon="DILU", iterations=4),
        # the headline workload: the 1M-cell channel in FP64
        dict(name="channel_100", kind="simple", mesh="box", nx=100, ny=100, nz=100,
             order="random", precision="fp64", precon="DILU", iterations=4),
        # transient steps on a lexicographically numbered box (structured
        # meshes come numbered so), two pressure correctors per step
        dict(name="piso_79x66x59", kind="piso", mesh="box", nx=79, ny=66, nz=59, order="natural",
             precision="fp64", precon="DILU", iterations=2),
        # a small k-omega backward-facing step with the reference example's
        # Jacobi settings
        dict(name="komega_9k", kind="komega", ratio=0.45, cells=9000, precon="Jacobi",
             iterations=5),
        # a k-omega step near the top of the serving range
        dict(name="komega_130k", kind="komega", ratio=0.37, cells=130000, precon="Jacobi",
             iterations=2),
        # parameter sweep: 256 cavities on one batch mesh, FP64
        dict(name="cavities_256", kind="cavities", cases=256, smallest=32, largest=256,
             precision="fp64", iterations=3),
        # four k-omega requests of unlike size stepped as one batch, as the
        # server steps the cases in flight
        dict(name="steps_4", kind="steps", cases=4, smallest=4000, largest=60000,
             precon="Jacobi", iterations=3),
        # requests through the serving engine: submit, wait, fetch
        dict(name="serve_3", kind="serve", cases=3, smallest=4000, largest=9000,
             precon="Jacobi", iterations=20),
        # one pressure equation solved tightly on an unstructured box
        dict(name="pressure_70", kind="pressure", nx=70, ny=71, nz=69, order="random",
             precision="fp64"),
        # one turbulence-like transport equation on a 2D step mesh
        dict(name="transport_50k", kind="transport", ratio=0.41, cells=50000, precon="DILU"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["simple", "simple", "simple", "piso", "komega", "cavities", "steps",
                       "serve", "pressure", "transport"])
    order = rng.choice(["random", "random", "natural"])
    if kind in ("simple", "piso") and rng.random() < 0.3:
        return dict(kind=kind, mesh="cavity", nx=_log(rng, 16, 260), ny=0, nz=0, order="natural",
                    precision="fp64", precon=rng.choice(["DILU", "Jacobi"]),
                    iterations=rng.randint(2, 8))
    if kind in ("simple", "piso", "pressure"):
        cells = _log(rng, 3000, 700000 if order == "random" else 300000)
        a, b = rng.uniform(0.75, 1.3), rng.uniform(0.75, 1.3)
        e = cells ** (1 / 3)
        nx, ny, nz = (max(5, int(round(v))) for v in (e * a, e * b, e / (a * b)))
        prec = rng.choice(["fp64", "fp64", "fp32-ir", "fp32-precon"])
        if kind == "pressure":
            return dict(kind=kind, nx=nx, ny=ny, nz=nz, order=order, precision=prec)
        if kind == "piso":
            prec = "fp64"
        return dict(kind=kind, mesh="box", nx=nx, ny=ny, nz=nz, order=order, precision=prec,
                    precon="DILU", iterations=rng.randint(2, 4) if order == "random" else 2)
    if kind == "transport":
        return dict(kind=kind, ratio=round(rng.uniform(0.3, 0.6), 3),
                    cells=_log(rng, 4000, 160000), precon=rng.choice(["Jacobi", "DILU"]))
    if kind == "komega":
        dilu = rng.random() < 0.3
        return dict(kind=kind, ratio=round(rng.uniform(0.3, 0.6), 3),
                    cells=_log(rng, 4000, 20000 if dilu else 160000),
                    precon="DILU" if dilu else "Jacobi", iterations=rng.randint(2, 4 - 2 * dilu))
    if kind == "cavities":
        return dict(kind=kind, cases=_log(rng, 3, 160), smallest=rng.randint(17, 40),
                    largest=rng.randint(60, 256), precision=rng.choice(["fp64", "fp32-ir"]),
                    iterations=rng.randint(2, 3))
    if kind == "steps":
        dilu = rng.random() < 0.3
        return dict(kind=kind, cases=rng.randint(2, 5), smallest=rng.randint(3500, 6000),
                    largest=_log(rng, 8000, 20000 if dilu else 80000),
                    precon="DILU" if dilu else "Jacobi", iterations=rng.randint(2, 4 - 2 * dilu))
    return dict(kind=kind, cases=rng.randint(2, 4), smallest=rng.randint(3500, 5000),
                largest=rng.randint(6000, 12000), precon="Jacobi", iterations=rng.randint(8, 24))


# ------------------------------------------------- meshes and the device
@functools.lru_cache(maxsize=1)
def _context():
    """One context for the whole program, as api.run keeps one per device."""
    return _package().hip.Context(0)


@functools.lru_cache(maxsize=4)
def _box(nx, ny, nz, order):
    """Jittered hex box, renumbered by a seeded permutation or as meshed."""
    return _package().mesh.box3d(nx, ny, nz, jitter=0.1,
                                 seed_perm=0x5EED0003 if order == "random" else 0)


@functools.lru_cache(maxsize=4)
def _cavity(n):
    return _package().mesh.cavity2d(n)


@functools.lru_cache(maxsize=8)
def _step(ratio, cells):
    """2D backward-facing step of outlet height 1 with about `cells` cells."""
    ny = max(4, int(round(math.sqrt(cells / (5.0 - ratio)))))
    low = max(1, int(round(ratio * ny)))
    return _package().mesh.backward_facing_step_2d(ratio, 1.0, 1.0, 4.0, nx_in=ny, nx_out=4 * ny,
                                                   ny_low=low, ny_up=max(1, ny - low))


def _spread(case):
    """The sizes of a batch: log-uniform quantiles from smallest to largest."""
    k, lo, hi = case["cases"], case["smallest"], case["largest"]
    return [int(round(lo * (hi / lo) ** (i / max(1, k - 1)))) for i in range(k)]


def _ratios(case):
    return [0.3 + 0.3 * ((0.37 * (i + 1)) % 1.0) for i in range(case["cases"])]


def _mesh(case):
    kind = case["kind"]
    if kind in ("komega", "transport"):
        return _step(case["ratio"], case["cells"])
    if kind == "pressure" or case["mesh"] == "box":
        return _box(case["nx"], case["ny"], case["nz"], case["order"])
    return _cavity(case["nx"])


def _meshes(case):
    x = _package()
    if case["kind"] == "cavities":
        return [x.mesh.cavity2d(m) for m in _spread(case)]
    return [_step(r, c) for r, c in zip(_ratios(case), _spread(case))]


@functools.lru_cache(maxsize=1)
def _device_mesh(key):
    """The case's mesh on the device; a program keeps it from run to run."""
    case, H = dict(key), _package().hip
    if case["kind"] in ("cavities", "steps"):
        return H.DeviceMesh.batch(_context(), _meshes(case))
    return H.DeviceMesh(_context(), _mesh(case))


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items()
                        if k not in ("name", "iterations", "precision", "precon")))


def _modes(rng, centre, amplitude):
    """1 + a few smooth modes over the domain: a developed field's variation."""
    s = np.ones(centre.shape[0])
    lo, hi = centre.min(axis=0), centre.max(axis=0)
    xi = (centre - lo) / np.maximum(hi - lo, 1e-300)
    for _ in range(4):
        k, ph = rng.integers(1, 5, centre.shape[1]), rng.uniform(0, 2 * np.pi)
        s += amplitude * rng.uniform(-1, 1) * np.sin(np.pi * (xi @ k) + ph)
    return s


def _centres(mesh):
    return np.asarray(mesh.cell_centre).reshape(mesh.n_cells, 3)


# ---------------------------------------------------------------- settings
def _models(case, mesh, nu):
    """(model, configuration, pref) of a run case on one mesh."""
    api = _package().api
    kind, its = case["kind"], case["iterations"]
    P = getattr(api, case.get("precon", "DILU"))

    def S(solver, relax, **tol):
        return api.SolverSetup(solver=solver, preconditioner=P(), convergence=1e-14, relax=relax,
                               **tol)
    schemes = {f: api.Schemes(divergence=api.Upwind) for f in ("U", "p", "k", "omega")}
    runtime = api.Runtime(iterations=its, write_interval=-1)
    hw = api.Hardware(backend=api.HIPBackend(0))
    fluid = api.Fluid(nu=nu)
    if kind in ("komega", "steps", "serve"):
        u, k_in, w_in = 1.5, 1.0, 1000.0
        model = api.Physics(domain=mesh, fluid=fluid, turbulence=api.RANS(api.KOmega))
        t = model.turbulence
        for f, v in ((model.momentum.U, [u, 0.0, 0.0]), (t.k, k_in), (t.omega, w_in),
                     (t.nut, k_in / w_in)):
            api.initialise(f, v)
        bc = dict(
            U=[api.Dirichlet("inlet", [u, 0.0, 0.0]), api.Extrapolated("outlet"),
               api.Wall("walls", [0, 0, 0]), api.Wall("top", [0, 0, 0])],
            p=[api.Neumann("inlet", 0.0), api.Dirichlet("outlet", 0.0), api.Wall("walls"),
               api.Wall("top")],
            k=[api.Dirichlet("inlet", k_in), api.Extrapolated("outlet"),
               api.KWallFunction("walls"), api.KWallFunction("top")],
            omega=[api.Dirichlet("inlet", w_in), api.Extrapolated("outlet"),
                   api.OmegaWallFunction("walls"), api.OmegaWallFunction("top")],
            nut=[api.Dirichlet("inlet", k_in / w_in), api.Extrapolated("outlet"),
                 api.NutWallFunction("walls"), api.NutWallFunction("top")])
        tol = dict(atol=1e-10)
        solvers = dict(U=S(api.Bicgstab(), 0.7, rtol=1e-2, **tol),
                       p=S(api.Cg(), 0.3, rtol=1e-3, **tol),
                       k=S(api.Bicgstab(), 0.7, rtol=1e-2, **tol),
                       omega=S(api.Bicgstab(), 0.7, rtol=1e-2, **tol))
        return model, api.Configuration(solvers=solvers, schemes=schemes, runtime=runtime,
                                        hardware=hw, boundaries=api.assign(mesh, **bc)), None
    model = api.Physics(domain=mesh, fluid=fluid)
    if kind == "cavities" or case["mesh"] == "cavity":
        walls = ("bottom", "top", "left", "right")
        bc = dict(U=[api.Wall(w, [1.0 if w == "top" else 0.0, 0, 0]) for w in walls],
                  p=[api.Wall(w) for w in walls])
        pref, rtol = 0.0, 0.1
    else:
        api.initialise(model.momentum.U, [1.0, 0.0, 0.0])
        bc = dict(U=[api.Dirichlet("inlet", [1.0, 0.0, 0.0]), api.Extrapolated("outlet"),
                     api.Wall("walls", [0.0, 0.0, 0.0])],
                  p=[api.Extrapolated("inlet"), api.Dirichlet("outlet", 0.0),
                     api.Extrapolated("walls")])
        pref, rtol = None, 1e-10
    if kind == "piso":
        model.time = api.Transient()
        schemes["U"] = api.Schemes(divergence=api.Upwind, time=api.Euler)
        runtime.time_step = 0.5 / max(case["nx"], case["ny"], case["nz"])
        solvers = dict(U=S(api.Bicgstab(), 1.0, rtol=1e-3), p=S(api.Cg(), 1.0, rtol=1e-6))
    else:
        solvers = dict(U=S(api.Bicgstab(), 0.7, rtol=0.1), p=S(api.Cg(), 0.3, rtol=rtol))
    solvers["p"].precision = case["precision"]
    return model, api.Configuration(solvers=solvers, schemes=schemes, runtime=runtime,
                                    hardware=hw, boundaries=api.assign(mesh, **bc)), pref


def _start(case, mesh, model, rng):
    """Initial fields: the model's uniform start with smooth variations."""
    c = _centres(mesh)
    U, p = model.momentum.U, model.momentum.p
    if case["kind"] == "cavities" or case.get("mesh") == "cavity":
        # a lid-driven start: a vortex of random strength, at rest at the walls
        a = rng.uniform(0.05, 0.2)
        X, Y = np.pi * c[:, 0], np.pi * c[:, 1]
        U[0], U[1] = -a * np.sin(X) ** 2 * np.sin(2 * Y), a * np.sin(2 * X) * np.sin(Y) ** 2
    else:
        U[0] *= _modes(rng, c, 0.05)
    p[:] = 0.01 * (_modes(rng, c, 1.0) - 1.0)
    t = model.turbulence
    if getattr(t, "k", None) is not None:
        for f in (t.k, t.omega, t.nut):
            f *= _modes(rng, c, 0.03)


def _nu(case, rng):
    if case["kind"] in ("simple", "piso"):
        return rng.uniform(0.8, 1.2) * (1e-2 if case["mesh"] == "cavity" else 1e-3)
    return 1e-3  # k-omega: the reference example's


# ----------------------------------------------------------------- prepare
def prepare(case, seed):
    x = _package()
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind in ("pressure", "transport"):
        return _prepare_equation(case, rng)
    H, api = x.hip, x.api
    if kind == "serve":
        meshes = _meshes(case)
        requests = []
        for mesh in meshes:
            model, config, _ = _models(case, mesh, 1e-3)
            _start(case, mesh, model, rng)
            requests.append((mesh, api.simple_setup(model, config),
                             api.turbulence_setup(model, config), model))
        return dict(case=case, server=_serve_server(case["iterations"]), requests=requests)
    dm = _device_mesh(_key(case))
    meshes = dm.mesh.cases if kind in ("cavities", "steps") else [dm.mesh]
    parts = []
    for mesh in meshes:
        model, config, pref = _models(case, mesh, _nu(case, rng))
        _start(case, mesh, model, rng)
        parts.append(model)
    setup = api.simple_setup(model, config, pref)
    fields = dict(U=np.concatenate([m.momentum.U for m in parts], axis=1),
                  p=np.concatenate([m.momentum.p for m in parts]))
    if kind in ("komega", "steps"):
        # a k-omega run starts with zero eddy viscosity on the faces, which
        # only a new solver object has: each pass makes its own, as run! does
        for f in ("k", "omega", "nut"):
            fields[f] = np.concatenate([getattr(m.turbulence, f) for m in parts])
        return dict(case=case, mesh=dm, setup=setup, fields=fields,
                    turbulence=api.turbulence_setup(model, config))
    sim = H.Simple(dm, setup)
    if kind == "cavities":
        sim.set_case_nu(1.0 / rng.uniform(50.0, 400.0, len(parts)))
    return dict(case=case, sim=sim, fields=fields)


@functools.lru_cache(maxsize=1)
def _serve_server(iterations):
    """A serving engine whose requests stop after `iterations`."""
    return _package().hip.Server(0, slots=4, max_iterations=iterations)


def _face_geometry(mesh):
    """|E_f| (over-relaxed decomposition), delta, area, (owner, neighbour) of
    the faces, 0-based; boundary faces come first."""
    nf = mesh.n_faces
    n = np.asarray(mesh.face_normal).reshape(nf, 3)
    e = np.asarray(mesh.face_e).reshape(nf, 3)
    area, delta = np.asarray(mesh.face_area), np.asarray(mesh.face_delta)
    Ef = area / np.sum(n * e, axis=1)
    own = np.asarray(mesh.face_owner).reshape(nf, 2) - 1
    return Ef, delta, area, own


def _equation_inputs(case, mesh, rng):
    """Face and cell fields of a linear-solve case (host arrays)."""
    nf = mesh.n_faces
    fc = np.asarray(mesh.face_centre).reshape(nf, 3)
    c = _centres(mesh)
    if case["kind"] == "pressure":
        # rDf = V / a_P on the faces, and div(H/a_P) of a predicted velocity
        h = (1.0 / mesh.n_cells) ** (1 / 3)
        return dict(g=0.3 * h * _modes(rng, fc, 0.1), src=_modes(rng, c, 1.0) - 1.0)
    # a recirculating divergence-free flow, an eddy viscosity, a decay rate
    # and a production field
    a = rng.uniform(0.2, 0.5)
    X, Y = np.pi * fc[:, 0] / 5.0, np.pi * fc[:, 1]
    u = np.stack([1.0 - a * np.sin(X) * np.cos(Y), a * np.cos(X) * np.sin(Y) / 5.0,
                  np.zeros(nf)], axis=1)
    n = np.asarray(mesh.face_normal).reshape(nf, 3)
    md = np.sum(u * n, axis=1) * np.asarray(mesh.face_area)
    return dict(md=md, g=1e-3 * _modes(rng, fc, 0.1), decay=2.0 * _modes(rng, c, 0.1),
                src=_modes(rng, c, 0.5), phi=_modes(rng, c, 0.1))


def _equation_bcs(case, mesh):
    """(patch, kind, value) of the equation: fixed at one end, zero gradient
    elsewhere."""
    fixed = ("outlet", 0.0) if case["kind"] == "pressure" else ("inlet", 1.0)
    return [(p, "fixed" if p == fixed[0] else "zero", fixed[1] if p == fixed[0] else 0.0)
            for p in mesh.patch_names]


RELAX = 0.7  # implicit relaxation of the transport equation


def _prepare_equation(case, rng):
    x = _package()
    A, H = x._abi, x.hip
    dm = _device_mesh(_key(case))
    mesh = dm.mesh
    h = _equation_inputs(case, mesh, rng)
    bcs = [(A.BC_DIRICHLET if k == "fixed" else A.BC_ZEROGRADIENT, mesh.patch_index(p), v)
           for p, k, v in _equation_bcs(case, mesh)]
    f = {k: H.Field(dm, A.FACE_SCALAR if k in ("g", "md") else A.CELL_SCALAR).upload(v)
         for k, v in h.items()}
    if case["kind"] == "pressure":
        terms = [(A.LAPLACIAN_LINEAR, -1, f["g"])]
        srcs = [(f["src"], -1)]
        prec = {"fp64": A.PREC_FP64, "fp32-ir": A.PREC_FP32_IR,
                "fp32-precon": A.PREC_FP32_PRECON}[case["precision"]]
        setup = A.SolverSetupC(A.SOLVER_CG, A.PRECON_DILU, prec, 2000, 1e-7, 1.0, 1e-14, 1e-10,
                               1e-6, 0, 0.0)
    else:
        terms = [(A.TIME_STEADY, 1, 1.0), (A.DIV_UPWIND, 1, f["md"]),
                 (A.LAPLACIAN_LINEAR, -1, f["g"]), (A.SI, 1, f["decay"])]
        srcs = [(f["src"], 1)]
        pre = A.PRECON_DILU if case["precon"] == "DILU" else A.PRECON_JACOBI
        setup = A.SolverSetupC(A.SOLVER_BICGSTAB, pre, A.PREC_FP64, 2000, 1e-7, RELAX, 1e-14, 1e-9,
                               1e-6, 0, 0.0)
    phi0 = h.get("phi", np.zeros(mesh.n_cells))
    return dict(case=case, eqn=H.Equation(dm, False), terms=terms, srcs=srcs, setup=setup,
                bcs=A.bc_array(bcs), fields=f, phi=H.Field(dm, A.CELL_SCALAR), phi0=phi0)


# --------------------------------------------------------------------- run
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("pressure", "transport"):
        e, phi = state["eqn"], state["phi"].upload(state["phi0"])
        e.discretise(state["terms"], state["srcs"])
        e.apply_bcs(state["terms"], state["bcs"], phi)
        if kind == "transport":
            e.relax_implicit_diagdom(phi, 0, RELAX)
        e.precond_update(state["setup"].precon)
        e.solve(state["setup"], phi)
        return phi.download()
    if kind == "serve":
        srv = state["server"]
        ids = [srv.submit(mesh, setup, m.momentum.U, m.momentum.p, turbulence=ts,
                          k0=m.turbulence.k, omega0=m.turbulence.omega, nut0=m.turbulence.nut)
               for mesh, setup, ts, m in state["requests"]]
        for i in ids:
            srv.wait(i, 0.0)
        out = [srv.fetch(i) for i in ids]
        for i in ids:
            srv.release(i)
        return out
    f = state["fields"]
    if "turbulence" in state:
        sim = _package().hip.Simple(state["mesh"], state["setup"])
        sim.set_turbulence(state["turbulence"])
    else:
        sim = state["sim"]
    sim.set_U(f["U"])
    for name in f:
        if name != "U":
            sim.set_scalar(name, f[name])
    if kind == "piso":
        sim.run_piso(case["iterations"], 2)
    elif kind in ("cavities", "steps"):
        sim.run_batch(case["iterations"])
    else:
        sim.run(case["iterations"])
    return {name: sim.get(name) for name in f if name != "nut"}


# -------------------------------------------------------------------- work
def _cells(case):
    kind = case["kind"]
    if kind == "cavities":
        return sum(m * m for m in _spread(case))
    if kind in ("steps", "serve"):
        return sum(_spread(case))
    if kind in ("komega", "transport"):
        return case["cells"]
    if case.get("mesh") == "cavity":
        return case["nx"] ** 2
    return case["nx"] * case["ny"] * case["nz"]


def work(case):
    """Bytes and flops of one pass: fields in and out, the assembly's face and
    cell streams, and per Krylov iteration one read of the matrix and its
    factors with the vectors.  The Krylov counts are those that the settings'
    tolerances take, as rates per mesh edge."""
    kind, n = case["kind"], _cells(case)
    three = kind == "pressure" or case.get("mesh") == "box"
    nnz = (7 if three else 5) * n
    matvec = 12 * nnz + 24 * n        # values, columns, x, y
    sweeps = 2 * (6 * (nnz - n) + 32 * n)   # both triangles, D, vectors
    dilu = case.get("precon", "DILU") == "DILU"
    krylov = matvec + (sweeps if dilu else 8 * n) + 64 * n
    flops = (4 if dilu else 2) * nnz + 12 * n
    edge = n ** (1 / 3) if three else math.sqrt(n / max(1, case.get("cases", 1)))
    tight = {"pressure": 1.8, "simple": 1.8 if three else 0.1, "piso": 2.2 if three else 0.3,
             "komega": 1.0, "steps": 1.0, "serve": 1.0, "cavities": 0.1, "transport": 0.2}[kind]
    its = max(4.0, tight * edge)
    if kind in ("pressure", "transport"):
        return dict(bytes=its * krylov + 150 * n, flops=its * flops + 100 * n)
    comps = 3 if three else 2
    step = (its + 2 * comps) * krylov + 1200 * n
    return dict(bytes=case["iterations"] * step + 64 * n,
                flops=case["iterations"] * ((its + 2 * comps) * flops + 400 * n))


# --------------------------------------------------------------- tolerance
def tolerance(case):
    """64-bit arithmetic, but the Krylov solves inside stop at their own
    tolerance, and a sum in another order travels through a hundred and more
    iterations and can move the stop.  Measured with the sums in another order
    or the inputs moved in their last bit: 1e-14 to 1e-12 (2e-10 at the worst
    value) for the laminar and linear-solve cases, 7e-12 (4e-10) for k-omega with
    Jacobi, 2e-5 (1e-3) for k-omega with DILU, whose loose solves take one or
    two iterations and amplify what they are given; FP32 inner solves 1.4e-11
    (7e-11) under refinement to 1e-10, and FP32's own rounding where a loose
    tolerance takes a single FP32 solve (the cavities)."""
    kind = case["kind"]
    if kind in ("komega", "steps", "serve"):
        if case["precon"] == "DILU":
            return {"rel": 1e-4, "max": 8e-3}
        return {"rel": 1e-9, "max": 1e-7}
    if case.get("precision") == "fp32-ir":
        loose = kind == "cavities" or case.get("mesh") == "cavity"
        return {"rel": 1e-5, "max": 1e-3} if loose else {"rel": 1e-9, "max": 1e-7}
    return {"rel": 1e-10, "max": 1e-8}


# ------------------------------------------------------------------- exact
def exact(case, seed):
    """The solution of a linear-solve case in 64 bits by plain torch.  The run
    cases stop inner solves at loose tolerances (0.1 for momentum), so their
    result depends on the solver's path and has no exact value."""
    if case["kind"] not in ("pressure", "transport"):
        return None
    mesh = _mesh(case)
    h = _equation_inputs(case, mesh, np.random.default_rng(seed))
    Ef, delta, area, own = _face_geometry(mesh)
    nb = mesh.n_bfaces
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def T(a):
        return torch.as_tensor(np.ascontiguousarray(a), device=dev)
    V = T(np.asarray(mesh.cell_volume))
    P, N = T(own[nb:, 0]), T(own[nb:, 1])
    g = T(h["g"][nb:] * Ef[nb:] / delta[nb:])
    md = T(h["md"][nb:]) if "md" in h else torch.zeros_like(g)
    lower, upper = -g - md.clamp(min=0), -g + md.clamp(max=0)  # a_NP, a_PN
    diag = torch.zeros_like(V)
    diag.index_add_(0, P, g + md.clamp(min=0)).index_add_(0, N, g - md.clamp(max=0))
    b = T(h["src"]) * V * (-1.0 if case["kind"] == "pressure" else 1.0)
    cells = np.asarray(mesh.boundary_cellsID) - 1
    ranges = np.asarray(mesh.patch_range).reshape(-1, 2)
    for patch, kind, value in _equation_bcs(case, mesh):
        f0, f1 = ranges[mesh.patch_index(patch)]
        f = np.arange(f0 - 1, f1)
        c = T(cells[f])
        mb = T(h["md"][f]) if "md" in h else torch.zeros(len(f), dtype=V.dtype, device=dev)
        if kind == "fixed":
            k = T(h["g"][f] * area[f] / delta[f])
            diag.index_add_(0, c, k)
            b.index_add_(0, c, (k - mb) * value)
        else:
            diag.index_add_(0, c, mb)
    phi = T(h["phi"]) if "phi" in h else torch.zeros_like(V)
    if case["kind"] == "transport":
        diag += T(h["decay"]) * V
        off = torch.zeros_like(V).index_add_(0, P, upper.abs()).index_add_(0, N, lower.abs())
        dmax = torch.maximum(diag.abs(), off) / RELAX
        b = b + (dmax - diag) * phi
        diag = dmax

    def mul(v):
        y = diag * v
        y.index_add_(0, P, upper * v[N])
        return y.index_add_(0, N, lower * v[P])

    # BiCGSTAB with a diagonal preconditioner, restarted on its true residual
    sol = phi.clone()
    target = 1e-15 * float((b - mul(sol)).norm())
    for _ in range(12):
        r = b - mul(sol)
        if float(r.norm()) <= target:
            break
        d, c0, p, goal = torch.zeros_like(r), r.clone(), r.clone(), 1e-7 * float(r.norm())
        rho = torch.dot(c0, r)
        for it in range(3000):
            q = p / diag
            v = mul(q)
            alpha = rho / torch.dot(c0, v)
            s = r - alpha * v
            t = s / diag
            w = mul(t)
            om = torch.dot(w, s) / torch.dot(w, w)
            d = d + alpha * q + om * t
            r = s - om * w
            new = torch.dot(c0, r)
            p = r + (new / rho) * (alpha / om) * (p - om * v)
            rho = new
            if it % 25 == 24 and not float(r.norm()) > goal:
                break
        if not bool(torch.isfinite(d).all()):
            break
        sol = sol + d
    return sol.cpu().numpy()
