"""Lean one-workgroup DILU sweeps against level stepping, bit for bit.

On naturally numbered meshes below the cone form's size, a sweep over all
levels is one launch of one workgroup (one per case of a batch).  Rows keep
the reference's summation order and the dot products the launch form's, so
preconditioner applies, CG and BiCGSTAB solves equal those of XCAL_NO_PIPE=1
(level launches and level-stepping runs) exactly.  Shapes: level counts on
both sides of a multiple of the step padding, levels of one row up to several
steps, two and three entries per row, dependencies that need the longer LDS
ring, and long meshes above the cone form's size, whose levels are too many
for bands."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(x):
    return x.hip.Context(0)


def _mesh(x, shape):
    if shape[0] == "step":
        ny = shape[1]
        return x.mesh.backward_facing_step_2d(0.41, 1.0, 1.0, 4.0, nx_in=ny, nx_out=4 * ny,
                                              ny_low=int(0.41 * ny), ny_up=ny - int(0.41 * ny))
    if len(shape) == 2:
        nx, ny = shape
        return x.mesh.block_mesh_2d(
            [(0.0, 0.0, 0.0), (1.0, 0.0, 0.0), (0.0, 1.0, 0.0), (1.0, 1.0, 0.0)],
            [(1, 2, nx), (3, 4, nx), (1, 3, ny), (2, 4, ny)], [(1, 2, 3, 4)],
            [("bottom", [1]), ("top", [2]), ("left", [3]), ("right", [4])])
    return x.mesh.box3d(*shape, jitter=0.1, seed_perm=0)


def _system(x, A, dm, mesh, sym, seed=3):
    H = x.hip
    rng = np.random.default_rng(seed)
    nf, n = dm.mesh.n_faces, dm.n
    g = H.Field(dm, A.FACE_SCALAR).upload(0.5 + rng.random(nf))
    md = H.Field(dm, A.FACE_SCALAR).upload(0.02 * rng.standard_normal(nf))
    s = H.Field(dm, A.CELL_SCALAR).upload(rng.standard_normal(n))
    eq = H.Equation(dm, False)
    terms = [(A.LAPLACIAN_LINEAR, -1, g)] + ([] if sym else [(A.DIV_UPWIND, 1, md),
                                                            (A.SI, 1, 5.0)])
    bcs = A.bc_array([(A.BC_DIRICHLET if i == 0 else A.BC_ZEROGRADIENT, i, 0.0)
                      for i in range(len(mesh.patch_names))])
    phi = H.Field(dm, A.CELL_SCALAR).upload(rng.standard_normal(n))
    eq.discretise(terms, [(s, 1)])
    eq.apply_bcs(terms, bcs, phi)
    eq.precond_update(A.PRECON_DILU)
    return eq, phi, (g, md, s)


def _setup(A, solver, prec):
    return A.SolverSetupC(getattr(A, solver), A.PRECON_DILU, getattr(A, prec), 200, 1e-7, 1.0,
                          1e-14, 1e-9, 1e-5, 0, 0.0)


SHAPES = [(9, 8), (9, 9), (40, 1), (23, 18), (63, 37), (130, 260), (200, 255), (5, 6, 7),
          (16, 17, 18), (37, 21, 29), ("step", 24), ("step", 104), (1000, 90), (600, 12, 12)]


@pytest.mark.parametrize("shape", SHAPES)
def test_lean_sweeps_equal_level_stepping(x, A, ctx, monkeypatch, shape):
    H = x.hip
    mesh = _mesh(x, shape)
    out = []
    for off in (False, True):
        if off:
            monkeypatch.setenv("XCAL_NO_PIPE", "1")
        dm = H.DeviceMesh(ctx, mesh)
        monkeypatch.delenv("XCAL_NO_PIPE", raising=False)
        assert dm.lean_form() == ((0, 0) if off else (8192, 8192) if shape == ("step", 104)
                                  else (4096, 4096))  # the ring
        got = []
        for solver, prec in (("SOLVER_CG", "PREC_FP64"), ("SOLVER_BICGSTAB", "PREC_FP64"),
                             ("SOLVER_CG", "PREC_FP32_IR"), ("SOLVER_BICGSTAB", "PREC_FP32_IR")):
            eq, phi, _ = _system(x, A, dm, mesh, solver == "SOLVER_CG")
            z = H.Field(dm, A.CELL_SCALAR)
            eq.precond_apply(phi, z)
            n, res, rc = eq.solve(_setup(A, solver, prec), phi)
            got += [z.download(), np.array([n, rc]), np.array([res]), phi.download()]
        out.append(got)
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("shapes", [[(9, 8)], [(9, 9), (130, 40), (23, 18), (40, 1)],
                                    [("step", 24), ("step", 30)]])
def test_lean_batch_sweeps_equal_level_stepping(x, A, ctx, monkeypatch, shapes):
    H = x.hip
    ms = [_mesh(x, s) for s in shapes]
    monkeypatch.setenv("XCAL_PIPE_ROWS", "1")  # the lean body's rows per thread
    out = []
    for off in (False, True):
        if off:
            monkeypatch.setenv("XCAL_NO_PIPE", "1")
        dm = H.DeviceMesh.batch(ctx, ms)
        monkeypatch.delenv("XCAL_NO_PIPE", raising=False)
        assert dm.lean_form() == ((0, 0) if off else (4096, 4096))
        got = []
        for solver, prec in (("SOLVER_CG", "PREC_FP64"), ("SOLVER_BICGSTAB", "PREC_FP64"),
                             ("SOLVER_CG", "PREC_FP32_IR")):
            eq, phi, _ = _system(x, A, dm, ms[0], solver == "SOLVER_CG")
            its, outer, res, rc = eq.solve_batch(_setup(A, solver, prec), phi)
            got += [its, outer, res, phi.download()]
        out.append(got)
    for a, b in zip(*out):
        assert np.array_equal(a, b)
