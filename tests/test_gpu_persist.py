"""Resident CG (diagonal preconditioner, one launch per solve) against the
launch chain, bit for bit.

The resident solve adds the same row sums and partial sums in the same order
as the chain (XCAL_NO_PERSIST=1 at mesh creation), so fields, residuals and
iteration counts are equal.  Sizes sit at the edges of its tiles: 64-row
groups, one workgroup of 512 rows (no meeting between workgroups), a second
one, two rows per thread, the most it takes (256 workgroups, 262 144 rows), and
more.  The mesh's counts say which form ran."""
import fcntl
import glob
import struct

import numpy as np
import pytest

from conftest import cavity_case

pytestmark = pytest.mark.gpu


def _mesh(x, shape):
    if len(shape) == 2:
        nx, ny = shape
        return x.mesh.block_mesh_2d(
            [(0.0, 0.0, 0.0), (1.0, 0.0, 0.0), (0.0, 1.0, 0.0), (1.0, 1.0, 0.0)],
            [(1, 2, nx), (3, 4, nx), (1, 3, ny), (2, 4, ny)], [(1, 2, 3, 4)],
            [("bottom", [1]), ("top", [2]), ("left", [3]), ("right", [4])])
    return x.mesh.box3d(*shape, jitter=0.1)


def _solve(x, mesh, prec, monkeypatch, **env):
    """Two pressure-like CG solves (Jacobi, singular-free by a fixed patch) and
    the mesh's resident counts."""
    A, H = x._abi, x.hip
    ctx = x.api._context(0)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    dm = H.DeviceMesh(ctx, mesh)
    for k in env:
        monkeypatch.delenv(k)
    rng = np.random.default_rng(5)
    g = H.Field(dm, A.FACE_SCALAR).upload(0.5 + rng.random(mesh.n_faces))
    s = H.Field(dm, A.CELL_SCALAR).upload(rng.standard_normal(mesh.n_cells))
    eq = H.Equation(dm, False)
    terms = [(A.LAPLACIAN_LINEAR, -1, g)]
    bcs = A.bc_array([(A.BC_DIRICHLET if i == 0 else A.BC_ZEROGRADIENT, i, 0.0)
                      for i in range(len(mesh.patch_names))])
    setup = A.SolverSetupC(A.SOLVER_CG, A.PRECON_JACOBI, prec, 400, 1e-7, 1.0, 1e-14, 1e-8, 1e-4,
                           0, 0.0)
    out = []
    for _ in range(2):  # the second solve starts where the first ended
        phi = H.Field(dm, A.CELL_SCALAR).upload(rng.standard_normal(mesh.n_cells))
        eq.discretise(terms, [(s, 1)])
        eq.apply_bcs(terms, bcs, phi)
        eq.precond_update(A.PRECON_JACOBI)
        n, res, rc = eq.solve(setup, phi)
        out.append((n, res, rc, phi.download()))
    return out, dm.resident()


def _same(a, b):
    """Equal solves; the second side ran by launches alone."""
    assert len(a[0]) == len(b[0])
    assert b[1] == (0, 0, 0, 0)
    for u, v in zip(a[0], b[0]):
        assert u[:3] == v[:3]
        assert np.array_equal(u[3], v[3])


@pytest.mark.parametrize("shape", [(1, 1), (5, 1), (8, 8), (13, 5), (32, 16), (27, 19), (64, 16),
                                   (131, 67), (300, 117), (511, 129), (11, 13, 9), (512, 511),
                                   (512, 512), (513, 512), (600, 450)])
@pytest.mark.parametrize("prec", ["fp64", "fp32-ir"])
def test_resident_cg_equals_launch_chain(x, monkeypatch, shape, prec):
    mesh = _mesh(x, shape)
    p = {"fp64": x._abi.PREC_FP64, "fp32-ir": x._abi.PREC_FP32_IR}[prec]
    a = _solve(x, mesh, p, monkeypatch)
    _same(a, _solve(x, mesh, p, monkeypatch, XCAL_NO_PERSIST="1"))
    wgs, solves, given_up, refused = a[1]
    n, k = mesh.n_cells, 1 if mesh.n_cells <= 64 * 512 else 2  # rows per thread
    if n <= 1 << 18:
        assert wgs == -(-n // (512 * k)) and solves >= 2 and given_up == refused == 0
    else:
        assert a[1] == (0, 0, 0, 0)


@pytest.mark.parametrize("shape", [(27, 19), (131, 67)])
def test_resident_cg_gives_up_to_launch_chain(x, monkeypatch, shape):
    """With no time to wait, the first resident solve gives up (some workgroup
    of some meeting comes first); this solve and those after it run by launches
    and the results are the same."""
    mesh = _mesh(x, shape)
    a = _solve(x, mesh, x._abi.PREC_FP64, monkeypatch, XCAL_PERSIST_WAIT_US="0")
    _same(a, _solve(x, mesh, x._abi.PREC_FP64, monkeypatch, XCAL_NO_PERSIST="1"))
    assert a[1][1:] == (1, 1, 0)


def test_resident_cg_without_room_runs_the_launch_chain(x, monkeypatch):
    """Compute units that another process holds (a lock on the device's file,
    taken here through an open file of the test's own) are not waited for."""
    mesh = _mesh(x, (131, 67))
    free = _solve(x, mesh, x._abi.PREC_FP64, monkeypatch)
    assert free[1][1:] == (2, 0, 0)
    files = [open(f, "r+b") for f in glob.glob("/dev/shm/xcal-resident-*")]
    assert files
    for f in files:
        fcntl.fcntl(f, fcntl.F_OFD_SETLK, struct.pack("hhqqi4x", fcntl.F_WRLCK, 0, 0, 64, 0))
    held = _solve(x, mesh, x._abi.PREC_FP64, monkeypatch)
    for f in files:
        f.close()
    assert held[1][1:] == (0, 0, 2)
    _same(free, _solve(x, mesh, x._abi.PREC_FP64, monkeypatch, XCAL_NO_PERSIST="1"))
    for u, v in zip(free[0], held[0]):
        assert u[:3] == v[:3] and np.array_equal(u[3], v[3])


def _batch(x, sizes, prec, monkeypatch, **env):
    api, H = x.api, x.hip
    ctx = api._context(0)
    ms = [x.mesh.cavity2d(n) for n in sizes]
    model, config = cavity_case(api, ms[0], iterations=8, precon="Jacobi", rtol_p=1e-3,
                                precision_p=prec)
    setup = api.simple_setup(model, config, pref=0.0)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    dm = H.DeviceMesh.batch(ctx, ms)
    for k in env:
        monkeypatch.delenv(k)
    sim = H.Simple(dm, setup)
    sim.set_case_nu(np.linspace(0.0025, 0.01, len(ms)))
    out = sim.run_batch(8)
    return out, sim.get("U"), sim.get("p"), dm.resident()


def _same_batch(a, b):
    (oa, Ua, pa, _), (ob, Ub, pb, counts) = a, b
    assert counts == (0, 0, 0, 0)
    assert oa["done"] == ob["done"] == 8
    assert np.array_equal(oa["krylov_iters"], ob["krylov_iters"])
    assert np.array_equal(oa["residuals"], ob["residuals"])
    assert np.array_equal(Ua, Ub) and np.array_equal(pa, pb)


# the last two: 256 workgroups of one case each, and one case more than fits
@pytest.mark.parametrize("sizes", [(5,), (12, 40, 16, 23), (90, 33, 64, 8, 150), (4,) * 256,
                                   (4,) * 257])
@pytest.mark.parametrize("prec", ["fp64", "fp32-ir"])
def test_resident_batch_cg_equals_launch_chain(x, monkeypatch, sizes, prec):
    a = _batch(x, sizes, prec, monkeypatch)
    _same_batch(a, _batch(x, sizes, prec, monkeypatch, XCAL_NO_PERSIST="1"))
    wgs, solves, given_up, refused = a[3]
    if len(sizes) <= 256:
        assert len(sizes) <= wgs <= 256 and solves >= 8 and given_up == refused == 0
    else:
        assert a[3] == (0, 0, 0, 0)


@pytest.mark.parametrize("prec", ["fp64", "fp32-ir"])
def test_resident_batch_cg_gives_up_to_launch_chain(x, monkeypatch, prec):
    sizes = (90, 33, 64, 8, 150)
    a = _batch(x, sizes, prec, monkeypatch, XCAL_PERSIST_WAIT_US="0")
    _same_batch(a, _batch(x, sizes, prec, monkeypatch, XCAL_NO_PERSIST="1"))
    assert a[3][1:] == (1, 1, 0)
