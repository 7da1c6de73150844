"""Fields cross the C ABI renumbered, by host loops or on the device: what goes
up comes back bit for bit, per component and in the reference numbering (an
equation built from an uploaded source keeps each value in its cell's row)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1), (4, 8, 8), (3, 5, 17), (16, 16, 17),
                                   (48, 32, 32), (49153, 1, 1)])
def test_field_round_trip_in_reference_numbering(x, shape):
    A, H = x._abi, x.hip
    ctx = x.api._context(0)
    mesh = x.mesh.box3d(*shape, jitter=0.1)
    dm = H.DeviceMesh(ctx, mesh)
    rng = np.random.default_rng(1)
    # face fields last: the transfer buffer grows between the calls.  Cell or
    # face counts on both sides of 49 152, where kernels take over from host
    # loops, and just at it
    for kind in (A.CELL_SCALAR, A.CELL_VECTOR, A.CELL_TENSOR, A.FACE_SCALAR, A.FACE_VECTOR):
        f = H.Field(dm, kind)
        v = rng.standard_normal((f.ncomp, f.len))
        v[0, 0], v[-1, -1] = -0.0, np.inf
        got = f.upload(v).download().reshape(f.ncomp, f.len)
        assert np.array_equal(got.view(np.int64), v.view(np.int64))
    src = rng.standard_normal(mesh.n_cells)
    eq = H.Equation(dm, False)
    g = H.Field(dm, A.FACE_SCALAR).fill(1.0)
    eq.discretise([(A.LAPLACIAN_LINEAR, -1, g)], [(H.Field(dm, A.CELL_SCALAR).upload(src), 1)])
    assert np.array_equal(eq.download()[1], src * np.asarray(mesh.cell_volume))


def test_transfers_of_one_mesh_from_several_threads(x):
    """Uploads and downloads of different fields of one mesh at the same time,
    of lengths that make the transfer buffer grow in between: every thread gets
    its own values back."""
    from concurrent.futures import ThreadPoolExecutor

    A, H = x._abi, x.hip
    ctx = x.api._context(0)
    mesh = x.mesh.box3d(41, 40, 43, jitter=0.1)
    dm = H.DeviceMesh(ctx, mesh)
    kinds = (A.CELL_SCALAR, A.FACE_SCALAR, A.CELL_VECTOR, A.FACE_VECTOR)
    fields = [H.Field(dm, k) for k in kinds]

    def work(i):
        f, rng = fields[i], np.random.default_rng(i)
        for _ in range(12):
            v = rng.standard_normal((f.ncomp, f.len))
            if not np.array_equal(f.upload(v).download().reshape(v.shape), v):
                return False
        return True

    with ThreadPoolExecutor(len(kinds)) as ex:
        assert all(ex.map(work, range(len(kinds))))


def test_transfer_while_another_device_is_current(x):
    """A field on device 0 moves through a buffer of device 0 while a later
    context has made device 1 the thread's current one."""
    import torch

    if torch.cuda.device_count() < 2:
        pytest.skip("needs two GPUs")
    A, H = x._abi, x.hip
    mesh = x.mesh.box3d(41, 40, 43, jitter=0.1)
    dm = H.DeviceMesh(H.Context(0), mesh)
    f = H.Field(dm, A.CELL_SCALAR)
    other = H.Context(1)
    v = np.random.default_rng(4).standard_normal(f.len)
    assert np.array_equal(f.upload(v).download(), v)
    del other
