"""Transfers through page-locked slots, and the plain copies that take their place where that memory cannot be
had: what is set is read back bit for bit, from one triangle over sizes on both sides of a
staging slot (524,256 bytes: 43,688 positions, 131,064 words) to more slots than there are, and another
mesh's positions stay as they were."""
import ctypes

import numpy as np
import pytest

import gaia_amd

from gaia_amd.detector import ContactDetector
from vbd_cases import build_gpu, multi_spec

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[True, False], ids=["page-locked", "plain"])
def ctx(gpu_ctx, request):
    gpu_ctx.page_locked_transfers(request.param)
    yield gpu_ctx
    gpu_ctx.page_locked_transfers(True)


def test_states_come_back(ctx):
    sim = build_gpu(ctx, multi_spec())
    rng = np.random.default_rng(1)
    for m in range(sim.numMeshes()):
        x, v = (rng.normal(size=(sim.meshInfo(m)[0], 3)).astype(np.float32) for _ in range(2))
        sim.setState(m, x, v)
        sim.setState(m, velocities=v + 1)
        got = sim.getState(m)
        assert np.array_equal(got[0], x) and np.array_equal(got[1], v + 1)
    sim.destroy()


@pytest.mark.parametrize("n", [3, 43688, 43689, 87377, 131065, 349505, 700001])
def test_positions_come_back(ctx, n):
    rng = np.random.default_rng(n)
    face = np.array([[0, 1, 2]], np.int32)
    first, second = rng.normal(size=(3, 3)).astype(np.float32), rng.normal(size=(n, 3)).astype(np.float32)
    cd = ContactDetector(ctx, [(first, face), (second, face)], max_query_dis=np.float32(1e-9))
    for _ in range(2):
        second = rng.normal(size=(n, 3)).astype(np.float32)
        cd.set_positions(1, second)
        assert np.array_equal(cd.positions(), np.concatenate([first, second]))
    cd.updateBVH(True)
    cd.query()
    v, f, e = cd.min_distances()
    assert all((a == np.float32(1e-9)).all() for a in (v, f, e)) and len(v) == n + 3  # no contact: the query radius
    cd.destroy()


def test_results_of_a_detector_without_meshes(gpu_ctx):
    """Before finalize there is nothing to read, which is no error until there are elements."""
    L, h, cd = gaia_amd.lib(), gpu_ctx.handle, ctypes.c_int32()
    gpu_ctx.check(L.gvbd_cd_create(h, ctypes.c_float(0.1), 8, 8, ctypes.byref(cd)))
    one = np.full(64, 7, np.int32)
    ip, fp = (one.ctypes.data_as(ctypes.POINTER(t)) for t in (ctypes.c_int32, ctypes.c_float))
    reads = [lambda: L.gvbd_cd_vf_results(h, cd.value, ip, None), lambda: L.gvbd_cd_ee_results(h, cd.value, ip, None),
             lambda: L.gvbd_cd_min_distances(h, cd.value, fp, fp, fp)]
    assert [r() for r in reads] == [0, 0, 0] and (one == 7).all()
    assert L.gvbd_cd_vf_results(h, cd.value, None, None) == 0
    tri, face = np.eye(3, dtype=np.float32).reshape(-1), np.arange(3, dtype=np.int32)
    m = ctypes.c_int32()
    gpu_ctx.check(L.gvbd_cd_add_mesh(h, cd.value, 3, tri.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), 1,
                                     face.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)), ctypes.byref(m)))
    assert all(r() != 0 for r in reads) and (one == 7).all()
    gpu_ctx.check(L.gvbd_cd_finalize(h, cd.value))
    assert [r() for r in reads] == [0, 0, 0]
    gpu_ctx.check(L.gvbd_cd_destroy(h, cd.value))
