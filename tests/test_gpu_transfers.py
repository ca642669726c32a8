"""Transfers through page-locked slots, and the plain copies that take their place where that memory cannot be
had: what is set is read back bit for bit, from one triangle over sizes on both sides of a
staging slot (524,256 bytes: 43,688 positions, 131,064 words) to more slots than there are, and another
mesh's positions stay as they were."""
import numpy as np
import pytest

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
