"""Staged transfers: what is set is read back bit for bit, from one triangle over sizes on both sides of a
staging slot (524,256 bytes: 43,688 positions, 131,064 words) to more slots than there are, and another
mesh's positions stay as they were."""
import numpy as np
import pytest

from gaia_amd.detector import ContactDetector

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 43688, 43689, 87377, 131065, 349505, 700001])
def test_positions_come_back(gpu_ctx, n):
    rng = np.random.default_rng(n)
    face = np.array([[0, 1, 2]], np.int32)
    first, second = rng.normal(size=(3, 3)).astype(np.float32), rng.normal(size=(n, 3)).astype(np.float32)
    cd = ContactDetector(gpu_ctx, [(first, face), (second, face)], max_query_dis=np.float32(1e-9))
    for _ in range(2):
        second = rng.normal(size=(n, 3)).astype(np.float32)
        cd.set_positions(1, second)
        assert np.array_equal(cd.positions(), np.concatenate([first, second]))
    cd.updateBVH(True)
    cd.query()
    v, f, e = cd.min_distances()
    assert all((a == np.float32(1e-9)).all() for a in (v, f, e)) and len(v) == n + 3  # no contact: the query radius
    cd.destroy()
