"""Tree refit in blocks of 1,024 leaves and windows of 64 blocks: two parallel sheets of face and edge
counts on both sides of one block, several blocks and one window (65,536 leaves). After the sheets were
turned and shifted, every vertex of the upper one that lies over the lower finds it at their distance
(a box that was not refitted, or not completely, loses some of them), and the contact lists are those of
trees built anew. Distances are exact to the rounding of coordinates up to 4 sheet extents: 2^-21 of it."""
import numpy as np
import pytest

from gaia_amd.detector import ContactDetector

pytestmark = pytest.mark.gpu


def sheet(n, m, cell):
    x, y = np.meshgrid(np.arange(n), np.arange(m), indexing="ij")
    i = (np.arange(n - 1)[:, None] * m + np.arange(m - 1)).ravel()
    faces = np.concatenate([np.stack([i, i + m, i + m + 1], 1), np.stack([i, i + m + 1, i + 1], 1)])
    return np.stack([cell * x.ravel(), cell * y.ravel(), np.zeros(n * m)], 1), faces.astype(np.int32)


# faces of both sheets: 4, 1,024, 1,028, 65,536 (edges 98,816), 66,048, 270,848 (edges 407,316)
@pytest.mark.parametrize("n,m", [(2, 2), (2, 257), (2, 258), (129, 129), (130, 129), (369, 185)])
def test_refitted_boxes_hold_their_primitives(gpu_ctx, n, m):
    cell, gap, r = 0.01, 0.002, 0.004
    low, faces = sheet(n, m, cell)
    high = low + [0.3 * cell, 0.2 * cell, gap]
    cd = ContactDetector(gpu_ctx, [(low.astype(np.float32), faces), (high.astype(np.float32), faces)],
                         max_query_dis=r, vf_capacity=4, ee_capacity=4)
    c, s = np.cos(2.0), np.sin(2.0)
    turn = np.array([[c, -s, 0], [s, c, 0], [0, 0, 1]]) @ np.array([[1, 0, 0], [0, c, -s], [0, s, c]])
    over = np.ones((n, m), bool)  # vertices of the upper sheet over the lower one
    over[-1], over[:, -1] = False, False
    extent = cell * max(n, m)
    for k in (1, 2):
        for mesh, x in enumerate((low, high)):
            cd.set_positions(mesh, (x @ np.linalg.matrix_power(turn, k).T + k * extent).astype(np.float32))
        cd.updateBVH(False)
        cd.query()
        vmin, _, _ = cd.min_distances()
        np.testing.assert_allclose(vmin[n * m:][over.ravel()], gap, rtol=0, atol=4 * 4 * extent * 2.0 ** -23 + 1e-7)
        lists = cd.results()
        cd.updateBVH(True)
        cd.query()
        for name, got, want in zip(("vf counts", "vf", "ee counts", "ee"), lists, cd.results()):
            if name.endswith("counts"):
                counts = want
                np.testing.assert_array_equal(got, want, err_msg=name)
            else:
                filled = np.arange(want.shape[1]) < counts[:, None]
                assert np.array_equal(got[filled], want[filled]), name
    cd.destroy()
