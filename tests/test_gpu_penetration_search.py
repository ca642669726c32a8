"""The closest-face search of the penetration contact, one wave per contained vertex: trees from a dozen
faces to some thousand, vertices just under the surface and deep in the other body, and vertices whose
nearest faces are rejected, every detection equal to the oracle's."""
import numpy as np
import pytest

from gaia_amd import scenes
from test_gpu_tet_penetration import oracle_rows
from vbd_cases import build_gpu, build_oracle, penetration_spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,depth,turn", [(1, 0.06, 0), (2, 0.1, 1), (4, 0.03, 2), (8, 0.2, 3), (12, 0.35, 4), (16, 0.25, 5)])
def test_contained_vertices_find_the_oracles_faces(gpu_ctx, oracle, n, depth, turn):
    spec = penetration_spec(steps=1)
    edge = 0.1 * max(n, 2) if n < 8 else 0.8
    material = spec["meshes"][0]["material"]
    spec["meshes"] = []
    for b in range(3):
        pos, tets = scenes.cube_tet_mesh(n, edge / n, origin=(-edge / 2,) * 3)
        rng = np.random.default_rng(10 * turn + b)
        pos = pos @ scenes.random_rotation(rng).T + np.array([0.3 * edge * (b == 2), 0.5 + (edge - depth) * b, 0.0])
        spec["meshes"].append(dict(pos=pos, tets=tets, material=material, fixed=(), vel=None, coloring="greedy"))
    sim = build_gpu(gpu_ctx, spec)
    ref = build_oracle(oracle, spec)
    sizes = [len(m["pos"]) for m in spec["meshes"]]
    for m in range(3):
        sim.setState(m, *ref.get_state(m))
    sim.runStep()
    ref.step(1, threads=8)
    rows, counts = sim.penetrationResults()
    want = oracle_rows(ref, sizes)
    sim.destroy()
    print(f"\n[{n}^3 cells] counts {counts.tolist()}", flush=True)
    np.testing.assert_array_equal(rows, want)
    assert counts[0] == int(((want[:, 4] == 1) & (want[:, 3] >= 0)).sum())
    if n > 1:
        assert counts[0] > 0


@pytest.mark.parametrize("n", [2, 5])
def test_searches_past_the_nearest_faces(gpu_ctx, oracle, n):
    """A mesh of two parts, a small cube (48 or 300 faces) floating inside a large one, and vertices of another body
    beside the small part: the walk inside the large part reaches none of the small part's faces, so that more than
    the 8 nearest are rejected and the search goes on over all the rest."""
    spec = penetration_spec(steps=1)
    material = spec["meshes"][0]["material"]
    large, small = scenes.cube_tet_mesh(3, 0.3, origin=(-0.45, 0.5, -0.45)), scenes.cube_tet_mesh(n, 0.1 / n, origin=(0.1, 0.9, 0.0))
    probe = scenes.cube_tet_mesh(1, 0.04, origin=(0.22, 0.93, 0.03))
    parts = [(np.concatenate([large[0], small[0]]), np.concatenate([large[1], small[1] + len(large[0])])), probe]
    spec["meshes"] = [dict(pos=pos, tets=tets.astype(np.int32), material=material, fixed=(), vel=None, coloring="greedy")
                      for pos, tets in parts]
    sim, ref = build_gpu(gpu_ctx, spec), build_oracle(oracle, spec)
    for m in range(2):
        sim.setState(m, *ref.get_state(m))
    sim.runStep()
    ref.step(1, threads=8)
    rows, counts = sim.penetrationResults()
    sim.destroy()
    print(f"\n[{12 * n * n} faces] counts {counts.tolist()}", flush=True)
    np.testing.assert_array_equal(rows, oracle_rows(ref, [len(pos) for pos, _ in parts]))
    assert counts[4] > 0
