"""The closest-face search of the penetration contact, one wave per contained vertex: trees from a dozen
faces to some thousand, vertices just under the surface and deep in the other body (whose nearest faces
are rejected, up to the search over all the rest), every detection equal to the oracle's."""
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
