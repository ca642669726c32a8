"""Containment and CCD queries of the penetration contact with 8, 16 and 32 surface vertices per wave (up to 49,152
vertices, up to 262,144, and more): three one-cell slabs, the second sunk into the first, the third falling through the
second's upper side within the step. Every vertex's detection equals the oracle's."""
import itertools

import numpy as np
import pytest

from test_gpu_tet_penetration import oracle_rows
from vbd_cases import build_gpu, build_oracle, penetration_spec

pytestmark = pytest.mark.gpu
H = 0.04


def slab(n):
    """n x 1 x n cells of edge H, each of 6 tets around its diagonal (all surface vertices)."""
    i, j, k = (a.ravel() for a in np.meshgrid(np.arange(n + 1), np.arange(2), np.arange(n + 1), indexing="ij"))
    pos = H * np.stack([i, j, k], 1).astype(float)
    stride = np.array([2 * (n + 1), n + 1, 1])
    ci, ck = (a.ravel() for a in np.meshgrid(np.arange(n), np.arange(n), indexing="ij"))
    base = ci * stride[0] + ck * stride[2]
    tets = []
    for p in itertools.permutations(range(3)):
        a, b = base + stride[p[0]], base + stride[p[0]] + stride[p[1]]
        even = p in ((0, 1, 2), (1, 2, 0), (2, 0, 1))
        tets.append(np.stack([base, a, b, base + stride.sum()] if even else [base, b, a, base + stride.sum()], 1))
    return pos, np.concatenate(tets).astype(np.int32)


def spec_with(n_idle):
    """The three slabs of 882 vertices, and one of n_idle x n_idle cells above the detection's height: its surface
    vertices only raise the number of queries."""
    spec = penetration_spec(steps=1, iterations=1)
    spec["physics"]["collision_off_height"] = 10.0
    material = spec["meshes"][0]["material"]
    pos, tets = slab(20)
    c, s = np.cos(0.05), np.sin(0.05)
    turn = np.array([[c, 0, s], [0, 1, 0], [-s, 0, c]])
    spec["meshes"] = []
    for b, (y, vy) in enumerate([(1.0, 0.0), (1.0 + 0.7 * H, 0.0), (1.0 + 1.9 * H, -0.5 * H * 60)]):
        x = pos @ np.linalg.matrix_power(turn, b).T + [0.3 * H * b, y, 0.2 * H * b]
        spec["meshes"].append(dict(pos=x, tets=tets, material=material, fixed=(), coloring="greedy",
                                   vel=np.tile([0.0, vy, 0.0], (len(x), 1))))
    if n_idle:
        pos, tets = slab(n_idle)
        spec["meshes"].insert(1, dict(pos=pos + [0.0, 20.0, 0.0], tets=tets, material=material, fixed=(),
                                      coloring="greedy", vel=None))
    return spec


@pytest.mark.parametrize("n_idle", [0, 160, 365])  # 2,646, 54,488 and 270,558 surface vertices
def test_slabs_detected_as_by_the_oracle(gpu_ctx, oracle, n_idle):
    spec = spec_with(n_idle)
    sim, ref = build_gpu(gpu_ctx, spec), build_oracle(oracle, spec)
    sizes = [len(m["pos"]) for m in spec["meshes"]]
    for m in range(len(sizes)):
        sim.setState(m, *ref.get_state(m))
    sim.runStep()
    ref.step(1, threads=8)
    rows, counts = sim.penetrationResults()
    want = oracle_rows(ref, sizes)
    sim.destroy()
    print(f"\n[{sum(sizes)} vertices] counts {counts.tolist()}", flush=True)
    np.testing.assert_array_equal(rows, want)
    assert counts[0] > 200 and counts[2] > 200
