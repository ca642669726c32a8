"""The tet incidence records: every place of a vertex in its tet (the records' signs and the order of the
other three), well-shaped, needle and sliver rest shapes, and a fan of tets around one edge, with the
short records and (with material damping) the rows, one step from a deformed state against the
oracles: no farther from the FP64 one than four times the FP32 oracle is, or twice the rounding that
positions bring into F (an edge difference is off by eps |x|, F by eps |x| / h with h the smallest
height, and the step moves a vertex by that strain's share of the tet's extent), or 1e-6."""
import itertools

import numpy as np
import pytest

from gaia_amd.vbd import physics_dict
from vbd_cases import build_gpu, build_oracle, rel_err

pytestmark = pytest.mark.gpu

SHAPES = {
    "regular": [[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]],
    "needle": [[0, 0, 0], [0.05, 0, 0], [0, 0.05, 0], [0.02, 0.02, 2]],
    "sliver": [[0, 0, 0], [1, 0, 0], [0.9, 0.3, 0.02], [0.1, 0.3, 0]],
}


@pytest.mark.parametrize("shape", [*SHAPES, "fan"])
@pytest.mark.parametrize("damped", [False, True])
def test_records_of_every_place_in_a_tet(gpu_ctx, oracle, shape, damped):
    material = dict(density=1000.0, mu=1e5, lmbd=1e6)
    if damped:
        material.update(damping_hydrostatic=1e-3, damping_deviatoric=2e-3)
    meshes = []
    if shape == "fan":  # 7 tets around one edge
        a = 2 * np.pi * np.arange(7) / 7
        pos = np.concatenate([[[0, 0, 0], [0, 0, 0.2]], np.stack([0.2 * np.cos(a), 0.2 * np.sin(a), 0.1 + 0 * a], 1)])
        meshes.append((pos, np.array([[0, 2 + i, 2 + (i + 1) % 7, 1] for i in range(7)], np.int32)))
    else:
        p = 0.2 * np.array(SHAPES[shape], float)
        for perm in itertools.permutations(range(4)):
            q = p[list(perm)]
            if np.linalg.det(q[1:] - q[0]) > 0:  # the even ones keep the orientation
                meshes.append((q, np.array([[0, 1, 2, 3]], np.int32)))
        assert len(meshes) == 12
    rng = np.random.default_rng(3)
    spec = dict(physics=physics_dict(gravity=(0.0, -9.8, 0.0), time_step=1 / 60, num_substeps=1, iterations=6,
                                     world_lower=(-1e7, -1e7, -1e7)), steps=1,
                meshes=[dict(pos=pos, tets=tets, material=material, fixed=(), coloring="greedy",
                             vel=rng.normal(scale=0.3, size=pos.shape)) for pos, tets in meshes])
    o32, o64, sim = build_oracle(oracle, spec), build_oracle(oracle, spec, precision=64), build_gpu(gpu_ctx, spec)
    for m, (pos, _) in enumerate(meshes):
        x = (pos * (1 + rng.uniform(-0.05, 0.05, 3)) + 0.002 * rng.normal(size=pos.shape)).astype(np.float32)
        v = rng.normal(scale=0.3, size=pos.shape).astype(np.float32)
        for s in (o32, o64):
            s.set_state(m, x.astype(np.float64), v.astype(np.float64))
        sim.setState(m, x, v)
    for s in (o32, o64):
        s.step(1)
    sim.runStep()
    for m in range(len(meshes)):
        x, ref = sim.getState(m)[0], o64.get_state(m)[0]
        err, own = rel_err(x, ref), rel_err(o32.get_state(m)[0], ref)
        pos, tets = meshes[m]
        rows = np.linalg.inv((pos[tets[0, 1:]] - pos[tets[0, 0]]).T)  # rows of DmInv: 1 / heights
        h = 1 / max(np.linalg.norm(r) for r in (*rows, rows.sum(0)))
        bound = max(4 * own, 2 * np.finfo(np.float32).eps / 2 * np.abs(x).max() / h, 1e-6)
        assert err < bound, f"mesh {m}: {err:.2e} from FP64, the FP32 oracle {own:.2e}, bound {bound:.2e}"
    sim.destroy()
