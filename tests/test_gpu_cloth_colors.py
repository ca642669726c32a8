"""Cloth whose given colours do not keep an element's vertices apart (colours without the bending stencils, and
a mesh of a single colour): every vertex is solved through positionsNext and copied back after its group, as the
oracle does, with and without contact, in group launches, in the work queue and where small scenes are stepped
whole by one block. Per step from identical state within 1e-5 of the FP32 oracle, and twice the same bits."""
import numpy as np
import pytest

import gaia_amd
from gaia_amd import VBDPhysics
from vbd_cases import contact_drape_spec, curtain_spec, rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5


def mesh_colors(m, kind):
    if kind == "one":
        return np.zeros(len(m["pos"]), np.int32)
    return gaia_amd.color_tri_mesh(len(m["pos"]), m["faces"], "mcs", with_bending=kind == "bending")


def build(ctx, oracle, spec, kind):
    sim = VBDPhysics(ctx)
    o32, o64 = (oracle.ClothScene(spec["physics"], precision=p) for p in (32, 64))
    sim.setPhysicsParams(**spec["physics"])
    for m in spec["meshes"]:
        colors = mesh_colors(m, kind)
        sim.addClothMesh(m["pos"], m["faces"], fixed_points=m["fixed"], vertex_colors=colors, velocities=m["vel"],
                         **m["material"])
        f64 = [None if a is None else np.asarray(a, np.float32).astype(np.float64) for a in (m["pos"], m["vel"])]
        for o in (o32, o64):
            o.add_mesh(f64[0], m["faces"], m["material"], colors, fixed=m["fixed"], vel=f64[1])
    for o in (sim.initialize, o32.finalize, o64.finalize):
        o()
    return sim, o32, o64


# (spec, lanes, mode, stepped whole): 400 vertices fit the passes of one block with 4 lanes, 3,600 do not
CASES = [(lambda: curtain_spec(20, steps=4), 4, "group", True), (lambda: curtain_spec(60, steps=3), 8, "group", False),
         (lambda: curtain_spec(20, steps=4), 8, "queue", False),
         (lambda: contact_drape_spec(steps=8, density=1.0), 8, "group", False),
         (lambda: contact_drape_spec(steps=8, density=1.0), 16, "group", False)]


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("kind", ["bending", "edges", "one"])
def test_colors_that_share_elements(gpu_ctx, oracle, case, kind):
    make, lanes, mode, whole = CASES[case]
    spec = make()
    if kind == "one":
        # all vertices of a mesh at once: plain Jacobi, which needs the inertia to dominate
        for m in spec["meshes"]:
            m["material"] = dict(m["material"], density=100 * m["material"]["density"])
    sim, o32, o64 = build(gpu_ctx, oracle, spec, kind)
    sim.setSchedule(lanes, 128, mode=mode)
    free = sum(len(m["pos"]) - len(m["fixed"]) for m in spec["meshes"])
    got_whole, committed = sim.planInfo()
    if kind == "one":
        assert committed == free
    else:
        assert got_whole == whole
        # "bending": merged groups may still hold two colours of a mesh
        assert committed == free if kind == "edges" else committed < free
    meshes = range(len(spec["meshes"]))
    for step in range(spec["steps"]):
        start = [o32.get_state(m) for m in meshes]
        for m in meshes:
            o64.set_state(m, *start[m])
        for o in (o32, o64):
            o.step(1, threads=8)
        runs = []
        for _ in range(2):
            for m in meshes:
                sim.setState(m, *start[m])
            sim.runSteps(1)
            runs.append([a for m in meshes for a in sim.getState(m)])
        assert all(np.array_equal(a, b) for a, b in zip(*runs))
        err = max(rel_err(runs[0][2 * m], o32.get_state(m)[0]) for m in meshes)
        spread = max(rel_err(o32.get_state(m)[0], o64.get_state(m)[0]) for m in meshes)
        print(f"step {step}: {err:.2e}, FP32 and FP64 oracle {spread:.2e}", flush=True)
        assert err < max(TOL, 4 * spread), f"step {step}: {err:.2e}, FP32 and FP64 oracle {spread:.2e}"
    sim.destroy()
