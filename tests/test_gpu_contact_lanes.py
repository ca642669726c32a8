"""Contact pairs of a vertex spread over the lanes of its solve: every lane count, with vertices whose
incident faces and edges are fewer than, as many as and more than the lanes (a fan's centre has 23),
per step against the FP32 oracle from identical state."""
import numpy as np
import pytest

from vbd_cases import build_gpu, build_oracle, build_oracle_cloth, contact_drape_spec, penetration_spec, rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5  # the per-step contract of the contact parity tests


def fan_drape_spec(valence=23):
    """The drape with the falling sheet replaced by a fan: one centre vertex in `valence` faces."""
    spec = contact_drape_spec(steps=8)
    a = 2 * np.pi * np.arange(valence) / valence
    ring = np.stack([0.12 * np.cos(a), np.zeros(valence), 0.12 * np.sin(a)], axis=1)
    pos = np.concatenate([[[0.0, 0.0, 0.0]], ring])
    pos[:, 1] = 0.02 * pos[:, 0] + 0.0085  # within the contact radius of the lower sheet from the start
    i = np.arange(valence)
    faces = np.stack([np.zeros(valence, int), 1 + (i + 1) % valence, 1 + i], axis=1).astype(np.int32)
    spec["meshes"][1] = dict(spec["meshes"][1], pos=pos, faces=faces, vel=np.tile([0.05, -0.1, 0.0], (len(pos), 1)))
    return spec


@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("scene", ["drape", "fan", "penetration"])
def test_contact_pairs_over_lanes(gpu_ctx, oracle, lanes, scene):
    spec = {"drape": lambda: contact_drape_spec(steps=8), "fan": fan_drape_spec,
            "penetration": lambda: penetration_spec(steps=14)}[scene]()
    sim = build_gpu(gpu_ctx, spec)
    sim.setSchedule(lanes, 64)
    ref = (build_oracle if scene == "penetration" else build_oracle_cloth)(oracle, spec)
    worst, pairs = 0.0, 0
    for _ in range(spec["steps"]):
        for m in range(len(spec["meshes"])):
            sim.setState(m, *ref.get_state(m))
        sim.runStep()
        ref.step(1)
        worst = max([worst] + [rel_err(sim.getState(m)[0], ref.get_state(m)[0]) for m in range(len(spec["meshes"]))])
        pairs = max(pairs, sim.contactStats()["vf_pairs"])
    sim.destroy()
    print(f"\n[{scene}, {lanes} lanes] worst per-step rel err {worst:.2e}, up to {pairs} vertex-face pairs", flush=True)
    assert pairs > 0
    assert worst < TOL
