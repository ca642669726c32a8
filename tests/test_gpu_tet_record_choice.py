"""Which incidence records a scene's tets have, by the bytes that the gather model counts for them: rows (88 B
per incident tet) in scenes with material damping, the accelerator or collision handling, short records (68 B)
otherwise."""
import pytest

from gaia_amd import Batch
from vbd_cases import build_gpu, penetration_spec, tet_drop_spec

pytestmark = pytest.mark.gpu


def plain(**physics):
    spec = penetration_spec()
    spec["physics"].update(dict(handle_collision=0), **physics)
    return spec


def damped():
    spec = plain()
    spec["meshes"][0]["material"].update(damping_deviatoric=1e-3)
    return spec


@pytest.mark.parametrize("make,per_tet", [(plain, 68), (damped, 88), (lambda: plain(use_accelerator=1), 88),
                                          (penetration_spec, 88), (tet_drop_spec, 88)])
def test_records_by_scene(gpu_ctx, make, per_tet):
    spec = make()
    sim = build_gpu(gpu_ctx, spec)
    batch = Batch(gpu_ctx, [sim])
    tets = [m for m in spec["meshes"] if "tets" in m]
    want = sum(72 * len(m["pos"]) + per_tet * m["tets"].size for m in tets)  # the sheet of tet_drop_spec is fixed
    assert sum(batch.group_work(g)[0] for g in range(batch.num_groups())) == want
    batch.destroy()
    sim.destroy()
