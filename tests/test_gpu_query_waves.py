"""The contact queries of a wave (8, 16 or 32 vertices or edges share its lanes) against the record
pass, which walks the trees one query per thread: counts, capped lists (the lowest ids) and minimum
distances, from a single triangle to sizes on both sides of each rule, capacities 1 to 16, and spots
with more contacts than a wave's hit list holds at once."""
import numpy as np
import pytest

from gaia_amd import scenes
from gaia_amd.detector import ContactDetector

pytestmark = pytest.mark.gpu


def crowd(n):
    """n small triangles around one point: every vertex is near every other triangle."""
    rng = np.random.default_rng(n)
    tri = rng.normal(size=(n, 3, 3)) * 4e-4
    return [(t.astype(np.float32), np.array([[0, 1, 2]], np.int32)) for t in tri]


def tori(grid, nu, nv):
    return scenes.c3_tori(seed=1, grid=grid, nu=nu, nv=nv)[0]


CASES = {
    "one triangle": lambda: crowd(1),
    "two triangles": lambda: crowd(2),
    "crowd": lambda: crowd(150),
    "crowd of 3": lambda: crowd(3) + [(np.array([[9, 9, 9], [9.1, 9, 9], [9, 9.1, 9]], np.float32), np.array([[0, 1, 2]], np.int32))],
    "8 per wave": lambda: tori(2, 40, 20),
    "16 per wave": lambda: tori(2, 128, 63),  # 64,512 vertices, 193,536 edges
    "32 edges per wave": lambda: tori(3, 120, 60),  # 194,400 vertices (16 per wave), 583,200 edges
    "32 per wave": lambda: tori(4, 66, 63),  # 266,112 vertices, 798,336 edges
}


def test_one_face_within_the_largest_distance(gpu_ctx):
    """A tree of one leaf, and query boxes that overflow to infinity in every direction."""
    tri = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0]], np.float32)
    points = np.array([[0.25, 0.25, 2.0], [-3.0, 0.0, 0.0], [1.5, 1.5, 0.0]], np.float32)
    cd = ContactDetector(gpu_ctx, [(tri, np.array([[0, 1, 2]], np.int32)), (points, np.zeros((0, 3), np.int32))],
                         max_query_dis=np.finfo(np.float32).max)
    cd.updateBVH(True)
    cd.query()
    want = np.array([2.0, 3.0, np.sqrt(2.0)], np.float32)
    vertex, face, _ = cd.min_distances()
    np.testing.assert_allclose(vertex[3:], want, rtol=1e-6)
    np.testing.assert_allclose(face, [want.min()], rtol=1e-6)
    vc, vr, _, _ = cd.results()
    assert vc.tolist() == [0, 0, 0, 1, 1, 1] and (vr["face"][3:, 0] == 0).all()
    cd.destroy()


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("cap", [1, 8, 16])
def test_wave_queries_equal_the_record_pass(gpu_ctx, name, cap):
    r = np.float32(0.002)
    cd = ContactDetector(gpu_ctx, CASES[name](), max_query_dis=r, vf_capacity=cap, ee_capacity=cap)
    cd.updateBVH(True)
    cd.query(record=True)
    rec, counts = cd.recorded(), cd.counts()
    vc, vr, ec, er = cd.results()
    vmin, fmin, _ = cd.min_distances()
    cd.destroy()
    # every vertex's contacts by ascending face, cut at the capacity
    v = rec["vf_contacts"]
    d = rec["vf_contact_d"][np.lexsort((v[:, 3], v[:, 0]))]
    v = v[np.lexsort((v[:, 3], v[:, 0]))]
    rank = np.arange(len(v)) - np.searchsorted(v[:, 0], v[:, 0])
    keep = rank < cap
    want = np.zeros(len(vc), int)
    np.add.at(want, v[keep, 0], 1)
    np.testing.assert_array_equal(vc, want)
    got = vr[v[keep, 0], rank[keep]]
    for k, col in (("face", 3), ("type", 1), ("prim", 2)):
        np.testing.assert_array_equal(got[k], v[keep, col])
    np.testing.assert_array_equal(got["d"], d[keep])
    assert counts["vf_overflow"] == len(np.unique(v[~keep, 0]))
    e = rec["ee_contacts"]
    o = np.lexsort((e[:, 1], e[:, 0]))
    e, mu, d = e[o], rec["ee_mu"][o], rec["ee_d"][o]
    rank = np.arange(len(e)) - np.searchsorted(e[:, 0], e[:, 0])
    keep = rank < cap
    want = np.zeros(len(ec), int)
    np.add.at(want, e[keep, 0], 1)
    np.testing.assert_array_equal(ec, want)
    got = er[e[keep, 0], rank[keep]]
    np.testing.assert_array_equal(got["edge"], e[keep, 1])
    np.testing.assert_array_equal(np.stack([got["mu1"], got["mu2"], got["d"]], 1), np.column_stack([mu[keep], d[keep]]))
    assert counts["ee_overflow"] == len(np.unique(e[~keep, 0]))
    pv, pf, pd = rec["vf_pairs"][:, 0], rec["vf_pairs"][:, 1], rec["vf_pair_d"]
    for got, ids in ((vmin, pv), (fmin, pf)):
        ref = np.full(len(got), r, np.float32)
        np.minimum.at(ref, ids, pd)
        np.testing.assert_array_equal(got, ref)
    print(f"\n[{name}, capacity {cap}] {counts}", flush=True)
