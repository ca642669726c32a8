"""Performance cases of the framework: what its users have it do, through its public entry points.

A case is one of these uses (sizes come from the benchmark configurations and the tests):
  tet          one soft body (a cube of n^3 cells) advanced frame by frame and read back: an interactive scene
  cloth        one hanging sheet of n x n vertices, a rollout from a given state
  batch        many independent tet and cloth scenes advanced together from given states (data sets, ensembles)
  serve        step requests for resident bodies, continuously batched by the server, states sent back
  penetration  tet bodies in a pile with the tet solver's own contact (DCD + CCD), a rollout from a given state
  contact      tet bodies landing on a pinned sheet with the cloth contact model, a rollout from a given state
  detector     the contact detector on its own: new positions, refit, queries, bounds and minimum distances

`exact` is vertex block descent (and the detector's distances) in 64-bit torch. The contact rollouts have no such
value: their forces switch on at a distance threshold, so a 64-bit run takes other branches within a few iterations.
"""
import functools
import math
import sys

import numpy as np
import torch

import gaia_amd
from gaia_amd import VBDPhysics, scenes
from gaia_amd.detector import ContactDetector
from gaia_amd.vbd import Batch, Server

DT = 1.0 / 60.0
GRAVITY = -9.8
TET_MAT = dict(density=1000.0, mu=1e5, lmbd=1e6)
DAMPING = dict(damping_hydrostatic=1e-3, damping_deviatoric=2e-3)
CLOTH_MU, CLOTH_LM = scenes.stvk_lame(1e5, 0.3)
CLOTH_MAT = dict(density=0.2, mu=CLOTH_MU, lmbd=CLOTH_LM, bending_stiffness=1e-4, initialization_type=0)
RHO = 0.9  # Chebyshev acceleration of the tet iterations


# ---- the cases -----------------------------------------------------------------------------------

def listed():
    return [
        # the smallest call there is: one frame of a 125-vertex body (launches and latency only)
        dict(name="tet 125", kind="tet", n=4, iterations=10, substeps=1, frames=1, damped=False, accelerated=False,
             schedule="default"),
        # the soft cube of the plain configuration, 1,331 vertices, one frame at a time
        dict(name="tet 1331", kind="tet", n=10, iterations=10, substeps=1, frames=1, damped=False, accelerated=False,
             schedule="default"),
        # a body of 50,653 vertices with material damping, substeps and the accelerator, frame by frame
        dict(name="tet 50k damped", kind="tet", n=36, iterations=10, substeps=2, frames=1, damped=True,
             accelerated=True, schedule="8x128"),
        # the largest single body served: 205,379 vertices; a few frames between two readbacks
        dict(name="tet 205k", kind="tet", n=58, iterations=10, substeps=1, frames=4, damped=False, accelerated=False,
             schedule="8x128"),
        # a small garment-sized sheet of 24 x 24 vertices
        dict(name="cloth 576", kind="cloth", n=24, iterations=10, frames=1, damped=False, schedule="default"),
        # a finely meshed sheet of 333 x 333 vertices with membrane and bending damping
        dict(name="cloth 111k damped", kind="cloth", n=333, iterations=10, frames=4, damped=True, schedule="8x128"),
        # an ensemble of 24 small scenes (500 to 2,000 vertices), a tenth of a second each
        dict(name="batch 24 small", kind="batch", scenes=24, vmin=500, vmax=2000, frames=6, schedule="default"),
        # the batched configuration's size range, 500 to 50,000 vertices per scene
        dict(name="batch 48 mixed", kind="batch", scenes=48, vmin=500, vmax=50000, frames=6, schedule="8x128"),
        # a burst of step requests to the server over a population of uneven scenes
        dict(name="serve 32", kind="serve", scenes=32, vmin=1000, vmax=20000, requests=100, schedule="8x128"),
        # 32 bodies of 8,640 tets in a pile, the tet solver's penetration contact
        dict(name="penetration 32", kind="penetration", bodies=32, n=12, iterations=20, frames=3, schedule="16x256"),
        # bodies landing on a pinned sheet, cloth contact model with friction and conservative bounds
        dict(name="contact 8 on sheet", kind="contact", bodies=8, n=10, sheet=61, iterations=20, frames=3,
             schedule="16x256"),
        # the detector configuration's tori (4 mm edges, 2 mm radius): 27 of them
        dict(name="detector 27", kind="detector", grid=3, nu=128, nv=64, lists=False),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["tet", "tet", "cloth", "cloth", "batch", "serve", "penetration", "contact", "detector"])
    schedule = rng.choice(["default", "8x128", "8x256", "4x128", "16x128"])
    if kind == "tet":
        n = max(3, round(_log(rng, 64, 195000) ** (1.0 / 3.0)) - 1)
        return dict(kind=kind, n=n, iterations=rng.randint(5, 12), substeps=rng.randint(1, 2), frames=rng.randint(1, 3),
                    damped=rng.random() < 0.5, accelerated=rng.random() < 0.3, schedule=schedule)
    if kind == "cloth":
        n = max(5, round(math.sqrt(_log(rng, 64, 110000))))
        return dict(kind=kind, n=n, iterations=rng.randint(5, 12), frames=rng.randint(1, 3), damped=rng.random() < 0.5,
                    schedule=schedule)
    if kind == "batch":
        vmax = round(_log(rng, 1500, 40000))
        return dict(kind=kind, scenes=rng.randint(5, 40), vmin=rng.randint(200, 1000), vmax=vmax,
                    frames=rng.randint(1, 6), schedule=schedule)
    if kind == "serve":
        return dict(kind=kind, scenes=rng.randint(6, 30), vmin=rng.randint(300, 1500), vmax=round(_log(rng, 2000, 20000)),
                    requests=rng.randint(10, 90), schedule=schedule)
    if kind == "penetration":
        return dict(kind=kind, bodies=rng.randint(4, 31), n=rng.randint(5, 11), iterations=rng.randint(8, 20),
                    frames=rng.randint(2, 4), schedule=rng.choice(["16x256", "8x128", "default"]))
    if kind == "contact":
        return dict(kind=kind, bodies=rng.randint(2, 8), n=rng.randint(4, 9), sheet=rng.randint(25, 60),
                    iterations=rng.randint(8, 20), frames=rng.randint(1, 3),
                    schedule=rng.choice(["16x256", "8x128", "default"]))
    grid = rng.choice([1, 2, 2])
    return dict(kind=kind, grid=grid, nu=rng.randint(11, 128), nv=rng.randint(7, 64), lists=rng.random() < 0.5)


# ---- meshes, colours and initial states ------------------------------------------------------------

@functools.lru_cache(maxsize=64)
def _cube(n):
    """Cube of n^3 cells of 5 cm standing on the ground plane, coloured by the parity of the grid coordinates."""
    pos, tets = scenes.cube_tet_mesh(n, 0.05, origin=(0.0, 0.0, 0.0), dtype=np.float32)
    i = np.arange(len(pos))
    a, b, c = i % (n + 1), i // (n + 1) % (n + 1), i // (n + 1) ** 2
    return pos, tets, (a % 2 + 2 * (b % 2) + 4 * (c % 2)).astype(np.int32)


@functools.lru_cache(maxsize=64)
def _curtain(n):
    """Sheet of n x n vertices hanging from its top row; colours of a 3 x 3 pattern (no two vertices of a bending
    stencil share one)."""
    pos, faces, top = scenes.cloth_curtain(n, 1.0, 2.0, dtype=np.float32)
    i = np.arange(n * n)
    return pos, faces, (i % n % 3 + 3 * (i // n % 3)).astype(np.int32), tuple(top)


def _waves(rng, pos, amplitude):
    """A smooth vector field of the given root-mean-square size: three random sine waves over the body."""
    x = pos.astype(np.float64)
    out = np.zeros_like(x)
    scale = max(float(np.ptp(x)), 1e-9)
    for _ in range(3):
        k = rng.normal(size=3) * 4.0 / scale
        out += np.sin(x @ k + rng.uniform(0, 2 * np.pi))[:, None] * rng.normal(size=3)
    return amplitude * out / math.sqrt(4.5)


def _tet_state(rng, pos):
    x = pos + _waves(rng, pos, 0.004 * float(np.ptp(pos[:, 0])) + 1e-3)
    v = _waves(rng, pos, 0.1) + rng.uniform(-0.5, 0.5, 3) * (1, 0.4, 1)
    return x.astype(np.float32), v.astype(np.float32)


def _cloth_state(rng, pos, fixed):
    # a hung sheet under tension, still being stretched, rippled out of its plane. (In compression the exact membrane
    # Hessian is indefinite and a step amplifies rounding by orders of magnitude; a sheet left to itself gets there
    # within some dozens of frames, so that each pass starts from the given state.)
    x = pos.astype(np.float64).copy()
    x[:, 0] = 0.5 + (x[:, 0] - 0.5) * 1.002
    x[:, 1] = 2.0 + (x[:, 1] - 2.0) * 1.01
    x[:, 2] += _waves(rng, pos, 2e-3)[:, 2]
    v = _waves(rng, pos, 0.05)
    stretch = rng.uniform(0.2, 0.4)
    v[:, 0] = stretch * (pos[:, 0] - 0.5)
    v[:, 1] = 2 * stretch * (pos[:, 1] - 2.0)
    x[list(fixed)] = pos[list(fixed)]
    v[list(fixed)] = 0.0
    return x.astype(np.float32), v.astype(np.float32)


def _rng(seed):
    return np.random.default_rng([7, seed])


# ---- scenes ----------------------------------------------------------------------------------------

class _Held:
    """Scenes, batches, servers and detectors of one state; they leave the device with it."""

    def __init__(self):
        self.items = []

    def add(self, item):
        self.items.append(item)
        return item

    def __del__(self):
        if sys.is_finalizing():
            return
        for item in reversed(self.items):
            item.destroy()


@functools.lru_cache(maxsize=1)
def _ctx():
    return gaia_amd.Context(0)


def _physics(case):
    return dict(gravity=(0.0, GRAVITY, 0.0), time_step=DT, num_substeps=case.get("substeps", 1),
                iterations=case.get("iterations", 10), world_lower=(-1e7, 0.0, -1e7), world_upper=(1e7, 1e7, 1e7),
                use_accelerator=int(case.get("accelerated", False)), accelerator_rho=RHO)


def _cloth_material(damped):
    return dict(CLOTH_MAT, **(dict(damping_stvk=1e-4, damping_bending=1e-4) if damped else {}))


@functools.lru_cache(maxsize=48)
def _template(kind, n, iterations, substeps, damped, accelerated):
    """A scene created once with its mesh; states are instances of it (clones share the host-side preparation)."""
    sim = VBDPhysics(_ctx())
    sim.setPhysicsParams(**_physics(dict(iterations=iterations, substeps=substeps, accelerated=accelerated)))
    if kind == "tet":
        pos, tets, colors = _cube(n)
        sim.addTetMesh(pos, tets, vertex_colors=colors, **dict(TET_MAT, **(DAMPING if damped else {})))
    else:
        pos, faces, colors, top = _curtain(n)
        sim.addClothMesh(pos, faces, fixed_points=list(top), vertex_colors=colors, **_cloth_material(damped))
    sim.initialize(defer_upload=True)
    return sim


def _instance(held, kind, n, case, upload=True):
    t = _template(kind, n, case.get("iterations", 10), case.get("substeps", 1), case.get("damped", False),
                  case.get("accelerated", False))
    return held.add(t.clone(defer_upload=not upload))


def _start(rng, kind, n):
    if kind == "tet":
        return _tet_state(rng, _cube(n)[0])
    pos, _, _, top = _curtain(n)
    return _cloth_state(rng, pos, top)


def _schedule(case):
    if case["schedule"] == "default":
        return None
    lanes, block = case["schedule"].split("x")
    return int(lanes), int(block)


def _many(case):
    """(kind, grid size) of a batch's or a server's scenes: log-spaced vertex targets, every second one of a batch a
    sheet. From the sizes alone, so that states of several seeds are instances of the same meshes."""
    out = []
    for i in range(case["scenes"]):
        # sizes in a shuffled order: golden-ratio steps through the log range
        target = case["vmin"] * (max(case["vmax"], case["vmin"]) / case["vmin"]) ** ((i * 0.6180339887 + 0.3) % 1.0)
        if i % 2 and case["kind"] == "batch":
            out.append(("cloth", max(5, round(math.sqrt(target)))))
        else:
            out.append(("tet", max(3, round(target ** (1.0 / 3.0)) - 1)))
    return out


def _bodies(case):
    """Cubes and balls in a pile (penetration: neighbours overlap slightly where rotated corners meet) or in a grid
    just above a sheet (contact)."""
    if case["kind"] == "penetration":
        return scenes.c2_bodies(seed=5, n=case["n"], spacing=0.33, layers_y=(0.19, 0.52))[:case["bodies"]]
    out = []
    cube, cube_tets = scenes.cube_tet_mesh(case["n"], 0.24 / case["n"], origin=(-0.12,) * 3)
    ball, ball_tets = scenes.tet_ball(case["n"], 0.13)
    for b in range(case["bodies"]):
        base, tets = (cube, cube_tets) if b % 2 == 0 else (ball, ball_tets)
        low = float(base[:, 1].min())
        centre = np.array([-0.45 + 0.3 * (b % 4), 0.5015 - low, -0.15 + 0.3 * (b // 4)])
        out.append(dict(pos=base + centre, tets=tets, material=dict(density=300.0, mu=2e5, lmbd=2e6,
                                                                     friction_dynamic=0.2, friction_eps_v=0.01)))
    return out


@functools.lru_cache(maxsize=16)
def _contact_template(kind, bodies, n, sheet, iterations):
    case = dict(kind=kind, bodies=bodies, n=n, sheet=sheet)
    sim = VBDPhysics(_ctx())
    if kind == "penetration":
        sim.setPhysicsParams(**dict(scenes.c2_physics(iterations=iterations), tet_contact_model=1,
                                    collision_stiffness=500.0))
    else:
        sim.setPhysicsParams(**dict(scenes.c2_physics(iterations=iterations), contact_stiffness=30.0))
    start = []
    for b in _bodies(case):
        pos = b["pos"].astype(np.float32)
        colors = gaia_amd.color_tet_mesh(len(pos), b["tets"], "greedy")
        sim.addTetMesh(pos, b["tets"], vertex_colors=colors, **b["material"])
        start.append(pos)
    if kind == "contact":
        pos, faces = scenes.cloth_sheet(sheet, 1.3, 0.5, origin=(-0.65, -0.65), dtype=np.float32)
        grid = np.arange(sheet * sheet).reshape(sheet, sheet)
        rim = sorted(set(np.concatenate([grid[0], grid[-1], grid[:, 0], grid[:, -1]]).tolist()))
        sim.addClothMesh(pos, faces, fixed_points=rim,
                         vertex_colors=gaia_amd.color_tri_mesh(len(pos), faces, "mcs"),
                         **dict(CLOTH_MAT, density=1.0, friction_dynamic=0.2, friction_eps_v=0.01))
        start.append(pos)
    sim.initialize(defer_upload=True)
    return sim, start


def _prepare_contact(case, seed, held):
    template, start = _contact_template(case["kind"], case["bodies"], case["n"], case.get("sheet", 0),
                                        case["iterations"])
    sim = held.add(template.clone(defer_upload=False))
    rng = _rng(seed)
    states = []
    for m, pos in enumerate(start):
        if case["kind"] == "contact" and m == len(start) - 1:
            states.append((pos, np.zeros_like(pos)))
            continue
        vel = np.array([0.0, -0.4 if case["kind"] == "contact" else -0.8, 0.0]) + rng.uniform(-0.3, 0.3, 3) * (1, 0.3, 1)
        states.append((pos, (vel + _waves(rng, pos, 0.02)).astype(np.float32)))
    sc = _schedule(case)
    if sc:
        sim.setSchedule(*sc)
    for m, (x, v) in enumerate(states):
        sim.setState(m, x, v)
    if case["kind"] == "penetration":
        sim.recordVBDSolveGraph(True)
    return dict(sim=sim, states=states)


def _tori(case, seed):
    rng = _rng(seed)
    meshes, drifts = scenes.c3_tori(seed=3, grid=case["grid"], nu=case["nu"], nv=case["nv"])
    steps = []
    for k in range(3):  # positions of three successive steps: drift and 1 mm of noise
        steps.append([(x + (k + 1) * d + rng.normal(scale=1e-3, size=x.shape)).astype(np.float32)
                      for (x, _), d in zip(meshes, drifts)])
    return meshes, steps


def _burst(rng, case):
    """The scenes of one burst of requests, in the order in which they ask for a frame."""
    return rng.permutation(np.arange(case["requests"]) % case["scenes"]).tolist()


def prepare(case, seed):
    kind, held = case["kind"], _Held()
    state = dict(case=case, held=held)
    rng = _rng(seed)
    if kind in ("tet", "cloth"):
        sim = _instance(held, kind, case["n"], case)
        sc = _schedule(case)
        if sc:
            sim.setSchedule(*sc)
        state["start"] = _start(rng, kind, case["n"])
        sim.setState(0, *state["start"])
        sim.recordVBDSolveGraph(True)
        state["sim"] = sim
    elif kind == "batch":
        sims, start = [], []
        for k, n in _many(case):
            sims.append(_instance(held, k, n, case))
            start.append(_start(rng, k, n))
            sims[-1].setState(0, *start[-1])
        batch = held.add(Batch(_ctx(), sims))
        sc = _schedule(case)
        if sc:
            batch.set_schedule(*sc)
        batch.record_graph(True)
        state.update(sims=sims, batch=batch, start=start)
    elif kind == "serve":
        sims = []
        for k, n in _many(case):
            sims.append(_instance(held, k, n, case))
            sims[-1].setState(0, *_start(rng, k, n))
        server = held.add(Server(_ctx(), 64 << 30))
        sc = _schedule(case)
        if sc:
            server.set_schedule(*sc)
        for s in sims:
            server.add_scene(s)
        state.update(sims=sims, server=server, burst=_burst(rng, case))
    elif kind == "detector":
        meshes, steps = _tori(case, seed)
        state.update(cd=held.add(ContactDetector(_ctx(), meshes, max_query_dis=0.002)), steps=steps, at=0)
    else:
        state.update(_prepare_contact(case, seed, held))
    return state


def _read(sims):
    both = [s.getState(0) for s in sims]
    return dict(x=np.concatenate([b[0] for b in both]), v=np.concatenate([b[1] for b in both]))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("tet", "cloth"):
        if kind == "cloth":
            state["sim"].setState(0, *state["start"])
        state["sim"].runSteps(case["frames"])
        x, v = state["sim"].getState(0)
        return dict(x=x, v=v)
    if kind == "batch":
        for sim, start in zip(state["sims"], state["start"]):
            sim.setState(0, *start)
        state["batch"].run_steps(case["frames"])
        return _read(state["sims"])
    if kind == "serve":
        server, sims = state["server"], state["sims"]
        for tag, i in enumerate(state["burst"]):
            server.request_step(sims[i], tag)
        while server.tick()["pending"]:
            pass
        done = server.poll()
        frames = np.zeros(len(state["burst"]), np.int32)
        frames[done["tag"]] = done["frame"]
        return dict(_read([sims[i] for i in sorted(set(state["burst"]))]), frames=frames)
    if kind == "detector":
        cd = state["cd"]
        for m, x in enumerate(state["steps"][state["at"] % len(state["steps"])]):
            cd.set_positions(m, x)
        state["at"] += 1
        cd.updateBVH(False)
        cd.query()
        bounds = cd.bounds(0.0, 0.45)
        vertex, face, edge = cd.min_distances()
        out = dict(bounds=bounds, vertex=vertex, face=face, edge=edge)
        if case["lists"]:
            vc, vr, ec, er = cd.results()
            # the lists' filled entries (the others are not written)
            vr[np.arange(vr.shape[1]) >= vc[:, None]] = 0
            er[np.arange(er.shape[1]) >= ec[:, None]] = 0
            out.update(vcount=vc, vface=vr["face"], vtype=vr["type"], vprim=vr["prim"], vd=vr["d"], ecount=ec,
                       eedge=er["edge"], emu1=er["mu1"], emu2=er["mu2"], ed=er["d"])
        return out
    sim = state["sim"]
    for m, (x, v) in enumerate(state["states"]):
        sim.setState(m, x, v)
    sim.runSteps(case["frames"])
    both = [sim.getState(m) for m in range(len(state["states"]))]
    return dict(x=np.concatenate([b[0] for b in both]), v=np.concatenate([b[1] for b in both]))


# ---- the work that cannot be avoided ----------------------------------------------------------------

def _scene_work(kind, n, sweeps, steps):
    """(bytes, flops) of one scene: its mesh and constants read once, positions and velocities in and out; and the
    element arithmetic of `sweeps` iterations and `steps` substeps."""
    if kind == "tet":
        nv, nt = (n + 1) ** 3, 5 * n ** 3
        return (16 + 36 + 4) * nt + 52 * nv, sweeps * (4 * nt * 155 + 100 * nv) + 40 * steps * nv
    nv, nf = n * n, 2 * (n - 1) ** 2
    ne = 3 * n * n - 4 * n + 1
    return (12 + 16 + 4) * nf + (16 + 16) * ne + 52 * nv, sweeps * (3 * nf * 90 + 4 * ne * 45 + 120 * nv) + 40 * steps * nv


def work(case):
    kind = case["kind"]
    if kind in ("tet", "cloth"):
        steps = case["frames"] * case.get("substeps", 1)
        b, f = _scene_work(kind, case["n"], steps * case["iterations"], steps)
    elif kind == "batch":
        parts = [_scene_work(k, n, 10 * case["frames"], case["frames"]) for k, n in _many(case)]
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    elif kind == "serve":
        parts = [_scene_work(k, n, 10, 1) for k, n in _many(case)]
        share = case["requests"] / case["scenes"]
        b, f = sum(p[0] for p in parts), share * sum(p[1] for p in parts)
    elif kind == "detector":
        nv = case["grid"] ** 3 * case["nu"] * case["nv"]
        # positions, topology and trees in; minimum distances and bounds out; about 6 tests a primitive
        b, f = nv * (12 + 2 * 16 + 3 * 24 + 5 * 64 + 4 * 7), nv * 4 * 6 * 100
        if case["lists"]:
            b += nv * 4 * 20
    else:
        nb, n = case["bodies"], case["n"]
        one = _scene_work("tet", n, case["iterations"] * case["frames"], case["frames"])
        b, f = nb * one[0], nb * one[1]
        surface = 6 * n * n * nb  # boundary vertices
        if kind == "contact":
            s = _scene_work("cloth", case["sheet"], case["iterations"] * case["frames"], case["frames"])
            b, f = b + s[0], f + s[1]
            surface += case["sheet"] ** 2
        b += surface * (2 * 16 + 3 * 16 + 5 * 64)
        f += surface * case["frames"] * 600
    return dict(bytes=float(b), flops=float(f))


def tolerance(case):
    """Of single-precision sums in another order over a whole rollout: about four times what was measured against
    `exact`, and for the contact rollouts against other lane counts of the solve (which sum the elements of a vertex in
    another order). Velocities are the larger: they are differences of positions over the time step."""
    kind = case["kind"]
    if kind == "serve" or (kind == "tet" and not case["accelerated"]):
        return {"rel": 1e-4, "max": 1e-2}  # seen: 1.5e-5 to 3e-5
    if kind == "tet":
        return {"rel": 4e-3, "max": 0.2}  # seen: 8e-4; the accelerator extrapolates rounding too
    if kind in ("cloth", "batch"):
        return {"rel": 5e-3, "max": 0.5}  # seen: 1.2e-3; single vertices come into compression
    if kind == "detector":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    return {"rel": 3e-2, "max": 0.9}  # seen: 9e-3, at vertices whose contact switches on or off an iteration earlier


# ---- 64-bit values ------------------------------------------------------------------------------------

def _t(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda").to(dtype)


def _groups(colors):
    """Vertices by colour, largest colour first (the solve's order)."""
    return sorted((np.flatnonzero(colors == c) for c in range(int(colors.max()) + 1)), key=lambda g: -len(g))


def _f32(v):
    return float(np.float32(v))


class _Elements:
    """One kind of element of a set of scenes: for each colour step, the (vertex, element, corner) incidences."""

    def __init__(self, elems, groups, nv):
        flat = elems.reshape(-1)
        order = np.argsort(flat, kind="stable")
        begin = np.searchsorted(flat[order], np.arange(nv + 1))
        k = elems.shape[1]
        self.steps = []
        for g in groups:
            cnt = begin[g + 1] - begin[g]
            at = np.repeat(begin[g] - np.concatenate([[0], np.cumsum(cnt)[:-1]]), cnt) + np.arange(int(cnt.sum()))
            inc = order[at]
            own = np.repeat(np.arange(len(g)), cnt)
            self.steps.append((_t(own, torch.int64), _t(inc // k, torch.int64), _t(inc % k, torch.int64)))
        self.ids = _t(elems, torch.int64)


def _solve(x, h, f, hit):
    d = torch.linalg.solve(h[hit], f[hit].unsqueeze(-1)).squeeze(-1)
    out = x.clone()
    out[hit] = x[hit] + d
    return out


def _exact_sim(kind, ns, starts, case, frames):
    """Vertex block descent in 64 bits of several scenes of one kind side by side; the state after each frame."""
    tet = kind == "tet"
    pos, elems, groups, fixed, off = [], [], [], [], 0
    for n in ns:
        if tet:
            p, e, c = _cube(n)
            free = np.ones(len(p), bool)
        else:
            p, e, c, top = _curtain(n)
            free = np.ones(len(p), bool)
            free[list(top)] = False
        for g, members in enumerate(_groups(c)):
            while len(groups) <= g:
                groups.append([])
            groups[g].append(members[free[members]] + off)
        pos.append(p)
        elems.append(e + off)
        fixed.append(~free)
        off += len(p)
    groups = [np.concatenate(g) for g in groups]
    rest, e, nv = _t(np.concatenate(pos)), np.concatenate(elems), off
    fixed = _t(np.concatenate(fixed), torch.bool)
    E = _Elements(e, groups, nv)
    ids = E.ids
    mass = torch.zeros(nv, dtype=torch.float64, device="cuda")
    damped = case.get("damped", False)
    if tet:
        D = torch.stack([rest[ids[:, k]] - rest[ids[:, 0]] for k in (1, 2, 3)], dim=2)
        vol = torch.linalg.det(D) / 6
        Di = torch.linalg.inv(D)
        mass.index_add_(0, ids.reshape(-1), (vol * TET_MAT["density"] / 4).repeat_interleave(4))
        mu, lm = TET_MAT["mu"], TET_MAT["lmbd"]
        a0 = 1 + mu / lm
    else:
        e1, e2 = rest[ids[:, 1]] - rest[ids[:, 0]], rest[ids[:, 2]] - rest[ids[:, 0]]
        nrm = torch.linalg.cross(e1, e2)
        area = nrm.norm(dim=1) / 2
        ax = e1 / e1.norm(dim=1, keepdim=True)
        ay = torch.linalg.cross(nrm / nrm.norm(dim=1, keepdim=True), ax)
        D = torch.stack([torch.stack([(e1 * ax).sum(1), (e2 * ax).sum(1)], 1),
                         torch.stack([(e1 * ay).sum(1), (e2 * ay).sum(1)], 1)], 1)
        vol, Di = area, torch.linalg.inv(D)
        mass.index_add_(0, ids.reshape(-1), (area * CLOTH_MAT["density"] / 3).repeat_interleave(3))
        mu, lm = _f32(CLOTH_MU), _f32(CLOTH_LM)
        # interior edges with the opposite vertices of their two faces, and their quadratic bending forms
        half = np.concatenate([np.stack([e[:, i], e[:, (i + 1) % 3], e[:, (i + 2) % 3]], 1) for i in range(3)])
        key = np.minimum(half[:, 0], half[:, 1]) * np.int64(nv) + np.maximum(half[:, 0], half[:, 1])
        o = np.argsort(key, kind="stable")
        pair = np.flatnonzero(key[o][1:] == key[o][:-1])
        hinge = np.concatenate([half[o[pair]], half[o[pair + 1]][:, 2:]], axis=1)
        B = _Elements(hinge, groups, nv)
        q = rest[B.ids]

        def cot(u, w):
            return (u * w).sum(1) / torch.linalg.cross(u, w).norm(dim=1)

        e01, e02, e03 = q[:, 1] - q[:, 0], q[:, 2] - q[:, 0], q[:, 3] - q[:, 0]
        e12, e13 = q[:, 2] - q[:, 1], q[:, 3] - q[:, 1]
        c01, c02, c03, c04 = cot(e02, e01), cot(e01, e03), cot(-e01, e12), cot(-e01, e13)
        K = torch.stack([c03 + c04, c01 + c02, -c01 - c03, -c02 - c04], 1)
        A2 = torch.linalg.cross(e01, e02).norm(dim=1) + torch.linalg.cross(e01, e03).norm(dim=1)
        Q = CLOTH_MAT["bending_stiffness"] * 3 * K[:, :, None] * K[:, None, :] / A2[:, None, None]
    # shape rows: corner 0 takes minus the sum of the others'
    rows = torch.cat([-Di.sum(1, keepdim=True), Di], dim=1)
    dt = _f32(_f32(DT) / case.get("substeps", 1))
    x = _t(np.concatenate([s[0] for s in starts]))
    v = _t(np.concatenate([s[1] for s in starts]))
    g = torch.tensor([0.0, _f32(GRAVITY), 0.0], dtype=torch.float64, device="cuda")
    eye = torch.eye(3, dtype=torch.float64, device="cuda")
    gh, gd = (DAMPING["damping_hydrostatic"], DAMPING["damping_deviatoric"]) if damped else (0.0, 0.0)
    cs, cb = (1e-4 / dt, 1e-4 / dt) if damped and not tet else (0.0, 0.0)
    kb, muf, epsu = 1e5, 0.1, 1.0 * dt  # ground: the default penalty stiffness, friction and friction speed
    free = ~fixed
    out = []
    for _ in range(frames):
        for _ in range(case.get("substeps", 1)):
            prev = x
            v = torch.where(fixed[:, None], torch.zeros_like(v), v + dt * g)
            y = x + dt * v
            x = y.clone()
            w1, back2, back1 = 1.0, x.clone(), x.clone()
            for it in range(case.get("iterations", 10)):
                for s, members in enumerate(groups):
                    if not len(members):
                        continue
                    m = _t(members, torch.int64)
                    n = len(members)
                    own, el, co = E.steps[s]
                    xs = x[ids[el]]
                    r = rows[el]
                    F = xs.transpose(1, 2) @ r  # sum over corners of x (outer) row
                    mv = r[torch.arange(len(el), device="cuda"), co]
                    A = vol[el]
                    f = torch.zeros(n, 3, dtype=torch.float64, device="cuda")
                    h = torch.zeros(n, 3, 3, dtype=torch.float64, device="cuda")
                    Fm = (F @ mv.unsqueeze(-1)).squeeze(-1)
                    xm, disp = x[m], x[m] - prev[m]
                    if tet:
                        c0, c1, c2 = F.unbind(2)
                        cof = torch.stack([torch.linalg.cross(c1, c2), torch.linalg.cross(c2, c0),
                                           torch.linalg.cross(c0, c1)], 2)
                        J = (c0 * cof[:, :, 0]).sum(1)
                        gg = (cof @ mv.unsqueeze(-1)).squeeze(-1)
                        f.index_add_(0, own, -A[:, None] * (mu * Fm + (lm * (J - a0))[:, None] * gg))
                        hl = torch.zeros_like(h).index_add_(0, own, (A * lm)[:, None, None] * gg[:, :, None] * gg[:, None])
                        hm = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, own, A * mu * (mv * mv).sum(1))
                        hm = hm[:, None, None] * eye
                        dh = (gh * hl + gd * hm) / dt
                        h = hl + hm + dh
                        f = f - (dh @ disp.unsqueeze(-1)).squeeze(-1)
                    else:
                        C = F.transpose(1, 2) @ F
                        G = (C - torch.eye(2, dtype=torch.float64, device="cuda")) / 2
                        S = 2 * mu * G + lm * (G[:, 0, 0] + G[:, 1, 1])[:, None, None] * torch.eye(2, dtype=torch.float64, device="cuda")
                        Sm = (S @ mv.unsqueeze(-1)).squeeze(-1)
                        f.index_add_(0, own, -A[:, None] * (F @ Sm.unsqueeze(-1)).squeeze(-1))
                        he = (mv * Sm).sum(1)[:, None, None] * eye + (mu * (mv * mv).sum(1))[:, None, None] * (F @ F.transpose(1, 2)) \
                            + (mu + lm) * Fm[:, :, None] * Fm[:, None]
                        h.index_add_(0, own, A[:, None, None] * he)
                        f = f - cs * (h @ disp.unsqueeze(-1)).squeeze(-1)
                        h = h * (1 + cs)
                        own, el, co = B.steps[s]
                        row = Q[el, co]
                        f.index_add_(0, own, -(row[:, :, None] * x[B.ids[el]]).sum(1))
                        qs = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(
                            0, own, row[torch.arange(len(el), device="cuda"), co])
                        f = f - (qs * cb)[:, None] * disp
                        h = h + (qs * (1 + cb))[:, None, None] * eye
                    mi = mass[m] / dt ** 2
                    f = f + mi[:, None] * (y[m] - xm)
                    h = h + mi[:, None, None] * eye
                    if tet:
                        pen = torch.clamp(-xm[:, 1], min=0.0)
                        below = (xm[:, 1] < 0).to(torch.float64)
                        u = disp[:, [2, 0]]
                        un = u.norm(dim=1)
                        f1 = torch.where(un > epsu, 1 / un.clamp(min=1e-300), (2 - un / epsu) / epsu)
                        c = torch.where(un > 0, muf * pen * kb * f1, torch.zeros_like(un))
                        f = f + torch.stack([-c * u[:, 1], pen * kb, -c * u[:, 0]], 1)
                        h = h + torch.diag_embed(torch.stack([c, below * kb, c], 1))
                    hit = (f * f).sum(1) > 1e-10 if tet else torch.ones(n, dtype=torch.bool, device="cuda")
                    x[m] = _solve(xm, h, f, hit)
                if case.get("accelerated", False):
                    rho2 = _f32(RHO) ** 2
                    w1 = 1.0 if it == 0 else (2 / (2 - rho2) if it == 1 else 4 / (4 - rho2 * w1))
                    x = torch.where(free[:, None], back2 + w1 * (x - back2), x)
                    back2, back1 = back1, x.clone()
                    x = x.clone()
            v = (x - prev) / dt
            v = torch.where(((v.norm(dim=1) > 1e-6) & free)[:, None], v, torch.zeros_like(v))
        out.append((x.cpu().numpy(), v.cpu().numpy()))
    sizes = np.cumsum([0] + [len(p) for p in pos])
    return [[(xf[a:b], vf[a:b]) for xf, vf in out] for a, b in zip(sizes[:-1], sizes[1:])]


def _point_triangle(p, a, b, c):
    """Distance of points to triangles (broadcast), by the closest of the face's and its edges' points."""
    ab, ac, ap = b - a, c - a, p - a
    n = torch.linalg.cross(ab, ac)
    nn = (n * n).sum(-1)
    w = (torch.linalg.cross(ab.expand_as(ap), ap) * n).sum(-1) / nn
    v = (torch.linalg.cross(ap, ac.expand_as(ap)) * n).sum(-1) / nn
    inside = (v >= 0) & (w >= 0) & (v + w <= 1)
    d = torch.where(inside, (ap * n).sum(-1).abs() / nn.sqrt(), torch.full_like(v, math.inf))
    for s, e in ((a, ab), (b, c - b), (a, ac)):
        t = (((p - s) * e).sum(-1) / (e * e).sum(-1)).clamp(0, 1)
        d = torch.minimum(d, (p - s - t.unsqueeze(-1) * e).norm(dim=-1))
    return d


def _exact_detector(case, seed):
    meshes, steps = _tori(case, seed)
    nvm, nfm = case["nu"] * case["nv"], 2 * case["nu"] * case["nv"]
    nv, nf = nvm * len(meshes), nfm * len(meshes)
    if nv * nf > 1.5e8:
        return None
    r = _f32(0.002)
    x = _t(np.concatenate(steps[0]))
    f = np.concatenate([faces + m * nvm for m, (_, faces) in enumerate(meshes)])
    F = _t(f, torch.int64)
    face = torch.full((nf,), r, dtype=torch.float64, device="cuda")
    vert = torch.full((nv,), r, dtype=torch.float64, device="cuda")
    a, b, c = (x[F[:, k]] for k in range(3))
    for s in range(0, nv, 256):
        p = x[s:s + 256]
        d = _point_triangle(p[:, None], a[None], b[None], c[None])
        own = (F[None] == torch.arange(s, s + len(p), device="cuda")[:, None, None]).any(-1)
        d = torch.where(own, torch.full_like(d, r), d)
        vert[s:s + 256] = torch.minimum(vert[s:s + 256], d.amin(1))
        face = torch.minimum(face, d.amin(0))
    # a segment pair's distance takes the routine's absolute parallel threshold, which edges of this size always
    # meet, so it is not the geometric one: no 64-bit value for the edges, nor for the bounds made from them
    return dict(bounds=None, vertex=vert.cpu().numpy(), face=face.cpu().numpy(), edge=None)


def exact(case, seed):
    kind = case["kind"]
    rng = _rng(seed)
    if kind in ("tet", "cloth"):
        x, v = _exact_sim(kind, [case["n"]], [_start(rng, kind, case["n"])], case, case["frames"])[0][-1]
        return dict(x=x, v=v)
    if kind in ("batch", "serve"):
        many = _many(case)
        starts = [_start(rng, k, n) for k, n in many]
        if kind == "batch":
            last = [case["frames"]] * len(many)
        else:
            burst = _burst(rng, case)
            last = [burst.count(i) for i in range(len(many))]
        got = {}
        for k in ("tet", "cloth"):
            at = [i for i, m in enumerate(many) if m[0] == k and last[i]]
            if at:
                sims = _exact_sim(k, [many[i][1] for i in at], [starts[i] for i in at], {}, max(last[i] for i in at))
                got.update({i: s[last[i] - 1] for i, s in zip(at, sims)})
        out = dict(x=np.concatenate([got[i][0] for i in sorted(got)]), v=np.concatenate([got[i][1] for i in sorted(got)]))
        if kind == "serve":
            out["frames"] = None
        return out
    if kind == "detector":
        got = _exact_detector(case, seed)
        if got is not None and case["lists"]:
            got.update({k: None for k in ("vcount", "vface", "vtype", "vprim", "vd", "ecount", "eedge", "emu1", "emu2", "ed")})
        return got
    return None
