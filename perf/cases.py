"""The work that a user of this framework has it do, as measurable cases.

A case is one simulation (or one network) and one pass over it through the public binding
(`lsdem2.0_amd/lsdem.py`, a thin layer over the C ABI).  A pass over a simulation restarts it from the
poses and velocities of its start (`set_particles`, `set_walls`, as a parameter sweep, a restart from a
saved frame or a repeated rollout does) and takes its steps; what comes back is the bodies' state, the
library's own device arrays (`device_view`), or host frames where the case is about frames.  Every
simulation starts close to contact and moving, so that candidate pairs, certificates, contacts,
tangential history and rebuilds all occur within a pass, and every pass takes the same path from the
same start, however often it is repeated.

Kinds, with what they stand for:

  box       superellipsoids in a closed box (1 shape, 6 walls): the tutorial scale; `per_call` = 1 is an
            app that steps one by one with host work in between, where launches and latency count
  packed    an ordered dense bed of the same shape, every particle touching its neighbours and the walls:
            a settled packing, where most pairs are evaluated every step
  frames    a packed bed, some steps, then the frame an app writes: all bodies and the contact lists
  column    superquadrics of 10 types and scattered sizes, periodic in x and y, above a floor
  surrogate the same column with the learned culling network switched on (audits included)
  hook      the same column with an external-force hook (the tutorials' damping helper) on every step
  sector    the same column with quarter-sector rotational periodicity
  drums     an ensemble of rotating drums in one simulation, replayed from a captured graph
  bonded    bonded agglomerate of 3 shapes between closing walls
  net       the culling network's own directions: forward (eval) and backward (gradient)
  train     the network's training on the shapes' grids
"""
from __future__ import annotations

import ctypes
import functools
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parents[1]


def _package():
    """lsdem2.0_amd (its folder's name is no identifier) as `lsdem_amd`, with its submodules."""
    if "lsdem_amd" not in sys.modules:
        pkg = ROOT / "lsdem2.0_amd"
        spec = importlib.util.spec_from_file_location("lsdem_amd", pkg / "__init__.py",
                                                      submodule_search_locations=[str(pkg)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["lsdem_amd"] = mod
        spec.loader.exec_module(mod)
    import lsdem_amd.lsdem as L
    import lsdem_amd.scenes as S
    return L, S


# ----------------------------------------------------------------------------------------------
# Cases
# ----------------------------------------------------------------------------------------------
def listed():
    return [
        # an app's own loop over a tutorial-sized box: one step a call
        {"name": "box27-single-steps", "kind": "box", "n": 27, "steps": 50, "per_call": 1},
        # the settling box: 1,000 superellipsoids, 40^3 grids, 500 nodes
        {"name": "box1000", "kind": "box", "n": 1000, "steps": 200, "per_call": 200},
        # a settled packing, tens of thousands of touching particles
        {"name": "packed27k", "kind": "packed", "n": 27000, "steps": 50, "per_call": 50},
        # a frame every 50 steps: bodies and contact lists to the host
        {"name": "frames1728", "kind": "frames", "n": 1728, "steps": 50, "per_call": 50},
        # the roofline workload's column at its full size and at an everyday one
        {"name": "column200k", "kind": "column", "n": 200000, "steps": 400, "per_call": 400},
        {"name": "column20k", "kind": "column", "n": 20000, "steps": 200, "per_call": 200},
        # learned culling in the loop
        {"name": "surrogate20k", "kind": "surrogate", "n": 20000, "steps": 200, "per_call": 200},
        # damped settling through the external-force hook
        {"name": "hook3001", "kind": "hook", "n": 3001, "steps": 100, "per_call": 100},
        # quarter-sector periodicity (pairs rebuilt on every step)
        {"name": "sector4000", "kind": "sector", "n": 4000, "steps": 50, "per_call": 50},
        # 256 uneven drums in one simulation, 100-step graphs
        {"name": "drums256-graph", "kind": "drums", "n": 256, "steps": 200, "per_call": 100},
        # bonded agglomerate under compression
        {"name": "bonded8000", "kind": "bonded", "n": 8000, "steps": 200, "per_call": 200},
        # training of the culling network
        {"name": "train", "kind": "train", "n": 2000000, "steps": 300, "per_call": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["box", "box", "packed", "frames", "column", "column", "surrogate", "hook", "sector", "drums",
                       "bonded", "net"])
    if kind == "box":
        n = _log(rng, 8, 4000)
        steps = rng.randrange(20, 201)
        return {"kind": kind, "n": n, "steps": steps, "per_call": rng.choice([1, 7, steps])}
    if kind == "packed":
        return {"kind": kind, "n": _log(rng, 300, 27000), "steps": 2 * rng.randrange(10, 26), "per_call": 10}
    if kind == "frames":
        steps = rng.randrange(10, 60)
        return {"kind": kind, "n": _log(rng, 100, 4000), "steps": steps, "per_call": steps}
    if kind == "column":
        n = _log(rng, 800, 200000)
        steps = rng.randrange(100, 301)
        return {"kind": kind, "n": n, "steps": steps, "per_call": rng.choice([10, 64, steps])}
    if kind == "surrogate":
        steps = rng.randrange(100, 250)
        return {"kind": kind, "n": _log(rng, 1000, 30000), "steps": steps, "per_call": steps}
    if kind == "hook":
        steps = rng.randrange(40, 150)
        return {"kind": kind, "n": _log(rng, 500, 20000), "steps": steps, "per_call": steps}
    if kind == "sector":
        steps = rng.randrange(20, 60)
        return {"kind": kind, "n": _log(rng, 500, 8000), "steps": steps, "per_call": steps}
    if kind == "drums":
        return {"kind": kind, "n": _log(rng, 4, 256), "steps": 100 * rng.randrange(1, 4), "per_call": 50}
    if kind == "bonded":
        steps = rng.randrange(50, 250)
        return {"kind": kind, "n": _log(rng, 216, 12000), "steps": steps, "per_call": steps}
    return {"kind": kind, "n": 64 * _log(rng, 4, 512), "steps": 1, "per_call": 1}


# ----------------------------------------------------------------------------------------------
# Scenes.  Shapes are made once a process (a user's program loads its shapes once, too); poses,
# velocities, sizes and kinds come from the seed.
# ----------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _shapes(which):
    """The shapes of the framework's own scenes: 10 superquadric types (50^3, 512 nodes), 8 drum types
    (32^3, 300 nodes) and the drum wall, or the 3 agglomerate types (40^3, 400 nodes)."""
    _, S = _package()
    if which == "column":
        return S.scene_c2(n=8).shapes[:10]
    if which == "drums":
        return S.scene_drum_ensemble([1], [1.0], [0.5], [0.5]).shapes
    return S.scene_c3(n=8, bonds=False).shapes[:3]


def _radius(s):
    """Largest distance of a node from its shape's origin."""
    return float(np.linalg.norm(s["nodes"], axis=1).max())


def _random_quats(rng, n):
    q = rng.normal(0.0, 1.0, (n, 4))
    return q / np.linalg.norm(q, axis=1, keepdims=True)


def _bodies(shapes, kind, scale, pos, quat, vel, angvel, mu=0.5, e=0.5):
    """Particles of the given kinds and sizes at 2,500 kg/m^3 with the configurations' contact law."""
    n = len(kind)
    mass = np.array([s["mass"] for s in shapes])[kind] * scale ** 3
    inertia = np.array([s["inv_inertia"] for s in shapes])[kind] / (scale ** 5)[:, None]
    return {"shape": kind.astype(np.int32), "scale": scale, "pos": pos, "quat": quat, "vel": vel, "angvel": angvel,
            "inv_mass": 1.0 / mass, "inv_inertia": inertia, "kn": np.full(n, 1e5), "ks": np.full(n, 4e4),
            "mu": np.full(n, 1.0) * mu, "e": np.full(n, 1.0) * e}


def _column(n, seed, vel):
    """Superquadrics of 10 types and lognormal sizes (median 3 mm, sigma 0.25), the largest first, in
    square layers 4 % tighter than the layer's largest bounding diameter, above a floor; periodic in x
    and y on a 0.3 m cell (a smaller one for fewer particles)."""
    _, S = _package()
    rng = np.random.default_rng(seed)
    shapes = list(_shapes("column"))
    cell = 0.3 * min(1.0, max(0.1, (n / 200000.0) ** (1.0 / 3.0)))
    kind = rng.integers(0, len(shapes), n)
    scale = 3e-3 * np.exp(0.25 * rng.standard_normal(n))
    bound = np.array([_radius(s) for s in shapes])[kind] * scale
    order = np.argsort(-bound, kind="stable")
    pos = np.zeros((n, 3))
    z, at = 0.0, 0
    while at < n:
        pitch = 2.0 * bound[order[at]] * 0.96
        m = max(1, int(cell / pitch))
        take = order[at:at + m * m]
        k = np.arange(len(take))
        slack = 0.5 * max(0.0, cell / m - pitch)
        zc = bound[order[at]] * 1.001 if at == 0 else z + 0.5 * pitch
        pos[take, 0] = (k % m + 0.5) * (cell / m) + rng.uniform(-slack, slack, len(take))
        pos[take, 1] = (k // m + 0.5) * (cell / m) + rng.uniform(-slack, slack, len(take))
        pos[take, 2] = zc
        z = zc + 0.5 * pitch
        at += len(take)
    top = z + 0.05
    y0 = top - cell  # max.y >= max.z, as the reference's ghost test wants it
    pos[:, 1] += y0
    cfg = {"domain_min": (0.0, y0, 0.0), "domain_max": (cell, y0 + cell, top), "gravity": (0.0, 0.0, -9.81),
           "dt": 5e-6, "periodic_x": 1, "periodic_y": 1}
    sc = S.Scene(cfg=cfg, shapes=shapes)
    sc.particles = _bodies(shapes, kind, scale, pos, _random_quats(rng, n), rng.normal(0.0, vel, (n, 3)),
                           rng.normal(0.0, 5.0, (n, 3)))
    sc.walls = S.floor_wall(shapes, (0.5 * cell, y0 + 0.5 * cell), 0.0, 0.75 * cell, 0.5, 0.5)
    return sc


def _box(n, seed):
    """scenes.scene_c1's box with a lattice tight enough for contacts from the start."""
    _, S = _package()
    pitch = 10.4e-3
    layers = -(-n // 81)
    sc = S.scene_c1(n=n, seed=seed, lattice=pitch, jitter=0.1e-3,
                    box=(9.02 * pitch, 9.02 * pitch, max(0.1, pitch * (layers + 2))))
    rng = np.random.default_rng(seed + 1)
    sc.particles["vel"] = rng.normal(0.0, 0.1, (n, 3))
    sc.particles["angvel"] = rng.normal(0.0, 5.0, (n, 3))
    return sc


TOUCH = 1.5e-5  # the half distance at which two such faces, as their grids interpolate them, just touch


def _packed(n, seed):
    """An ordered bed: particles of semi-axes 5/4/3 mm (exponent 4) axis by axis, face to face, each
    turned by a half-turn about one of its axes or not, filling a box from its floor up; the time step
    of such a stiff bed (many nodes per face)."""
    _, S = _package()
    rng = np.random.default_rng(seed)
    m = max(2, round(n ** (1.0 / 3.0)))
    axes = np.array([5e-3, 4e-3, 3e-3]) + TOUCH
    k = np.arange(n)
    at = np.stack([k % m, (k // m) % m, k // (m * m)], 1)
    box = 2.0 * axes * np.array([m, m, at[:, 2].max() + 1])
    sc = S.scene_c1(n=n, seed=seed, box=tuple(box + np.array([0.0, 0.0, 0.02])), dt=2e-6)
    P = sc.particles
    P["pos"] = (2.0 * at + 1.0) * axes + rng.uniform(-1e-6, 1e-6, (n, 3))
    half = rng.integers(0, 4, n)  # identity or a half-turn about x, y or z
    P["quat"] = np.eye(4)[half] + rng.normal(0.0, 1e-4, (n, 4))
    P["quat"] /= np.linalg.norm(P["quat"], axis=1, keepdims=True)
    P["vel"] = rng.normal(0.0, 2e-3, (n, 3))
    return sc


def _sector(n, seed):
    sc = _column(n, seed, 0.3)
    sc.cfg.update(periodic_x=0, periodic_y=0, periodic_sector=1)
    return sc


def _drums(count, seed):
    """`count` rotating drums (radius 0.1 m, depth 0.05 m, 1-30 rpm, uneven fillings, friction and
    restitution of their own) on a square array in one domain, their particles touching here and there."""
    _, S = _package()
    rng = np.random.default_rng(seed)
    shapes = list(_shapes("drums"))
    types, wall = shapes[:-1], shapes[-1]
    rb = max(_radius(s) for s in types)
    radius, depth = 0.1, 0.05
    # sites bottom-up; 20,000 (the largest count of the size distribution) fills half of them
    pitch = 2.0 * rb * 0.93
    g, gy = np.arange(-radius + rb, radius - rb, pitch), np.arange(-0.5 * depth + rb, 0.5 * depth - rb + 1e-9, pitch)
    site = np.stack([a.ravel() for a in np.meshgrid(g, gy, g, indexing="ij")], 1)
    site = site[np.hypot(site[:, 0], site[:, 2]) <= radius - rb]
    site = site[np.argsort(site[:, 2], kind="stable")]
    half_fill = len(site) // 2
    sizes = np.clip(np.random.default_rng(count).lognormal(math.log(4000.0), 0.8, count), 500, 20000) / 20000.0
    sizes = np.maximum(1, np.round(sizes * half_fill)).astype(int)
    half_box = 0.5 * (wall["sdf"].shape[2] - 1) * wall["spacing"]
    side = int(math.ceil(math.sqrt(count)))
    k = np.arange(count)
    centre = np.stack([k % side, 0 * k, k // side], 1) * (2.0 * half_box + 0.06)
    drum = np.repeat(k, sizes)
    n = len(drum)
    pos = centre[drum] + np.concatenate([site[:m] for m in sizes]) + rng.uniform(-1e-5, 1e-5, (n, 3))
    mu, e = rng.uniform(0.1, 0.8, count), rng.uniform(0.3, 0.9, count)
    margin = half_box + wall["spacing"]
    lo, hi = centre.min(0) - margin, centre.max(0) + margin
    lo[1], hi[1] = -0.5 * depth - 4 * wall["spacing"], 0.5 * depth + 4 * wall["spacing"]
    sc = S.Scene(cfg={"domain_min": tuple(lo), "domain_max": tuple(hi), "gravity": (0.0, 0.0, -9.81), "dt": 1e-5},
                 shapes=shapes)
    sc.particles = _bodies(types, rng.integers(0, len(types), n), np.ones(n), pos, _random_quats(rng, n),
                           rng.normal(0.0, 0.2, (n, 3)), rng.normal(0.0, 5.0, (n, 3)), mu[drum], e[drum])
    spin = np.zeros((count, 3))
    spin[:, 1] = rng.uniform(1.0, 30.0, count) * 2.0 * math.pi / 60.0
    sc.walls = {"shape": np.full(count, len(types), np.int32), "radius": np.full(count, math.hypot(radius, 0.5 * depth)),
                "pos": centre, "quat": np.tile([1.0, 0.0, 0.0, 0.0], (count, 1)), "vel": np.zeros((count, 3)),
                "angvel": spin, "mu": mu, "e": e}
    return sc


def _bonded(n, seed):
    """A bonded agglomerate (exponents 2/3/6) on a cubic lattice whose neighbours nearly touch, between
    walls closing at 0.05 m/s: bonds between neighbours whose surfaces are closer than 0.1 mm, radius 0.8
    x the smaller particle, E 1e8, Weibull(5, 1e6) strengths."""
    _, S = _package()
    rng = np.random.default_rng(seed)
    shapes = list(_shapes("bonded"))
    reach = np.array([np.abs(s["nodes"]).max(axis=0) for s in shapes])  # along each axis, unscaled
    pitch = 5.0e-3
    m = int(math.ceil(n ** (1.0 / 3.0)))
    k = np.arange(n)
    at = np.stack([k % m, (k // m) % m, k // (m * m)], 1)
    kind = rng.integers(0, len(shapes), n)
    scale = rng.uniform(2.46e-3, 2.5e-3, n) / reach.max(1)[kind]
    pos = (at + 0.5) * pitch + rng.uniform(-4e-6, 4e-6, (n, 3))
    quat = np.array([1.0, 0.0, 0.0, 0.0]) + rng.normal(0.0, 2e-3, (n, 4))  # as compacted grains: facing alike
    quat /= np.linalg.norm(quat, axis=1, keepdims=True)
    lo, hi = np.zeros(3), (at.max(axis=0) + 1) * pitch
    margin = 0.2 * m * pitch + 0.01
    sc = S.Scene(cfg={"domain_min": tuple(lo - margin), "domain_max": tuple(hi + margin), "gravity": (0.0, 0.0, 0.0),
                      "dt": 2e-6}, shapes=shapes)
    sc.particles = _bodies(shapes, kind, scale, pos, quat, rng.normal(0.0, 0.02, (n, 3)), rng.normal(0.0, 1.0, (n, 3)))
    sc.walls = S.box_walls(shapes, lo, hi, 0.5, 0.5)
    sc.walls["vel"][0], sc.walls["vel"][1] = (0.0, 0.0, 0.05), (0.0, 0.0, -0.05)
    for axis, stride in enumerate((1, m, m * m)):
        i = k[(at[:, axis] < m - 1) & (k + stride < n)]
        j = i + stride
        d = pos[i] - pos[j]
        dist = np.linalg.norm(d, axis=1)
        to_j = reach[kind[j], axis] * scale[j]
        gap = dist - reach[kind[i], axis] * scale[i] - to_j
        normal = d / dist[:, None]
        point = pos[j] + normal * (to_j + 0.5 * np.maximum(gap, 0.0))[:, None]
        r = 0.8 * np.minimum(scale[i], scale[j])
        strength = 1e6 * rng.weibull(5.0, (len(i), 2))
        for t in np.flatnonzero(gap < 1e-4):
            sc.bonds.append((int(i[t]), int(j[t]), point[t], normal[t], float(r[t]), float(dist[t]), 1e8, 0.3,
                             float(strength[t, 0]), float(strength[t, 1]), 0.0))
    return sc


def _scene(case, seed):
    kind, n = case["kind"], int(case["n"])
    seed = int(seed) % (1 << 31)
    if kind == "box":
        return _box(n, seed)
    if kind in ("packed", "frames"):
        return _packed(n, seed)
    if kind == "column":
        return _column(n, seed, 0.2)
    if kind == "hook":
        return _column(n, seed, 0.2)
    if kind == "surrogate":
        return _column(n, seed, 0.2)
    if kind == "sector":
        return _sector(n, seed)
    if kind == "drums":
        return _drums(n, seed)
    if kind == "bonded":
        return _bonded(n, seed)
    return _column(64, seed, 0.0)  # net, train: the shapes alone count


class _DeviceArray:
    """A device array of the library for torch.as_tensor.  The tensor keeps this object, and this object
    the simulation that owns the memory, for as long as the tensor is there."""

    def __init__(self, sim, ptr, shape):
        self.sim = sim
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f8", "data": (int(ptr), False), "version": 3,
                                         "strides": None}


def _views(sim):
    v = sim.device_view()
    n = int(v.num)
    out = {k: torch.as_tensor(_DeviceArray(sim, getattr(v, f), (n, w)), device="cuda")
           for k, f, w in (("pos", "position", 3), ("quat", "quaternion", 4), ("vel", "velocity", 3),
                           ("angvel", "angular_velocity", 3), ("force", "force", 3), ("torque", "torque", 3))}
    return out


# ----------------------------------------------------------------------------------------------
# The culling network's inputs
# ----------------------------------------------------------------------------------------------
N_SHAPES, N_FREQ, N_EMB, N_IN, N_HID = 10, 16, 16, 112, 64


def _net_inputs(n, seed, scene):
    """Weights (He-normal), local points in the shapes' boxes, their shapes and targets."""
    rng = np.random.default_rng(int(seed) % (1 << 31))
    w = [rng.normal(0, math.sqrt(2.0 / N_IN), N_IN * N_HID), np.zeros(N_HID)]
    for _ in range(3):
        w += [rng.normal(0, math.sqrt(2.0 / N_HID), N_HID * N_HID), np.zeros(N_HID)]
    w += [rng.normal(0, math.sqrt(1.0 / N_HID), N_HID), np.zeros(1), rng.normal(0, 0.5, N_SHAPES * N_EMB)]
    half = max(0.5 * (s["sdf"].shape[0] - 1) * s["spacing"] for s in scene.shapes[:N_SHAPES])
    return (np.concatenate(w).astype(np.float32), rng.uniform(-half, half, (n, 3)).astype(np.float32),
            rng.integers(0, N_SHAPES, n).astype(np.int32), rng.uniform(-0.6, 0.6, n).astype(np.float32))


# ----------------------------------------------------------------------------------------------
# prepare, run
# ----------------------------------------------------------------------------------------------
def prepare(case, seed):
    L, _ = _package()
    sc = _scene(case, seed)
    sim = sc.load(L.Sim(sc.cfg))
    kind = case["kind"]
    state = {"sim": sim, "case": case, "kind": kind}
    if kind == "train":
        state["seed"] = 1 + int(seed) % (1 << 31)
        return state
    if kind == "net":
        w, x, shape, t = _net_inputs(int(case["n"]), seed, sc)
        sim.surrogate_set_weights(w)
        state.update(x=x, shape=shape, t=t)
        return state
    if kind == "surrogate":
        sim.surrogate_train(iterations=300, samples=500000, validation=65536)
        sim.surrogate_enable(True)
    if kind == "hook":
        damp = sim.lib.launchAddGlobalDampingForceTorque
        damp.restype = None
        damp.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_double] + [ctypes.c_size_t] * 3 + [ctypes.c_void_p]
        sim.set_external_force(lambda time, v: damp(v.force, v.torque, v.velocity, v.angular_velocity, 0.3, v.num,
                                                    v.grid_dim, v.block_dim, v.stream))
    p = sc.particles
    zero = np.zeros_like(p["pos"])
    state["start"] = {"pos": p["pos"], "quat": sim.get_particles()["quat"], "vel": p["vel"], "angvel": p["angvel"],
                      "force": zero, "torque": zero}
    state["walls"] = sim.get_walls() if sim.n_walls else None
    if kind == "frames":  # a frame's buffers, of a fixed capacity
        rows = 24 * sim.n_particles
        state["frame"] = {lst: {k: np.zeros((rows, *w), t) for k, w, t in (
            ("master", (), np.int32), ("slave", (), np.int32), ("point", (3,), float), ("normal", (3,), float),
            ("overlap", (), float), ("spring", (3,), float), ("energy_n", (), float), ("energy_s", (), float))}
            for lst in ("pp", "pw")}
    else:
        state["views"] = _views(sim)
    return state


def run(state):
    sim, case, kind = state["sim"], state["case"], state["kind"]
    if kind == "train":
        sim.surrogate_train(iterations=int(case["steps"]), batch=int(case["per_call"]), samples=int(case["n"]),
                            seed=state["seed"])
        return sim.surrogate_weights(N_SHAPES)
    if kind == "net":
        out = sim.surrogate_eval(state["x"], state["shape"])
        loss, grad = sim.surrogate_gradient(state["x"], state["shape"], state["t"], N_SHAPES)
        return {"out": out, "loss": loss, "grad": grad}
    sim.set_particles(**state["start"])
    if state["walls"] is not None:
        sim.set_walls(**state["walls"])
    steps, per = int(case["steps"]), int(case["per_call"])
    step = sim.step_graph if kind == "drums" else sim.step
    for done in range(0, steps, per):
        step(min(per, steps - done))
    if kind == "frames":
        for which, name in enumerate(("pp", "pw")):
            found = sim.contacts(which)
            for k, a in state["frame"][name].items():
                m = len(found[k])
                a[:m], a[m:] = found[k], 0
        return {"bodies": sim.get_particles(), **state["frame"]}
    if kind == "bonded":
        return {**state["views"], "bonds": sim.bonds()}
    return state["views"]


# ----------------------------------------------------------------------------------------------
# work: the bodies' state in and out once a step (pose, velocities: 13 doubles; force and torque out: 6),
# and the arithmetic of its integration
# ----------------------------------------------------------------------------------------------
def work(case):
    kind, n, steps = case["kind"], int(case["n"]), int(case["steps"])
    if kind == "train":
        per = 3.0 * 2.0 * (N_IN * N_HID + 3 * N_HID * N_HID + N_HID) * case["per_call"]
        return {"bytes": 20.0 * n + steps * 20.0 * (19777 + N_EMB * N_SHAPES), "flops": steps * per}
    if kind == "net":
        return {"bytes": 36.0 * n + 8.0 * 19777, "flops": 4.0 * 2.0 * (N_IN * N_HID + 3 * N_HID * N_HID + N_HID) * n}
    bodies = 117 * n if kind == "drums" else n
    return {"bytes": float(bodies) * steps * (2 * 13 + 6) * 8, "flops": 300.0 * bodies * steps}


# ----------------------------------------------------------------------------------------------
# exact: the network in 64 bits, and the boxes (one particle shape, walls, no periodicity) stepped by
# plain torch in 64 bits
# ----------------------------------------------------------------------------------------------
def _net_exact(case, seed):
    sc = _scene(case, seed)
    w, x, shape, t = (torch.from_numpy(np.asarray(a)) for a in _net_inputs(int(case["n"]), seed, sc))
    w = w.double().requires_grad_(True)
    at, parts = 0, []
    for r, c in ((N_IN, N_HID), (1, N_HID)) + ((N_HID, N_HID), (1, N_HID)) * 3 + ((N_HID, 1), (1, 1),
                                                                                 (N_SHAPES, N_EMB)):
        parts.append(w[at:at + r * c].reshape(r, c))
        at += r * c
    box = 0.0
    for s in sc.shapes[:N_SHAPES]:
        hi = s["origin"] + (np.array(s["sdf"].shape[::-1]) - 1) * s["spacing"]
        box = max(box, float(np.linalg.norm(np.maximum(np.abs(s["origin"]), np.abs(hi)))))
    u = x.double() / box
    f = math.pi * 2.0 ** (torch.arange(N_FREQ, dtype=torch.float64) / 3.0)
    a = u[:, :, None] * f
    h = torch.cat([torch.stack([a.sin(), a.cos()], -1).reshape(len(u), -1), parts[-1][shape.long()]], 1)
    for k in range(4):
        h = torch.nn.functional.silu(h @ parts[2 * k] + parts[2 * k + 1])
    out = (h @ parts[8] + parts[9])[:, 0]
    loss = ((out - t.double()) ** 2).mean()
    loss.backward()
    return {"out": (out.detach() * box).numpy(), "loss": float(loss.detach()), "grad": w.grad.numpy()}


def _rot(q, v):
    u, v = torch.broadcast_tensors(q[..., 1:], v)
    t = 2.0 * torch.linalg.cross(u, v)
    return v + q[..., :1] * t + torch.linalg.cross(u, t)


def _conj(q):
    return q * q.new_tensor([1.0, -1.0, -1.0, -1.0])


def _grid_hits(sdf, origin, h, loc):
    """Points inside a level-set grid with a value <= 0: their indices, overlap (minus the trilinear
    value) and gradient, the gradient's x weight that of the cell's lower corner (the reference's)."""
    g = (loc - origin) * (1.0 / h)
    i = torch.floor(g).long()
    top = torch.tensor(sdf.shape[::-1], device=loc.device) - 1
    at = ((i >= 0) & (i < top)).all(-1).nonzero()[:, 0]
    g, i = g[at], i[at]
    f = g - i
    c = [sdf[i[:, 2] + (k >> 2), i[:, 1] + ((k >> 1) & 1), i[:, 0] + (k & 1)] for k in range(8)]

    def mix(v, *axes):  # v over the corners left, weights by axis
        for w in axes:
            v = [v[k] * (1 - w) + v[k + 1] * w for k in range(0, len(v), 2)]
        return v[0]

    x, y, z = f[:, 0], f[:, 1], f[:, 2]
    ov = -mix(c, x, y, z)
    keep = ov >= 0
    x0 = torch.zeros_like(x)
    gx = mix([c[k + 1] - c[k] for k in (0, 2, 4, 6)], y, z)
    gy = mix([c[k + 2] - c[k] for k in (0, 1, 4, 5)], x0, z)
    gz = mix([c[k + 4] - c[k] for k in (0, 1, 2, 3)], x0, y)
    return at[keep], ov[keep], torch.stack([gx, gy, gz], -1)[keep]


def _box_exact(case, seed):
    sc = _scene(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    T = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=dev)  # noqa: E731
    P, W, S = sc.particles, sc.walls, sc.shapes
    shape, wall = S[P["shape"][0]], S[W["shape"][0]]
    node, sdf, org, h = T(shape["nodes"]), T(shape["sdf"]), T(shape["origin"]), shape["spacing"]
    wsdf, worg, wh = T(wall["sdf"]), T(wall["origin"]), wall["spacing"]
    x, q, v, w = (T(P[k]).clone() for k in ("pos", "quat", "vel", "angvel"))
    q = q / q.norm(dim=1, keepdim=True)
    F, M = torch.zeros_like(x), torch.zeros_like(x)
    wx, wq = T(W["pos"]), T(W["quat"])
    wq = wq / wq.norm(dim=1, keepdim=True)
    im, kn, ks, mu, e = (float(P[k][0]) for k in ("inv_mass", "kn", "ks", "mu", "e"))
    xx, yy, zz, xy, xz, yz = (float(t) for t in P["inv_inertia"][0])
    inv = T([[xx, xy, xz], [xy, yy, yz], [xz, yz, zz]])
    grav, dt = T(sc.cfg["gravity"]), sc.cfg["dt"]
    r = float(node.norm(dim=1).max())
    nn, n, nw = len(node), len(x), len(wx)
    lr = math.log(e)
    diss = -lr / float(np.sqrt(np.float32(lr * lr + math.pi * math.pi)))
    half_thick = float(wh)
    history = (torch.zeros(0, dtype=torch.int64, device=dev), torch.zeros((0, 3), dtype=torch.float64, device=dev))

    def kick():
        nonlocal v, w
        v = v + (F * im + grav) * (0.5 * dt)
        w = w + _rot(q, _rot(_conj(q), M) @ inv.T) * (0.5 * dt)

    for _ in range(int(case["steps"])):
        kick()
        x = x + dt * v
        a = w * (0.5 * dt)
        u = q[:, 1:]
        q = q + torch.cat([-(u * a).sum(1, keepdim=True), q[:, :1] * a - torch.linalg.cross(u, a)], 1)
        q = q / q.norm(dim=1, keepdim=True)
        # node by node: particles below one another's bounding spheres, then the walls
        parts = []
        for i0 in range(0, n, 2048):
            d = torch.cdist(x[i0:i0 + 2048], x) if n <= 4096 else None
            ia, ib = ((d <= 2 * r + 1e-9) & (torch.arange(n, device=dev) > torch.arange(
                i0, min(n, i0 + 2048), device=dev)[:, None])).nonzero(as_tuple=True)
            parts.append((ia + i0, ib))
        A, B = torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])
        keys, rows = [], []
        for c0 in range(0, len(A), 20000):
            a_, b_ = A[c0:c0 + 20000], B[c0:c0 + 20000]
            pw = _rot(q[a_][:, None], node[None]) + x[a_][:, None]
            near = ((pw - x[b_][:, None]).norm(dim=2) <= r).nonzero()
            pt, a1, b1 = pw[near[:, 0], near[:, 1]], a_[near[:, 0]], b_[near[:, 0]]
            at, ov, g = _grid_hits(sdf, org, h, _rot(_conj(q[b1]), pt - x[b1]))
            nrm = _rot(q[b1[at]], g)
            keys.append((a1[at] * nn + near[at, 1]) * (n + nw) + b1[at])
            rows.append((a1[at], b1[at], pt[at], ov, nrm / nrm.norm(dim=1, keepdim=True), False))
        for k in range(nw):
            loc0 = _rot(_conj(wq[k]).expand(n, 4), x - wx[k])
            a_ = (loc0[:, 2].abs() <= r + half_thick).nonzero()[:, 0]
            pw = (_rot(q[a_][:, None], node[None]) + x[a_][:, None]).reshape(-1, 3)
            at, ov, g = _grid_hits(wsdf, worg, wh, _rot(_conj(wq[k]).expand(len(pw), 4), pw - wx[k]))
            nrm = _rot(wq[k].expand(len(at), 4), g)
            body = a_[at // nn]
            keys.append((body * nn + at % nn) * (n + nw) + n + k)
            rows.append((body, torch.full_like(body, k), pw[at], ov, nrm / nrm.norm(dim=1, keepdim=True), True))
        F, M = torch.zeros_like(x), torch.zeros_like(x)
        new = []
        order = torch.argsort(history[0])
        hk, hs = history[0][order], history[1][order]
        for key, (i, j, pt, ov, nrm, is_wall) in zip(keys, rows):
            pt = pt + 0.5 * ov[:, None] * nrm
            spring = torch.zeros_like(pt)
            if len(hk) and len(key):
                at = torch.searchsorted(hk, key).clamp(max=len(hk) - 1)
                spring = torch.where((hk[at] == key)[:, None], hs[at], spring)
            f = 1.0 if is_wall else 0.5
            kn_, ks_, m_ = kn * f, ks * f, (1.0 if is_wall else 0.5) / im
            cn = 2.0 * diss * float(np.sqrt(np.float32(m_ * kn_)))
            cs = 2.0 * diss * float(np.sqrt(np.float32(m_ * ks_)))
            arm_i = pt - x[i]
            vc = v[i] + torch.linalg.cross(w[i], arm_i)
            if not is_wall:
                vc = vc - v[j] - torch.linalg.cross(w[j], pt - x[j])
            vn = (vc * nrm).sum(1, keepdim=True) * nrm
            vs = vc - vn
            Fn = kn_ * ov[:, None] * nrm - cn * vn
            s1 = spring - (spring * nrm).sum(1, keepdim=True) * nrm
            l1 = s1.norm(dim=1, keepdim=True)
            s1 = torch.where(l1 > 1e-20, s1 * (spring.norm(dim=1, keepdim=True) / l1.clamp(min=1e-300)), s1)
            sp = s1 + vs * dt
            Fs = -ks_ * sp - cs * vs
            aF, cap = Fs.norm(dim=1, keepdim=True), mu * Fn.norm(dim=1, keepdim=True)
            slide = (aF > 1e-20) & (aF > cap)
            Fc = Fs * (cap / aF.clamp(min=1e-300))
            sp = torch.where(slide, -(Fc + cs * vs) / ks_, sp)
            Fs = -ks_ * sp - cs * vs
            tot = torch.where((ov > 0)[:, None], Fn + Fs, torch.zeros_like(Fn))
            sp = torch.where((ov > 0)[:, None], sp, torch.zeros_like(sp))
            F = F.index_add(0, i, tot)
            M = M.index_add(0, i, torch.linalg.cross(arm_i, tot))
            if not is_wall:
                F = F.index_add(0, j, -tot)
                M = M.index_add(0, j, torch.linalg.cross(pt - x[j], -tot))
            new.append((key, sp))
        history = (torch.cat([k for k, _ in new]), torch.cat([s for _, s in new]))
        kick()
    return {"pos": x, "quat": q, "vel": v, "angvel": w, "force": F, "torque": M}


def exact(case, seed):
    kind, n, steps = case["kind"], int(case["n"]), int(case["steps"])
    if kind == "net":
        return _net_exact(case, seed)
    if kind == "box" and n * steps <= 220000:
        return _box_exact(case, seed)
    if kind == "packed" and n * steps <= 100000:
        return _box_exact(case, seed)
    if kind == "frames" and n * steps <= 100000:
        none = {k: None for k in ("master", "slave", "point", "normal", "overlap", "spring", "energy_n", "energy_s")}
        return {"bodies": _box_exact(case, seed), "pp": none, "pw": none}
    return None  # (periodic images, bonds, drums and training: well over 20 s in plain torch)
