"""What a user has this framework do, as measurable cases.

Each case resets its scenes to a prepared state, steps them through a public
entry point and reads the result back, as a roll-out, a game loop or a training
step does:

  dropin  the reference's own call: rp_pbd_simulate on Entity records
  batch   falling and resting boxes and icospheres (rp_world_*), 1 to thousands
          of independent scenes
  uneven  scenes of very different sizes and hulls, some with joint chains
  chains  hanging chains of hinge and spherical joints
  mixed   spheres, boxes and compound bodies
  large   one scene of thousands of bodies (grid broad phase, coloured solve)
  throw   differentiable throws: torch.autograd forward and backward
"""
import ctypes
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent


def _package():
    """The product package (its directory's name is not an identifier)."""
    if "raw_physics_amd" not in sys.modules:
        d = ROOT / "raw-physics_amd"
        spec = importlib.util.spec_from_file_location("raw_physics_amd", d / "__init__.py",
                                                      submodule_search_locations=[str(d)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["raw_physics_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["raw_physics_amd"]


pkg = _package()
scenes = pkg.scenes
from raw_physics_amd.autograd import ThrowRun, ThrowSetup  # noqa: E402

DT, SUBSTEPS, GRAVITY = 1.0 / 60.0, 20, 10.0  # the reference's frame (src/examples/stack.cpp:86-104)


# --------------------------------------------------------------------------
# The cases
# --------------------------------------------------------------------------
# warm: frames stepped before the start state is taken (0 = still falling).
def listed():
    return [
        # a game that links the library in place of the reference's step and
        # calls it once per frame on its few entities (the reference's stack
        # example): launch- and latency-bound
        {"name": "dropin stack of 10", "kind": "dropin", "bodies": 10, "warm": 40, "iters": 1},
        # an interactive viewer: one scene, one frame, matrices for the renderer
        {"name": "viewer 1x16", "kind": "batch", "scenes": 1, "cubes": 8, "icos": 8, "subdiv": 1, "warm": 150,
         "frames": 1, "iters": 1, "render": True},
        # a small vectorised environment: 64 scenes, a few frames per action
        {"name": "batch 64x16", "kind": "batch", "scenes": 64, "cubes": 8, "icos": 8, "subdiv": 1, "warm": 120,
         "frames": 4, "iters": 1, "render": False},
        # the start of an episode: an odd number of scenes, all in free fall
        {"name": "batch 1021x13 falling", "kind": "batch", "scenes": 1021, "cubes": 6, "icos": 7, "subdiv": 1,
         "warm": 0, "frames": 10, "iters": 1, "render": False},
        # the batched workload of bench.py: 4096 scenes of 16 bodies mid-run
        {"name": "batch 4096x16", "kind": "batch", "scenes": 4096, "cubes": 8, "icos": 8, "subdiv": 1, "warm": 150,
         "frames": 20, "iters": 1, "render": False},
        # finely tessellated hulls (642 vertices) and two position iterations
        {"name": "batch 37x10 hull642", "kind": "batch", "scenes": 37, "cubes": 5, "icos": 5, "subdiv": 3, "warm": 90,
         "frames": 3, "iters": 2, "render": False},
        # piles of 4 to 256 bodies with 8-, 42- and 162-vertex hulls and chains
        {"name": "uneven 150", "kind": "uneven", "scenes": 150, "most": 256, "warm": 70, "frames": 4, "iters": 1},
        # articulated bodies: 500 chains of 6 links, four position iterations
        {"name": "chains 500x6", "kind": "chains", "scenes": 500, "length": 6, "warm": 60, "frames": 10, "iters": 4},
        # spheres and compound bodies (two hulls each)
        {"name": "mixed 256x10", "kind": "mixed", "scenes": 256, "spheres": 5, "cubes": 3, "dumbbells": 2, "warm": 90,
         "frames": 4, "iters": 1},
        # one big pile forming
        {"name": "large 20000", "kind": "large", "bodies": 20000, "warm": 60, "frames": 3, "iters": 1},
        # a short differentiable throw of a few scenes ...
        {"name": "throw 37x12", "kind": "throw", "scenes": 37, "frames": 12, "iters": 1},
        # ... and a long one of many (the bodies have hit the ramp)
        {"name": "throw 1024x30", "kind": "throw", "scenes": 1024, "frames": 30, "iters": 1},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dropin", "batch", "batch", "batch", "uneven", "chains", "mixed", "large", "throw", "throw"])
    iters = rng.choice([1, 1, 1, 2, 4])
    if kind == "dropin":
        return {"kind": kind, "bodies": rng.randint(2, 24), "warm": rng.randint(10, 50), "iters": iters}
    if kind == "batch":
        sub = rng.choice([1, 1, 1, 2, 3])
        n = _log_int(rng, 1, {1: 2000, 2: 200, 3: 37}[sub])
        return {"kind": kind, "scenes": n, "cubes": rng.randint(2, 8), "icos": rng.randint(2, 8), "subdiv": sub,
                "warm": rng.choice([0, 60, 120, 180]), "frames": rng.randint(1, 10), "iters": 1 if n > 500 else iters,
                "render": n < 100 and rng.random() < 0.5}
    if kind == "uneven":
        return {"kind": kind, "scenes": _log_int(rng, 8, 150), "most": rng.randint(40, 256),
                "warm": rng.randint(30, 90), "frames": rng.randint(1, 4), "iters": 1}
    if kind == "chains":
        return {"kind": kind, "scenes": _log_int(rng, 1, 2000), "length": rng.randint(2, 12),
                "warm": rng.randint(10, 90), "frames": rng.randint(1, 10), "iters": iters}
    if kind == "mixed":
        return {"kind": kind, "scenes": _log_int(rng, 1, 400), "spheres": rng.randint(1, 6), "cubes": rng.randint(1, 5),
                "dumbbells": rng.randint(1, 4), "warm": rng.randint(30, 120), "frames": rng.randint(1, 4), "iters": 1}
    if kind == "large":
        return {"kind": kind, "bodies": _log_int(rng, 4200, 20000), "warm": rng.randint(0, 60),
                "frames": rng.randint(1, 3), "iters": rng.choice([1, 1, 2])}
    return {"kind": "throw", "scenes": _log_int(rng, 1, 1024), "frames": rng.randint(5, 30), "iters": iters}


# --------------------------------------------------------------------------
# The drop-in's entities: rp_entity records (include/rawphys.h) in light
# arrays, whose element count is the size_t before the first element. A
# program keeps its entities and only their records' values change.
# --------------------------------------------------------------------------
_ENTITY = np.dtype({
    "names": ["id", "position", "rotation", "scale", "colliders", "radius", "forces", "inverse_mass", "inertia",
              "inverse_inertia", "angular_velocity", "linear_velocity", "fixed", "active", "deactivation_time",
              "static_friction", "dynamic_friction", "restitution", "previous_position", "previous_rotation",
              "previous_linear_velocity", "previous_angular_velocity"],
    "formats": ["u8", "3f8", "4f8", "3f8", "u8", "f8", "u8", "f8", "9f8", "9f8", "3f8", "3f8", "i4", "i4", "f8", "f8",
                "f8", "f8", "3f8", "4f8", "3f8", "3f8"],
    "offsets": [0, 24, 48, 80, 136, 144, 152, 160, 168, 240, 312, 336, 360, 364, 368, 376, 384, 392, 400, 424, 456, 480],
    "itemsize": 504})
_RECORD_STATE = {"position": "position", "rotation": "rotation", "linear_velocity": "linear_velocity",
                 "angular_velocity": "angular_velocity", "previous_position": "previous_position",
                 "previous_rotation": "previous_rotation", "previous_linear_velocity": "previous_linear_velocity",
                 "previous_angular_velocity": "previous_angular_velocity", "active": "active",
                 "deactivation_time": "deactivation_time"}


class _Entities:
    def __init__(self, world, gw):
        self.keep = []
        nb = world.num_bodies
        self.records = np.zeros(nb, dtype=_ENTITY)
        im, radius = np.zeros(nb), np.zeros(nb)
        inertia, inverse = np.zeros((nb, 9)), np.zeros((nb, 9))
        gw.lib.rp_world_body_info(gw.h, im.ctypes.data, inertia.ctypes.data, inverse.ctypes.data, radius.ctypes.data)
        material = np.asarray(world.body_material, dtype=np.float64).reshape(-1, 3)
        r = self.records
        r["id"], r["scale"], r["radius"], r["inverse_mass"] = np.arange(nb), world.body_scale, radius, im
        r["inertia"], r["inverse_inertia"], r["fixed"] = inertia, inverse, world.body_fixed
        r["static_friction"], r["dynamic_friction"], r["restitution"] = material.T
        self.transformed = []
        for b in range(nb):
            r["colliders"][b] = self._hull(gw, b)
            if not world.body_fixed[b]:  # the frame's gravity force at the origin
                force = np.zeros(1, dtype=np.dtype([("position", "3f8"), ("force", "3f8"), ("local", "i4")]))
                force["force"][0, 1] = -GRAVITY * 1.0 / im[b]
                r["forces"][b] = self._light(force, 1)
        self.pointers = np.zeros(1 + nb, dtype=np.uint64)
        self.pointers[0] = nb
        self.pointers[1:] = self.records.ctypes.data + 504 * np.arange(nb, dtype=np.uint64)

    def _light(self, data, count):
        raw = np.frombuffer(np.ascontiguousarray(data).tobytes(), dtype=np.uint8)
        buf = np.zeros(2 + (len(raw) + 7) // 8, dtype=np.uint64)
        buf[1] = count
        buf[2:].view(np.uint8)[:len(raw)] = raw
        self.keep.append(buf)
        return buf.ctypes.data + 16

    def _lists(self, off, el):
        """A light array of light arrays of u32."""
        ptr = [self._light(el[off[k]:off[k + 1]], int(off[k + 1] - off[k])) for k in range(len(off) - 1)]
        return ptr, self._light(np.array(ptr, dtype=np.uint64), len(ptr))

    def _hull(self, gw, b):
        n = np.zeros(6, dtype=np.uint32)
        gw.lib.rp_world_hull(gw.h, b, n.ctypes.data, *[None] * 10)
        nv, nf = int(n[0]), int(n[1])
        v, fn = np.zeros((nv, 3)), np.zeros((nf, 3))
        sizes = [nf + 1, int(n[2]), nv + 1, int(n[3]), nv + 1, int(n[4]), nf + 1, int(n[5])]
        t = [np.zeros(max(k, 1), dtype=np.uint32) for k in sizes]
        gw.lib.rp_world_hull(gw.h, b, n.ctypes.data, v.ctypes.data, fn.ctypes.data, *[a.ctypes.data for a in t])
        elements, _ = self._lists(t[0], t[1])
        faces = np.zeros(nf, dtype=np.dtype([("elements", "u8"), ("normal", "3f8")]))
        faces["elements"], faces["normal"] = elements, fn
        hull = [self._light(v, nv), self._light(v, nv), self._light(faces, nf), self._light(faces, nf)]
        self.transformed.append(self.keep[-3][2:].view(np.float64))  # written by the call where the body is awake
        hull += [self._lists(t[2], t[3])[1], self._lists(t[4], t[5])[1], self._lists(t[6], t[7])[1]]
        collider = np.zeros(8, dtype=np.uint64)
        collider[0] = 1  # RP_COLLIDER_CONVEX_HULL
        collider[1:] = hull
        return self._light(collider, 1)


_entities = {}  # the program's entity sets, by their number of bodies


# --------------------------------------------------------------------------
# Preparation and one pass
# --------------------------------------------------------------------------
def _world(case, seed):
    first = 100003 * (seed % 20011)
    kind = case["kind"]
    if kind == "dropin":
        return scenes.stack_scene(seed=first, num_cubes=case["bodies"])
    if kind == "batch":
        return scenes.batched_uniform(case["scenes"], first, n_cubes=case["cubes"], n_icos=case["icos"],
                                      ico_subdiv=case["subdiv"])
    if kind == "uneven":  # one set of scenes; the seed moves their initial velocities
        w = scenes.batched_uneven(case["scenes"], max_bodies=case["most"])
        v = np.asarray(w.body_linear_velocity, dtype=np.float64)
        v += np.random.default_rng(seed).normal(0.0, 0.3, v.shape) * (1 - np.asarray(w.body_fixed))[:, None]
        w.body_linear_velocity = [tuple(a) for a in v.tolist()]
        return w
    if kind == "chains":
        return scenes.chains(case["scenes"], length=case["length"], first_seed=first)
    if kind == "mixed":
        return scenes.batched_mixed(case["scenes"], first, n_spheres=case["spheres"], n_cubes=case["cubes"],
                                    n_dumbbells=case["dumbbells"])
    return scenes.large_scene(case["bodies"], seed=first)


def prepare(case, seed):
    if case["kind"] == "throw":
        desc, targets = scenes.ramps(case["scenes"], 100003 * (seed % 20011))
        setup = ThrowSetup(desc, case["frames"], dt=DT, substeps=SUBSTEPS, iters=case["iters"], gravity=GRAVITY)
        dyn = setup.dynamic
        leaf = lambda a: torch.tensor(np.asarray(a, dtype=np.float64), device="cuda")  # noqa: E731
        inputs = [leaf(setup.init["linear_velocity"][dyn]), leaf(setup.init["angular_velocity"][dyn]),
                  leaf(setup.mass0[dyn]), leaf(setup.material0[dyn, 0]), leaf(setup.material0[dyn, 1])]
        return {"case": case, "setup": setup, "inputs": inputs, "target": leaf(targets)}
    world = _world(case, seed)
    gw = pkg.World(world)
    step = {"dt": DT, "substeps": SUBSTEPS, "iters": case["iters"], "gravity": GRAVITY}
    if case["warm"]:
        gw.step(case["warm"], **step)
    state = {"case": case, "gw": gw, "step": step, "start": gw.state()}
    if case["kind"] == "dropin":
        key = case["bodies"]
        if key not in _entities:
            _entities[key] = _Entities(world, gw)
        state["entities"] = _entities[key]
    return state


def _run_dropin(s):
    e = s["entities"]
    for name, field in _RECORD_STATE.items():
        v = s["start"][name]
        e.records[field] = v[:, 0] if v.shape[1] == 1 else v
    for t in e.transformed:
        t[:] = 0.0
    err = pkg.library().rp_pbd_simulate(DT, e.pointers.ctypes.data + 8, None, SUBSTEPS, s["case"]["iters"], 1)
    if err:
        raise RuntimeError(f"rp_pbd_simulate: {err:#x}")
    out = {name: e.records[field].copy() for name, field in _RECORD_STATE.items()}
    out["transformed_vertices"] = np.concatenate(e.transformed)
    return out


def _run_throw(s):
    inputs = [t.detach().requires_grad_() for t in s["inputs"]]
    x = ThrowRun.apply(*inputs, s["setup"])
    loss = ((x - s["target"]) ** 2).sum(1).mean()
    loss.backward()
    return {"x": x.detach(), "loss": loss.detach(),
            "grad": {k: t.grad for k, t in zip(("v0", "w0", "mass", "mu_s", "mu_d"), inputs)}}


def run(s):
    case = s["case"]
    if case["kind"] == "throw":
        return _run_throw(s)
    if case["kind"] == "dropin":
        return _run_dropin(s)
    gw = s["gw"]
    gw.set_state(s["start"])
    gw.step(case["frames"], **s["step"])
    out = gw.state()
    if case.get("render"):
        out["model"] = gw.model_matrices(as_float=True)
    return out


# --------------------------------------------------------------------------
# Work and exact values
# --------------------------------------------------------------------------
def _bodies(case):
    """Dynamic bodies of a case, all scenes (the mean for uneven scenes)."""
    k = case["kind"]
    if k in ("dropin", "large"):
        return case["bodies"]
    if k == "batch":
        return case["scenes"] * (case["cubes"] + case["icos"])
    if k == "chains":
        return case["scenes"] * case["length"]
    if k == "mixed":
        return case["scenes"] * (case["spheres"] + case["cubes"] + case["dumbbells"])
    if k == "uneven":  # log-uniform on [4, 256], capped
        lo, hi, m = math.log(4.0), math.log(256.0), float(case["most"])
        mean = ((min(m, 256.0) - 4.0) + m * max(0.0, hi - math.log(m))) / (hi - lo)
        return case["scenes"] * mean
    return case["scenes"]


# FP64 operations per dynamic body and substep, counted by running the step
# with an op-counting scalar on resting piles (integration, GJK, EPA,
# manifold, constraint solve), and for free flight (integration and GJK only).
PILE_OPS, FLIGHT_OPS = 3.0e3, 1.0e3
STATE_BYTES = 27 * 8 + 4  # one body's ten state fields


def work(case):
    n = _bodies(case)
    frames = case.get("frames", 1)
    ops = FLIGHT_OPS if case.get("warm") == 0 or case["kind"] == "throw" else PILE_OPS
    flops = n * frames * SUBSTEPS * ops
    if case["kind"] == "throw":  # forward, and the substep's derivative in each of 16 inputs
        return {"bytes": 8.0 * n * (9 + 3 + 9), "flops": 3.0 * flops}
    extra = 64 * n if case.get("render") else 0
    return {"bytes": 2.0 * STATE_BYTES * n + extra, "flops": float(flops)}


def exact(case, seed):
    """Free flight in numpy: no body of a falling case reaches another or the
    floor, so a frame is integration and the velocity update alone (the
    bodies do not spin). None for every other case: its collisions are a
    sequential program of GJK, EPA, clipping and Gauss-Seidel over each
    scene, far over 20 seconds for a case's frames in plain numpy."""
    if case["kind"] != "batch" or case["warm"] or case["render"]:
        return None
    w = _world(case, seed)
    dyn = np.asarray(w.body_fixed) == 0
    x = np.array(w.body_position, dtype=np.float64)
    v = np.array(w.body_linear_velocity, dtype=np.float64)
    q = np.array(w.body_rotation, dtype=np.float64)
    nb, per = len(x), case["cubes"] + case["icos"] + 1
    half = np.asarray(w.body_scale, dtype=np.float64)[:, 0].reshape(-1, per)[:, 1:]
    box = np.arange(1, per) <= case["cubes"]
    # box axes: row k of a body's matrix is its local axis k in the world
    i, j, k, s = (q / np.sqrt((q * q).sum(1, keepdims=True))).T
    axes = np.stack([1 - 2 * (j * j + k * k), 2 * (i * j + s * k), 2 * (i * k - s * j),
                     2 * (i * j - s * k), 1 - 2 * (i * i + k * k), 2 * (j * k + s * i),
                     2 * (i * k + s * j), 2 * (j * k - s * i), 1 - 2 * (i * i + j * j)], 1)
    axes = axes.reshape(-1, per, 3, 3)[:, 1:]

    def reach(d):
        """How far each body (scene, body) extends along the unit directions d (scene, body, n, 3)."""
        along_box = np.abs(np.einsum("sbac,sbnc->sbna", axes, d)).sum(-1)
        return half[:, :, None] * np.where(box[None, :, None], along_box, 1.0)

    down = reach(np.broadcast_to(np.array([0.0, -1.0, 0.0]), axes.shape[:2] + (1, 3)))[:, :, 0]
    px, pq, pv, deact = x.copy(), q.copy(), v.copy(), np.zeros(nb)
    h = DT / SUBSTEPS
    for _ in range(case["frames"]):
        slow = np.sqrt((v * v).sum(1)) < 0.10
        deact = np.where(dyn & slow, deact + DT, 0.0)
        for _ in range(SUBSTEPS):
            px, pq = x.copy(), q.copy()
            v[dyn] += h * np.array([0.0, -GRAVITY, 0.0])
            x[dyn] += h * v[dyn]
            q[dyn] /= np.sqrt((q[dyn] * q[dyn]).sum(1, keepdims=True))
            pv = v.copy()
            v[dyn] = (x[dyn] - px[dyn]) / h
        # apart at the frame's end, along the line between centres and from the floor
        p = x.reshape(-1, per, 3)[:, 1:]
        if (p[:, :, 1] - down).min() <= -1.0:
            return None
        d = p[:, None] - p[:, :, None]
        dist = np.sqrt((d * d).sum(-1))
        r = reach(d / np.where(dist > 0.0, dist, 1.0)[..., None])
        if (dist - r - r.transpose(0, 2, 1) + 100.0 * np.eye(per - 1)).min() <= 0.0:
            return None
    zero = np.zeros((nb, 3))
    return {"position": x, "rotation": q, "linear_velocity": v, "angular_velocity": zero, "previous_position": px,
            "previous_rotation": pq, "previous_linear_velocity": pv, "previous_angular_velocity": zero,
            "active": None, "deactivation_time": deact[:, None]}
