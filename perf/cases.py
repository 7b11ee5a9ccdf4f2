"""Performance cases of box2d_amd: what its users run, through its public entry points.

A world case holds worlds that are already in motion. One pass steps them with ``b2World_Step`` (or
``b2amd_StepWorlds`` for a batch) at the repository's usual 1/60 s and four substeps, then reads
every body's transform and velocity back, as a game that draws, or a controller that observes, every
few steps does. Sleep is off, so that a pass always steps the whole world. A push case is one
evaluation of a differentiable simulation, forward and backward. A geometry case is one call of the
batched narrowphase or distance functions on host arrays.

Results are bit-identical by contract (the tests compare whole runs with the reference's hashes), so
every tolerance is "exact".
"""

import ctypes
import math

import numpy as np
import torch

import box2d_amd
from box2d_amd import WorldId
from box2d_amd.adjoint import push_simulation

SUBSTEPS = 4


def listed():
    return [
        # the smallest call: a handful of bodies (a menu, a toy, one agent's world), read every step
        {"name": "rain_8", "kind": "rain", "bodies": 8, "settle": 360, "steps": 1},
        # the small pyramid of the repository's configurations: one level of a game
        {"name": "pyramid_20", "kind": "pyramid", "rows": 20, "settle": 30, "steps": 4},
        # joints: a hanging net of balls on revolute joints (ropes, cloth, chains, ragdolls)
        {"name": "net_24", "kind": "net", "rows": 24, "settle": 30, "steps": 4},
        # an ordinary busy scene: every shape type, chain ground, landing and piling up
        {"name": "rain_1000", "kind": "rain", "bodies": 1000, "settle": 420, "steps": 4},
        # the benchmark's headline scene: 100 rows, 5050 boxes
        {"name": "pyramid_100", "kind": "pyramid", "rows": 100, "settle": 10, "steps": 4},
        # the largest single world of the configurations: 20,000 mixed shapes falling into a container
        {"name": "rain_20000", "kind": "rain", "bodies": 20000, "settle": 480, "steps": 4},
        # a batch of uneven small worlds, rolled out a few steps at a time (parallel environments)
        {"name": "batch_64", "kind": "batch", "worlds": 64, "lo": 8, "hi": 256, "settle": 8, "steps": 4},
        # the uneven-worlds batch of the configurations (8 to 1024 bodies), a rollout of 20 steps
        {"name": "batch_1024", "kind": "batch", "worlds": 1024, "lo": 8, "hi": 1024, "settle": 8, "steps": 20},
        # one gradient of a short differentiable push with few candidates
        {"name": "push_16", "kind": "push", "worlds": 16, "rows": 10, "steps": 20},
        # the differentiable push of the configurations: 256 candidates, 60 steps
        {"name": "push_256", "kind": "push", "worlds": 256, "rows": 10, "steps": 60},
        # contact manifolds of many shape pairs at once (placement checks, dataset labelling)
        {"name": "manifolds_32768", "kind": "manifolds", "count": 32768},
        # distances between many shape pairs at once (clearance checks of a planner)
        {"name": "distances_4096", "kind": "distances", "count": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rain", "pyramid", "net", "batch", "push", "manifolds", "distances"])
    if kind == "rain":
        n = _log(rng, 8, 20000)
        return {"kind": kind, "bodies": n, "settle": rng.randint(360, 480), "steps": rng.randint(1, 4)}
    if kind == "pyramid":
        return {"kind": kind, "rows": _log(rng, 4, 100), "settle": rng.randint(10, 40), "steps": rng.randint(1, 4)}
    if kind == "net":
        return {"kind": kind, "rows": _log(rng, 4, 60), "settle": rng.randint(10, 40), "steps": rng.randint(1, 4)}
    if kind == "batch":
        return {"kind": kind, "worlds": _log(rng, 16, 1000), "lo": rng.randint(8, 16), "hi": _log(rng, 64, 1024),
                "settle": rng.randint(4, 12), "steps": rng.randint(2, 16)}
    if kind == "push":
        return {"kind": kind, "worlds": _log(rng, 4, 256), "rows": rng.randint(4, 12), "steps": rng.randint(10, 50)}
    return {"kind": kind, "count": _log(rng, 64, 262144)}


# ---------------------------------------------------------------------------------------------
# Worlds

class Vec2(ctypes.Structure):
    _fields_ = [("x", ctypes.c_float), ("y", ctypes.c_float)]


class Rot(ctypes.Structure):
    _fields_ = [("c", ctypes.c_float), ("s", ctypes.c_float)]


class Transform(ctypes.Structure):
    _fields_ = [("p", Vec2), ("q", Rot)]


class ObjectId(ctypes.Structure):
    """b2BodyId, b2ShapeId and b2JointId."""
    _fields_ = [("index1", ctypes.c_int32), ("world0", ctypes.c_uint16), ("generation", ctypes.c_uint16)]


class BodyDef(ctypes.Structure):
    _fields_ = [("type", ctypes.c_int), ("position", Vec2), ("rotation", Rot), ("linearVelocity", Vec2),
                ("angularVelocity", ctypes.c_float), ("linearDamping", ctypes.c_float), ("angularDamping", ctypes.c_float),
                ("gravityScale", ctypes.c_float), ("sleepThreshold", ctypes.c_float), ("safetyFactor", ctypes.c_float),
                ("name", ctypes.c_char_p), ("userData", ctypes.c_void_p), ("motionLocks", ctypes.c_bool * 3),
                ("enableSleep", ctypes.c_bool), ("isAwake", ctypes.c_bool), ("isBullet", ctypes.c_bool),
                ("isEnabled", ctypes.c_bool), ("allowFastRotation", ctypes.c_bool), ("enableContactRecycling", ctypes.c_bool),
                ("internalValue", ctypes.c_int)]


class SurfaceMaterial(ctypes.Structure):
    _fields_ = [("friction", ctypes.c_float), ("restitution", ctypes.c_float), ("rollingResistance", ctypes.c_float),
                ("tangentSpeed", ctypes.c_float), ("userMaterialId", ctypes.c_uint64), ("customColor", ctypes.c_uint32)]


class Filter(ctypes.Structure):
    _fields_ = [("categoryBits", ctypes.c_uint64), ("maskBits", ctypes.c_uint64), ("groupIndex", ctypes.c_int)]


class ShapeDef(ctypes.Structure):
    _fields_ = [("userData", ctypes.c_void_p), ("material", SurfaceMaterial), ("density", ctypes.c_float),
                ("filter", Filter), ("enableCustomFiltering", ctypes.c_bool), ("isSensor", ctypes.c_bool),
                ("enableSensorEvents", ctypes.c_bool), ("enableContactEvents", ctypes.c_bool),
                ("enableHitEvents", ctypes.c_bool), ("enablePreSolveEvents", ctypes.c_bool),
                ("invokeContactCreation", ctypes.c_bool), ("updateBodyMass", ctypes.c_bool), ("internalValue", ctypes.c_int)]


class JointDef(ctypes.Structure):
    _fields_ = [("userData", ctypes.c_void_p), ("bodyIdA", ObjectId), ("bodyIdB", ObjectId), ("localFrameA", Transform),
                ("localFrameB", Transform), ("forceThreshold", ctypes.c_float), ("torqueThreshold", ctypes.c_float),
                ("constraintHertz", ctypes.c_float), ("constraintDampingRatio", ctypes.c_float),
                ("drawScale", ctypes.c_float), ("collideConnected", ctypes.c_bool)]


class RevoluteJointDef(ctypes.Structure):
    _fields_ = [("base", JointDef), ("targetAngle", ctypes.c_float), ("enableSpring", ctypes.c_bool),
                ("hertz", ctypes.c_float), ("dampingRatio", ctypes.c_float), ("enableLimit", ctypes.c_bool),
                ("lowerAngle", ctypes.c_float), ("upperAngle", ctypes.c_float), ("enableMotor", ctypes.c_bool),
                ("maxMotorTorque", ctypes.c_float), ("motorSpeed", ctypes.c_float), ("internalValue", ctypes.c_int)]


class Circle(ctypes.Structure):
    _fields_ = [("center", Vec2), ("radius", ctypes.c_float)]


class Capsule(ctypes.Structure):
    _fields_ = [("center1", Vec2), ("center2", Vec2), ("radius", ctypes.c_float)]


class Polygon(ctypes.Structure):
    _fields_ = [("vertices", Vec2 * 8), ("normals", Vec2 * 8), ("centroid", Vec2), ("radius", ctypes.c_float),
                ("count", ctypes.c_int)]


class Hull(ctypes.Structure):
    _fields_ = [("points", Vec2 * 8), ("count", ctypes.c_int)]


class BodyEvents(ctypes.Structure):
    _fields_ = [("moveEvents", ctypes.c_void_p), ("moveCount", ctypes.c_int)]


def _library():
    lib = box2d_amd.library()
    for name, result, arguments in (
            ("b2DefaultBodyDef", BodyDef, []), ("b2DefaultShapeDef", ShapeDef, []),
            ("b2DefaultRevoluteJointDef", RevoluteJointDef, []),
            ("b2CreateBody", ObjectId, [WorldId, ctypes.POINTER(BodyDef)]),
            ("b2CreateCircleShape", ObjectId, [ObjectId, ctypes.POINTER(ShapeDef), ctypes.POINTER(Circle)]),
            ("b2CreateRevoluteJoint", ObjectId, [WorldId, ctypes.POINTER(RevoluteJointDef)]),
            ("b2World_SetGravity", None, [WorldId, Vec2]), ("b2World_EnableSleeping", None, [WorldId, ctypes.c_bool]),
            ("b2World_Step", None, [WorldId, ctypes.c_float, ctypes.c_int]),
            ("b2World_GetBodyEvents", BodyEvents, [WorldId]),
            ("b2MakeRoundedBox", Polygon, [ctypes.c_float] * 3), ("b2MakeBox", Polygon, [ctypes.c_float] * 2),
            ("b2ComputeHull", Hull, [ctypes.POINTER(Vec2), ctypes.c_int]),
            ("b2MakePolygon", Polygon, [ctypes.POINTER(Hull), ctypes.c_float])):
        f = getattr(lib, name)
        f.restype, f.argtypes = result, arguments
    return lib


class Worlds:
    """The worlds of a case, destroyed with it."""

    def __init__(self):
        self.lib, self.scenes, self.handles = _library(), box2d_amd.scenes(), []

    def add(self, kind, iparams=(), fparams=()):
        self.handles.append(self.scenes.create(kind, iparams, fparams))
        return self.scenes.world_id(self.handles[-1])

    def __del__(self):
        for h in self.handles:
            self.scenes.destroy(h)


MOVE_EVENT = np.dtype([("userData", "<u8"), ("transform", "<f4", 4), ("bodyId", "<i4"), ("world0", "<u2"),
                       ("generation", "<u2"), ("fellAsleep", "u1"), ("padding", "u1", 7)])


def _move_events(w):
    """The transform of every body that the last step moved, from b2World_GetBodyEvents."""
    e = w.lib.b2World_GetBodyEvents(w.world)
    raw = ctypes.string_at(e.moveEvents, e.moveCount * MOVE_EVENT.itemsize)
    events = np.frombuffer(raw, dtype=MOVE_EVENT)
    return {"transforms": events["transform"], "bodies": events["bodyId"]}


def _net(lib, world, rows, rng):
    """rows x rows balls, each tied to its left and upper neighbour by a revolute joint; the top row is
    fixed in every fourth place. The balls start with small random velocities."""
    body, shape, joint = lib.b2DefaultBodyDef(), lib.b2DefaultShapeDef(), lib.b2DefaultRevoluteJointDef()
    shape.filter.categoryBits, shape.filter.maskBits = 2, 1  # they do not collide with each other
    circle = Circle(Vec2(0.0, 0.0), 0.4)
    above = []
    for i in range(rows):
        row = []
        for k in range(rows):
            body.type = 0 if i == 0 and k % 4 == 0 else 2
            body.position = Vec2(k, 20.0 + rows - i)
            body.linearVelocity = Vec2(rng.uniform(-1, 1), rng.uniform(-1, 1)) if body.type == 2 else Vec2(0, 0)
            b = lib.b2CreateBody(world, ctypes.byref(body))
            lib.b2CreateCircleShape(b, ctypes.byref(shape), ctypes.byref(circle))
            ties = [(row[-1], Vec2(0.5, 0.0), Vec2(-0.5, 0.0))] if k else []
            ties += [(above[k], Vec2(0.0, -0.5), Vec2(0.0, 0.5))] if i else []
            for other, at, of in ties:
                joint.base.bodyIdA, joint.base.bodyIdB = other, b
                joint.base.localFrameA.p, joint.base.localFrameB.p = at, of
                lib.b2CreateRevoluteJoint(world, ctypes.byref(joint))
            row.append(b)
        above = row


def _rain_columns(bodies):
    """The configurations' proportions: 200 columns of 0.6 m for 20,000 bodies."""
    return max(4, int(round(math.sqrt(2.0 * bodies))))


def _prepare_world(case, seed):
    rng = np.random.default_rng(seed)
    w = Worlds()
    if case["kind"] == "rain":
        columns = _rain_columns(case["bodies"])
        world = w.add(box2d_amd.SCENE_RAIN, (case["bodies"], columns, 0, 1 + seed % (1 << 30)), (0.6 * columns,))
    elif case["kind"] == "pyramid":
        # the ground is tilted a little, by the seed (friction 0.6 holds the boxes)
        world = w.add(box2d_amd.SCENE_PYRAMID, (case["rows"], 0), (100.0,))
        w.lib.b2World_SetGravity(world, Vec2(rng.uniform(-0.2, 0.2), -10.0))
    else:
        # the net hangs over the ground and the box of the scene driver's one-box world
        world = w.add(box2d_amd.SCENE_HELLO)
        w.lib.b2World_EnableSleeping(world, False)
        _net(w.lib, world, case["rows"], rng)
    w.world = world
    w.ids = (WorldId * 1)(world)
    for _ in range(case["settle"]):
        w.lib.b2World_Step(world, 1.0 / 60.0, SUBSTEPS)
    return w


def _run_world(case, w):
    for _ in range(case["steps"]):
        w.lib.b2World_Step(w.world, 1.0 / 60.0, SUBSTEPS)
    if case["kind"] == "net":
        return _move_events(w)
    h = w.handles[0]
    return {"transforms": w.scenes.transforms(h), "velocities": w.scenes.velocities(h)}


def _prepare_batch(case, seed):
    w = Worlds()
    specs = box2d_amd.batch_world_specs(case["worlds"], case["lo"], case["hi"], seed=seed)
    # the sizes and kinds (and the chains' numbers) of every seed are alike, the piles are not
    sizes = box2d_amd.batch_world_specs(case["worlds"], case["lo"], case["hi"])
    ids = [w.add(box2d_amd.SCENE_BATCH_WORLD, (size, kind, fixed if kind == 2 else own))
           for (size, kind, fixed), (_, _, own) in zip(sizes, specs)]
    tilt = np.random.default_rng(seed)
    for i in ids:
        w.lib.b2World_SetGravity(i, Vec2(tilt.uniform(-0.2, 0.2), -10.0))
    w.ids = (WorldId * len(ids))(*ids)
    box2d_amd.step_worlds(w.ids, case["settle"], 1.0 / 60.0, SUBSTEPS)
    return w


def _run_batch(case, w):
    box2d_amd.step_worlds(w.ids, case["steps"], 1.0 / 60.0, SUBSTEPS)
    return {"transforms": np.concatenate([w.scenes.transforms(h) for h in w.handles]),
            "velocities": np.concatenate([w.scenes.velocities(h) for h in w.handles])}


# ---------------------------------------------------------------------------------------------
# Differentiable push: the configurations' parameter ranges

def _prepare_push(case, seed):
    rng = np.random.default_rng(seed)
    n = case["worlds"]
    params = np.stack([rng.uniform(2, 6, n), rng.uniform(-0.5, 0.5, n), rng.uniform(-1, 1, n), rng.uniform(0.3, 0.9, n)], 1)
    top = case["rows"] * (case["rows"] + 1) // 2 - 1  # the pyramid's last box
    goals = rng.uniform(-2, 2, (n, 2)) + np.array([0.0, case["rows"] - 0.5])
    return {"params": torch.tensor(params, dtype=torch.float32, requires_grad=True), "top": top,
            "goals": torch.tensor(goals, dtype=torch.float32)}


def _run_push(case, s):
    centers = push_simulation(s["params"], case["steps"], case["rows"])
    loss = (centers[:, s["top"]] - s["goals"]).square().sum(1)
    (gradient,) = torch.autograd.grad(loss.sum(), s["params"])
    return {"centers": centers.detach(), "loss": loss.detach(), "gradient": gradient}


# ---------------------------------------------------------------------------------------------
# Geometry on host arrays

SHAPE_BYTES, MANIFOLD_BYTES = 152, 44  # b2amd_Shape, b2LocalManifold
PAIRS = [(0, 0), (1, 0), (1, 1), (3, 0), (3, 1), (3, 3), (2, 0), (2, 1), (2, 3)]  # the pair types, in primary order
DISTANCE_INPUT = np.dtype([("pointsA", "<f4", (8, 2)), ("countA", "<i4"), ("radiusA", "<f4"), ("pointsB", "<f4", (8, 2)),
                           ("countB", "<i4"), ("radiusB", "<f4"), ("p", "<f4", 2), ("q", "<f4", 2), ("useRadii", "u1"),
                           ("padding", "u1", 3)])
DISTANCE_OUTPUT = np.dtype([("pointA", "<f4", 2), ("pointB", "<f4", 2), ("normal", "<f4", 2), ("distance", "<f4"),
                            ("iterations", "<i4"), ("simplexCount", "<i4")])


def _shapes(lib, rng, kind, count):
    """`count` shapes of one type as b2amd_Shape records: a set of assets, as a program has."""
    out = np.zeros((count, SHAPE_BYTES), dtype=np.uint8)
    for i in range(count):
        if kind == 0:
            g = Circle(Vec2(*rng.uniform(-0.3, 0.3, 2)), rng.uniform(0.05, 0.6))
        elif kind == 1:
            a, h, c = rng.uniform(-np.pi, np.pi), rng.uniform(0.05, 0.7), rng.uniform(-0.2, 0.2, 2)
            d = h * np.array([np.cos(a), np.sin(a)])
            g = Capsule(Vec2(*(c - d)), Vec2(*(c + d)), rng.uniform(0.02, 0.3))
        elif kind == 2:
            p = rng.uniform(-1.0, 1.0, 2)
            g = (Vec2 * 2)(Vec2(*p), Vec2(*(p + rng.uniform(0.3, 1.5, 2))))
        elif i % 2 == 0:
            g = lib.b2MakeBox(rng.uniform(0.1, 0.8), rng.uniform(0.1, 0.8)) if i % 4 else \
                lib.b2MakeRoundedBox(rng.uniform(0.1, 0.6), rng.uniform(0.1, 0.6), rng.uniform(0.01, 0.2))
        else:
            hull = Hull()
            while hull.count < 3:
                n = int(rng.integers(3, 9))
                a, r = rng.uniform(-np.pi, np.pi, n), rng.uniform(0.2, 0.9, n)
                hull = lib.b2ComputeHull((Vec2 * 8)(*[Vec2(x, y) for x, y in zip(r * np.cos(a), r * np.sin(a))]), n)
            g = lib.b2MakePolygon(ctypes.byref(hull), rng.uniform(0.01, 0.15) if i % 4 == 1 else 0.0)
        raw = np.frombuffer(bytes(ctypes.c_int(kind)) + bytes(4) + bytes(g), dtype=np.uint8)
        out[i, :raw.size] = raw
    return out


def _poses(rng, n, reach):
    """Poses of B in A's frame: mostly touching or near."""
    angle = np.where(rng.uniform(size=n) < 0.8, rng.uniform(-np.pi, np.pi, n), np.pi / 2 * rng.integers(0, 4, n))
    return np.concatenate([rng.uniform(-reach, reach, (n, 2)), np.stack([np.cos(angle), np.sin(angle)], 1)], 1).astype(np.float32)


def _prepare_manifolds(case, seed):
    rng, n, lib = np.random.default_rng(seed), case["count"], _library()
    assets = {k: _shapes(lib, rng, k, 64) for k in (0, 1, 2, 3)}
    pair = rng.integers(0, len(PAIRS), n)
    a, b = np.zeros((n, SHAPE_BYTES), np.uint8), np.zeros((n, SHAPE_BYTES), np.uint8)
    for k, (ka, kb) in enumerate(PAIRS):
        at = np.flatnonzero(pair == k)
        a[at], b[at] = assets[ka][rng.integers(0, 64, at.size)], assets[kb][rng.integers(0, 64, at.size)]
    return {"a": a, "b": b, "poses": _poses(rng, n, 1.0), "lib": lib}


def _run_manifolds(case, s):
    out = np.zeros((case["count"], MANIFOLD_BYTES // 4), dtype=np.float32)
    rc = s["lib"].b2amd_CollideBatch(s["a"].ctypes.data_as(ctypes.c_void_p), s["b"].ctypes.data_as(ctypes.c_void_p),
                                     s["poses"].ctypes.data_as(ctypes.c_void_p), case["count"],
                                     out.ctypes.data_as(ctypes.c_void_p))
    if rc != 0:
        raise RuntimeError("b2amd_CollideBatch failed")
    # normal, then per point its position, separation and (in 16 bits) feature id, then the count
    words = out.view(np.uint32)
    return {"normal": out[:, 0:2], "points": out[:, [2, 3, 4, 6, 7, 8]],
            "ids": (words[:, [5, 9]] & 0xFFFF).astype(np.int32), "count": words[:, 10].astype(np.int32)}


def _prepare_distances(case, seed):
    rng, n = np.random.default_rng(seed), case["count"]
    d = np.zeros(n, dtype=DISTANCE_INPUT)
    for side in "AB":
        count = np.choose(rng.integers(0, 3, n), [np.full(n, 1), np.full(n, 2), rng.integers(3, 9, n)]).astype(np.int32)
        k = np.arange(8)[None, :]
        # convex by construction: points on a circle, in order, at random spacings
        angle = rng.uniform(0, 2 * np.pi, (n, 1)) + 2 * np.pi * (k + rng.uniform(-0.3, 0.3, (n, 8))) / count[:, None]
        points = rng.uniform(0.3, 0.9, (n, 1))[:, :, None] * np.stack([np.cos(angle), np.sin(angle)], 2)
        d["points" + side] = np.where((k < count[:, None])[:, :, None], points, 0.0)
        d["count" + side] = count
        d["radius" + side] = np.where(count > 2, rng.uniform(0.0, 0.1, n) * rng.integers(0, 2, n), rng.uniform(0.05, 0.3, n))
    poses = _poses(rng, n, 3.0)
    d["p"], d["q"], d["useRadii"] = poses[:, :2], poses[:, 2:], rng.integers(0, 2, n)
    return {"inputs": d, "lib": _library()}


def _run_distances(case, s):
    n = case["count"]
    caches = np.zeros((n, 8), dtype=np.uint8)
    out = np.zeros(n, dtype=DISTANCE_OUTPUT)
    s["lib"].b2amd_ShapeDistanceBatch(s["inputs"].ctypes.data_as(ctypes.c_void_p), caches.ctypes.data_as(ctypes.c_void_p),
                                      n, out.ctypes.data_as(ctypes.c_void_p))
    return {"distance": out["distance"], "pointA": out["pointA"], "pointB": out["pointB"], "normal": out["normal"],
            "iterations": out["iterations"], "caches": caches}


# ---------------------------------------------------------------------------------------------

PREPARE = {"batch": _prepare_batch, "push": _prepare_push, "manifolds": _prepare_manifolds, "distances": _prepare_distances}
RUN = {"batch": _run_batch, "push": _run_push, "manifolds": _run_manifolds, "distances": _run_distances}


def prepare(case, seed):
    return case, PREPARE.get(case["kind"], _prepare_world)(case, seed)


def run(state):
    case, s = state
    return RUN.get(case["kind"], _run_world)(case, s)


def _sizes(case):
    """(bodies, contacts, joints) of a world case, the contacts as the settled scenes hold them."""
    if case["kind"] == "rain":
        return case["bodies"], 2.0 * case["bodies"], 0
    if case["kind"] == "net":
        return case["rows"] ** 2, 0, 2 * case["rows"] * (case["rows"] - 1)
    n = case["rows"] * (case["rows"] + 1) // 2
    return n, 3.0 * n, 0


def work(case):
    """Bytes: over the pass each body's simulation record, state and flags (96 + 32 + 32 bytes) and each
    contact (184) or joint (468) read and written once and its shapes (248) read, however many steps
    it makes; for a push also the step records (88 bytes a body, 160 a contact) that the backward pass
    needs; the geometry calls' arrays. Flops: per substep some 600 for a contact (warm start, solve,
    relax) or a joint and 40 for a body, per step some 500 for a contact's manifold; the backward pass
    is three times that."""
    kind = case["kind"]
    if kind == "manifolds":
        return {"bytes": case["count"] * (2 * SHAPE_BYTES + 16 + MANIFOLD_BYTES), "flops": 500 * case["count"]}
    if kind == "distances":
        return {"bytes": case["count"] * (DISTANCE_INPUT.itemsize + 16 + DISTANCE_OUTPUT.itemsize), "flops": 500 * case["count"]}
    if kind == "batch":
        sizes = box2d_amd.batch_world_specs(case["worlds"], case["lo"], case["hi"])
        bodies = sum(min(s, 160) if k == 2 else s for s, k, _ in sizes)
        contacts = sum((3.0, 1.5, 0.0)[k] * s for s, k, _ in sizes)
        joints = sum(min(s, 160) for s, k, _ in sizes if k == 2)
    elif kind == "push":
        bodies = case["worlds"] * (case["rows"] * (case["rows"] + 1) // 2 + 1)
        contacts, joints = 3.0 * bodies, 0
    else:
        bodies, contacts, joints = _sizes(case)
    state_bytes = bodies * (320 + 248) + contacts * 368 + joints * 936
    record_bytes = 2 * case["steps"] * (88 * bodies + 160 * contacts) if kind == "push" else 0
    step_flops = SUBSTEPS * (600 * (contacts + joints) + 40 * bodies) + 500 * contacts
    passes = 4 if kind == "push" else 1
    return {"bytes": state_bytes + record_bytes, "flops": step_flops * case["steps"] * passes}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """Distances between convex shapes in 64 bits, over all pairs of their vertices and edges. The other
    outputs have no such value: which of two equal features a manifold or a simplex names is the
    algorithm's choice, and a stepped world follows its own rounding."""
    if case["kind"] != "distances":
        return None
    d = _prepare_distances(case, seed)["inputs"]
    n = d.size
    a = d["pointsA"].astype(np.float64)
    b0 = d["pointsB"].astype(np.float64)
    c, s = d["q"][:, 0].astype(np.float64)[:, None], d["q"][:, 1].astype(np.float64)[:, None]
    b = np.stack([c * b0[..., 0] - s * b0[..., 1], s * b0[..., 0] + c * b0[..., 1]], 2) + d["p"].astype(np.float64)[:, None, :]
    best = np.full(n, np.inf)
    inside = np.zeros(n, dtype=bool)
    for p, np_, q, nq in ((a, d["countA"], b, d["countB"]), (b, d["countB"], a, d["countA"])):
        within = np.ones((n, 8), dtype=bool)  # vertices of q on the inner side of every edge of p
        for i in range(8):
            j = np.where(i + 1 < np_, i + 1, 0)
            v1, v2 = p[:, i], p[np.arange(n), j]
            e = v2 - v1
            w = q - v1[:, None, :]
            t = np.clip((w * e[:, None, :]).sum(2) / np.maximum((e * e).sum(1), 1e-300)[:, None], 0.0, 1.0)
            r = np.linalg.norm(w - t[..., None] * e[:, None, :], axis=2)
            live = (i < np_)[:, None] & (np.arange(8)[None, :] < nq[:, None])
            best = np.minimum(best, np.where(live, r, np.inf).min(1))
            within &= ((e[:, None, 0] * w[..., 1] - e[:, None, 1] * w[..., 0]) >= 0.0) | (i >= np_)[:, None]
        inside |= (np_ > 2) & (within & (np.arange(8)[None, :] < nq[:, None])).any(1)
    # edges that cross with no vertex inside: the segments properly intersect
    for i in range(8):
        for k in range(8):
            p1, p2 = a[:, i], a[np.arange(n), np.where(i + 1 < d["countA"], i + 1, 0)]
            q1, q2 = b[:, k], b[np.arange(n), np.where(k + 1 < d["countB"], k + 1, 0)]

            def side(o, u, v):
                return (u - o)[:, 0] * (v - o)[:, 1] - (u - o)[:, 1] * (v - o)[:, 0]

            live = (i < d["countA"]) & (k < d["countB"]) & (d["countA"] > 1) & (d["countB"] > 1)
            inside |= live & (side(p1, p2, q1) * side(p1, p2, q2) < 0) & (side(q1, q2, p1) * side(q1, q2, p2) < 0)
    best[inside] = 0.0
    radii = (d["radiusA"].astype(np.float64) + d["radiusB"]) * (d["useRadii"] != 0)
    return {"distance": np.maximum(0.0, best - radii), "pointA": None, "pointB": None, "normal": None, "iterations": None,
            "caches": None}
