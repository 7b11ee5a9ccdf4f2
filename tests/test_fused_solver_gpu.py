"""The single-workgroup solver's forms (rows resident in registers, rows streamed, general) and the XCD
solver's (four or two rows resident and the rest streamed, joints of every type) against the color kernels,
bit for bit after every step, at the sizes where a form's chunks change: one chunk per color, partial
chunks, the last resident world and the first streamed one, several chunks of one color in a wavefront,
bodies without constraints, more bodies than registers. Each case states the form it is there for, and what
the library reports of every step must agree. Then what Auto takes on either side of its lines."""

import ctypes

import numpy as np
import pytest

import box2d_amd
from box2d_amd import WorldId
from b2types import c_float
from box2d_amd.scenes_api import SCENE_JOINT_ZOO
from nets import add_net

pytestmark = pytest.mark.gpu


class Id(ctypes.Structure):
    _fields_ = [("index1", ctypes.c_int32), ("world0", ctypes.c_uint16), ("generation", ctypes.c_uint16)]


class Material(ctypes.Structure):
    _fields_ = [("friction", c_float), ("restitution", c_float), ("rollingResistance", c_float), ("tangentSpeed", c_float),
                ("userMaterialId", ctypes.c_uint64), ("customColor", ctypes.c_uint32)]


class BodyEvents(ctypes.Structure):
    _fields_ = [("moveEvents", ctypes.c_void_p), ("moveCount", ctypes.c_int)]


def _set_materials(lib, world, restitution):
    """Every third moving body's shape gets rolling resistance and tangent speed (and restitution)."""
    lib.b2World_GetBodyEvents.restype, lib.b2World_GetBodyEvents.argtypes = BodyEvents, [WorldId]
    lib.b2Body_GetShapes.argtypes = [Id, ctypes.POINTER(Id), ctypes.c_int]
    lib.b2Shape_SetSurfaceMaterial.argtypes = [Id, ctypes.POINTER(Material)]
    events = lib.b2World_GetBodyEvents(world)
    raw = np.frombuffer(ctypes.string_at(events.moveEvents, 40 * events.moveCount), dtype=np.uint8).reshape(-1, 40)
    for body in sorted(raw[:, 24:32].tolist())[::3]:
        shapes = (Id * 4)()
        for k in range(lib.b2Body_GetShapes(Id.from_buffer_copy(bytes(body)), shapes, 4)):
            m = Material(0.5, 0.4 if restitution else 0.0, 0.15, 0.3, 0, 0)
            lib.b2Shape_SetSurfaceMaterial(shapes[k], ctypes.byref(m))


def _run(scenes, make, path, steps, materials):
    lib = box2d_amd.library()
    h = make()
    try:
        world = scenes.world_id(h)
        box2d_amd.set_solver_path(world, path)
        scenes.step(h, 1)
        if materials is not None:
            _set_materials(lib, world, materials == "bouncy")
        out, used = [], []
        for _ in range(steps):
            scenes.step(h, 1)
            out.append((scenes.transforms(h).tobytes(), scenes.velocities(h).tobytes()))
            info = box2d_amd.last_solver(world)
            used.append((info.path, info.form, info.threads, info.chunks))
        counters = scenes.counters(h)
        return out, used, counters["awake_contacts"] + counters["joints"]
    finally:
        scenes.destroy(h)


GENERAL, STREAMED, RESIDENT = 0, 1, 2

# (kind, size, materials, steps), the form that the last step takes
CASES = [("pyramid", rows, None, 40, RESIDENT) for rows in (1, 2, 7, 11, 16, 21, 22, 23, 24, 25)]
CASES += [("pyramid", rows, None, 40, STREAMED) for rows in (26, 40)]
CASES += [("pile", n, m, 150, RESIDENT) for n in (1, 3, 33, 130) for m in (None, "rolling")]
CASES += [("pile", n, "bouncy", 150, GENERAL) for n in (1, 3, 33, 130)]
CASES += [("pile", 600, "rolling", 200, STREAMED)]
CASES += [("chains", n, None, 40, GENERAL) for n in (8, 160)]
CASES += [("net", rows, None, 20, GENERAL) for rows in (2, 12, 40)]
CASES += [("zoo", 0, None, 60, GENERAL), ("hinges", 0, None, 100, GENERAL)]


def _make(scenes, kind, size):
    if kind == "pyramid":
        return scenes.pyramid(size, 100.0)
    if kind == "pile":
        return scenes.create(box2d_amd.SCENE_MIXED_PILE, (size, 0, 77))
    if kind == "zoo":
        return scenes.create(SCENE_JOINT_ZOO, (0,))
    if kind == "hinges":
        return scenes.create(box2d_amd.SCENE_FALLING_HINGES)
    if kind == "rain":
        # spaced so that only a few neighbours touch: most bodies have no constraint; more bodies than the
        # wavefronts keep in registers (16,384 with four rows, 32,768 with two)
        return scenes.create(box2d_amd.SCENE_RAIN, (size, 170, 0, 9), (136.0,))
    if kind == "net":
        h = scenes.create(box2d_amd.SCENE_HELLO)
        add_net(scenes.world_id(h), size, spring=size == 12)
        return h
    return scenes.create(box2d_amd.SCENE_BATCH_WORLD, (size, 2, 5))


@pytest.mark.parametrize("kind,size,materials,steps,form", CASES)
def test_fused_matches_color_kernels(gpu_scenes, kind, size, materials, steps, form):
    fused, used, constraints = _run(gpu_scenes, lambda: _make(gpu_scenes, kind, size), box2d_amd.SOLVER_FUSED, steps, materials)
    colored, reference, _ = _run(gpu_scenes, lambda: _make(gpu_scenes, kind, size), box2d_amd.SOLVER_COLOR_KERNELS, steps, materials)
    assert constraints > 0
    assert {u[0] for u in used} == {box2d_amd.SOLVER_FUSED} and {u[0] for u in reference} == {box2d_amd.SOLVER_COLOR_KERNELS}
    assert used[-1][1] == form, used[-1]
    for k, (a, b) in enumerate(zip(fused, colored)):
        assert a == b, f"step {k + 2}"


# ..., rows that a wavefront keeps in registers: 4 up to 512 chunks, else 2
XCD_CASES = [("pyramid", rows, None, 20, 4) for rows in (1, 2, 7, 25, 60)] + [("pyramid", 112, None, 6, 2)]
XCD_CASES += [("pile", n, m, 120, 4) for n in (1, 65, 600) for m in ("rolling", "bouncy")]
XCD_CASES += [("chains", 160, None, 40, 4), ("rain", 17000, None, 3, 4), ("rain", 34000, None, 2, 2), ("zoo", 0, None, 60, 4), ("hinges", 0, None, 100, 4)]
XCD_CASES += [("net", rows, None, 10, 4) for rows in (2, 12, 70)] + [("net", 140, None, 4, 2)]


@pytest.mark.parametrize("kind,size,materials,steps,rows", XCD_CASES)
def test_xcd_matches_color_kernels(gpu_scenes, kind, size, materials, steps, rows):
    xcd, used, constraints = _run(gpu_scenes, lambda: _make(gpu_scenes, kind, size), box2d_amd.SOLVER_XCD, steps, materials)
    colored, reference, _ = _run(gpu_scenes, lambda: _make(gpu_scenes, kind, size), box2d_amd.SOLVER_COLOR_KERNELS, steps, materials)
    assert constraints > 0
    assert {u[0] for u in used} == {box2d_amd.SOLVER_XCD} and {u[0] for u in reference} == {box2d_amd.SOLVER_COLOR_KERNELS}
    assert used[-1][1] == rows, used[-1]
    for k, (a, b) in enumerate(zip(xcd, colored)):
        assert a == b, f"step {k + 2}"


@pytest.mark.parametrize("size", [100, 257, 1000, 5000])
def test_bodies_in_the_air_have_lanes(gpu_scenes, size):
    """Free fall: next to no constraints, but a lane for every two bodies up to the workgroup's limit."""
    columns = 2 * int(size ** 0.5) + 4
    h = gpu_scenes.create(box2d_amd.SCENE_RAIN, (size, columns, 0, 5), (1.5 * columns,))
    try:
        gpu_scenes.step(h, 5)
        info = box2d_amd.last_solver(gpu_scenes.world_id(h))
        assert info.path == box2d_amd.SOLVER_FUSED and info.chunks <= 2
        assert 2 * info.threads >= min(size, 2048), info.threads
    finally:
        gpu_scenes.destroy(h)


# (kind, size, joint net's rows), what Auto takes: worlds without joints fill the resident form's 32 chunks
# first, those with joints go to the XCD solver above 16; beyond 9,000 contacts a color, 3,600 joints a
# color or 49,152 bodies the color kernels
AUTO = [("pyramid", 24, 0, box2d_amd.SOLVER_FUSED), ("pyramid", 26, 0, box2d_amd.SOLVER_XCD),
        ("pyramid", 1, 18, box2d_amd.SOLVER_FUSED), ("pyramid", 1, 26, box2d_amd.SOLVER_XCD),
        ("pyramid", 14, 2, box2d_amd.SOLVER_XCD), ("pyramid", 8, 2, box2d_amd.SOLVER_FUSED),
        ("pyramid", 225, 0, box2d_amd.SOLVER_XCD), ("pyramid", 250, 0, box2d_amd.SOLVER_COLOR_KERNELS),
        ("pyramid", 1, 90, box2d_amd.SOLVER_XCD), ("pyramid", 1, 125, box2d_amd.SOLVER_COLOR_KERNELS)]


@pytest.mark.parametrize("kind,size,net,path", AUTO)
def test_auto_takes(gpu_scenes, kind, size, net, path):
    h = gpu_scenes.pyramid(size, 1000.0)
    try:
        world = gpu_scenes.world_id(h)
        if net:
            add_net(world, net)
        gpu_scenes.step(h, 20 if max(size, net) < 90 else 4)
        info = box2d_amd.last_solver(world)
        assert info.path == path, (info.path, info.chunks)
        assert (info.chunks > (16 if net else 32)) == (path != box2d_amd.SOLVER_FUSED)
    finally:
        gpu_scenes.destroy(h)
