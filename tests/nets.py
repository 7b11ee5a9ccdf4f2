"""Bodies made through the public API: hanging nets of balls on revolute joints (worlds with many joints),
rows of static circles."""

import ctypes

import box2d_amd
from box2d_amd import WorldId


class Vec2(ctypes.Structure):
    _fields_ = [("x", ctypes.c_float), ("y", ctypes.c_float)]


class Id(ctypes.Structure):
    _fields_ = [("index1", ctypes.c_int32), ("world0", ctypes.c_uint16), ("generation", ctypes.c_uint16)]


class BodyDef(ctypes.Structure):
    _fields_ = [("type", ctypes.c_int), ("position", Vec2), ("rotation", ctypes.c_float * 2), ("linearVelocity", Vec2),
                ("rest", ctypes.c_float * 6), ("name", ctypes.c_void_p), ("userData", ctypes.c_void_p),
                ("flags", ctypes.c_bool * 9), ("internalValue", ctypes.c_int)]


class ShapeDef(ctypes.Structure):
    _fields_ = [("userData", ctypes.c_void_p), ("material", ctypes.c_uint64 * 4), ("density", ctypes.c_float),
                ("categoryBits", ctypes.c_uint64), ("maskBits", ctypes.c_uint64), ("groupIndex", ctypes.c_int64),
                ("flags", ctypes.c_bool * 7), ("internalValue", ctypes.c_int)]


class Circle(ctypes.Structure):
    _fields_ = [("center", Vec2), ("radius", ctypes.c_float)]


class JointDef(ctypes.Structure):
    _fields_ = [("userData", ctypes.c_void_p), ("bodyIdA", Id), ("bodyIdB", Id), ("frameA", ctypes.c_float * 4),
                ("frameB", ctypes.c_float * 4), ("rest", ctypes.c_float * 5), ("collideConnected", ctypes.c_bool),
                ("targetAngle", ctypes.c_float), ("enableSpring", ctypes.c_bool), ("hertz", ctypes.c_float),
                ("dampingRatio", ctypes.c_float), ("enableLimit", ctypes.c_bool), ("angles", ctypes.c_float * 2),
                ("enableMotor", ctypes.c_bool), ("motor", ctypes.c_float * 2), ("internalValue", ctypes.c_int)]


def _function(name, result, *arguments):
    f = getattr(box2d_amd.library(), name)
    f.restype, f.argtypes = result, arguments
    return f


def add_body(world, kind, x, y, vx=0.0):
    """A body without shapes; kind 0 static, 1 kinematic, 2 dynamic."""
    body = _function("b2DefaultBodyDef", BodyDef)()
    body.type, body.position, body.linearVelocity = kind, Vec2(x, y), Vec2(vx, 0.0)
    return _function("b2CreateBody", Id, WorldId, ctypes.POINTER(BodyDef))(world, ctypes.byref(body))


def add_circles(world, count, x):
    """Static circles of radius 0.1 in a row from x on, 50 m up."""
    shape = _function("b2DefaultShapeDef", ShapeDef)()
    make_shape = _function("b2CreateCircleShape", Id, Id, ctypes.POINTER(ShapeDef), ctypes.POINTER(Circle))
    for i in range(count):
        make_shape(add_body(world, 0, x + 0.5 * i, 50.0), ctypes.byref(shape), ctypes.byref(Circle(Vec2(0.0, 0.0), 0.1)))


def add_net(world, rows, spring=False):
    """rows x rows balls that collide with nothing, each tied to its left and upper neighbour, the top row
    fixed in every fourth place: 2 rows (rows - 1) joints."""
    shape = _function("b2DefaultShapeDef", ShapeDef)()
    shape.categoryBits, shape.maskBits = 2, 0
    joint = _function("b2DefaultRevoluteJointDef", JointDef)()
    joint.enableSpring, joint.hertz = spring, 2.0
    circle = Circle(Vec2(0.0, 0.0), 0.4)
    make_shape = _function("b2CreateCircleShape", Id, Id, ctypes.POINTER(ShapeDef), ctypes.POINTER(Circle))
    make_joint = _function("b2CreateRevoluteJoint", Id, WorldId, ctypes.POINTER(JointDef))
    above = []
    for i in range(rows):
        row = []
        for k in range(rows):
            fixed = i == 0 and k % 4 == 0
            b = add_body(world, 0 if fixed else 2, float(k), 20.0 + rows - i, 0.0 if fixed else 0.3 * ((7 * i + 3 * k) % 5 - 2))
            make_shape(b, ctypes.byref(shape), ctypes.byref(circle))
            ties = [(row[-1], (0.5, 0.0, 1.0, 0.0), (-0.5, 0.0, 1.0, 0.0))] if k else []
            ties += [(above[k], (0.0, -0.5, 1.0, 0.0), (0.0, 0.5, 1.0, 0.0))] if i else []
            for other, at, of in ties:
                joint.bodyIdA, joint.bodyIdB = other, b
                joint.frameA[:], joint.frameB[:] = at, of
                make_joint(world, ctypes.byref(joint))
            row.append(b)
        above = row
