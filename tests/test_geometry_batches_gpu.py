"""Batched manifolds, times of impact and distances at the counts where their split changes: part of a
wavefront, whole ones, one chunk, two, all slots, slots used again, whole arrays in device memory. Every
record gives what the reference's fixtures hold for it, bit for bit, whatever its place; a refused batch
writes nothing; inputs that earlier work on the device is still about to write are read after it."""

import ctypes

import numpy as np
import pytest

import box2d_amd
from b2types import DistanceInput, DistanceOutput, LocalManifold, Shape, SimplexCache, TOIInput, TOIOutput, Transform
from b2types import manifold_array_words
from earlier_work import EarlierWork
from test_manifolds import load_fixture
from test_toi_fixture import check_toi, distance_words, load

pytestmark = pytest.mark.gpu

# the last ones on either side of where the arrays go through device memory
COUNTS = [1, 63, 64, 65, 2879, 2881, 9000, 24001, 40000]
MANIFOLD_COUNTS = COUNTS + [92182, 92183]
TOI_COUNTS = COUNTS + [49932, 49933]
DISTANCE_COUNTS = COUNTS + [100824, 100825, 150001]


def _take(ctype, records, index):
    raw = np.frombuffer(bytes(records), dtype=np.uint8).reshape(-1, ctypes.sizeof(ctype))
    return (ctype * len(index)).from_buffer_copy(raw[index].tobytes())


@pytest.mark.parametrize("count", MANIFOLD_COUNTS)
def test_manifolds(count):
    a, b, x, want = load_fixture()
    index = np.random.default_rng(count).integers(0, len(a), count)
    lib = box2d_amd.library()
    a, b, x, out = _take(Shape, a, index), _take(Shape, b, index), _take(Transform, x, index), (LocalManifold * count)()
    assert lib.b2amd_CollideBatch(a, b, x, count, out) == 0
    assert np.array_equal(manifold_array_words(out), want[index])
    a[count - 1].type = 4  # chain segments are refused
    before = ctypes.string_at(ctypes.byref(out), ctypes.sizeof(out))
    assert lib.b2amd_CollideBatch(a, b, x, count, out) == -1
    assert ctypes.string_at(ctypes.byref(out), ctypes.sizeof(out)) == before


@pytest.mark.parametrize("count", TOI_COUNTS)
def test_times_of_impact(count):
    n, toi_in, toi_out, _, _, _ = load()
    index = np.random.default_rng(count).integers(0, n, count)
    out = (TOIOutput * count)()
    assert box2d_amd.library().b2amd_TimeOfImpactBatch(_take(TOIInput, toi_in, index), count, out) == 0
    check_toi(bytes(out), toi_out[index])


@pytest.mark.parametrize("count", DISTANCE_COUNTS)
def test_distances(count):
    n, _, _, dist_in, dist_out, dist_caches = load()
    index = np.random.default_rng(count).integers(0, n, count)
    out, caches = (DistanceOutput * count)(), (SimplexCache * count)()
    lib = box2d_amd.library()
    assert lib.b2amd_ShapeDistanceBatch(_take(DistanceInput, dist_in, index), caches, count, out) == 0
    assert np.array_equal(distance_words(bytes(out)), distance_words(dist_out[index].tobytes()))
    assert bytes(caches) == dist_caches[index].tobytes()


@pytest.mark.parametrize("blocking", [False, True])
def test_inputs_written_by_earlier_work(blocking):
    n, toi_in, toi_out, dist_in, dist_out, _ = load()
    a, b, x, want = load_fixture()
    lib = box2d_amd.library()
    with EarlierWork(blocking) as work:
        out = (TOIOutput * n)()
        assert lib.b2amd_TimeOfImpactBatch(work.writes(toi_in), n, out) == 0
        check_toi(bytes(out), toi_out)
        out, caches = (DistanceOutput * n)(), (SimplexCache * n)()
        assert lib.b2amd_ShapeDistanceBatch(work.writes(dist_in), caches, n, out) == 0
        assert np.array_equal(distance_words(bytes(out)), distance_words(dist_out.tobytes()))
        index = np.arange(9000) % len(a)
        a, b, x = _take(Shape, a, index), _take(Shape, b, index), _take(Transform, x, index)
        out = (LocalManifold * len(index))()
        assert lib.b2amd_CollideBatch(work.writes(a), work.writes(b), work.writes(x), len(index), out) == 0
        assert np.array_equal(manifold_array_words(out), want[index])
