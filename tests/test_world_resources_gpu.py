"""Worlds share streams and memory blocks: more worlds than streams, made, stepped and dropped from
several threads, or while the default stream is busy, each end bit for bit as a world that runs alone; and
transforms of more bodies than one readback holds."""

import ctypes
import threading

import numpy as np
import pytest

import box2d_amd
from earlier_work import EarlierWork

pytestmark = pytest.mark.gpu


def _state(scenes, h):
    return scenes.transforms(h).tobytes() + scenes.velocities(h).tobytes()


def _make(scenes, size):
    return scenes.create(box2d_amd.SCENE_MIXED_PILE, (size, 0, 77))


@pytest.mark.parametrize("threads,worlds,sizes", [(1, 20, (3, 130)), (4, 5, (1, 40, 600))])
def test_worlds_made_and_dropped_in_threads(gpu_scenes, threads, worlds, sizes):
    steps = 40
    alone = {}
    for size in sizes:
        h = _make(gpu_scenes, size)
        gpu_scenes.step(h, steps)
        alone[size] = _state(gpu_scenes, h)
        gpu_scenes.destroy(h)
    lock = threading.Lock()  # worlds are made and dropped by one thread at a time
    wrong = []

    def work(seed):
        rng = np.random.default_rng(seed)
        live = []
        for _ in range(worlds):
            size = int(rng.choice(sizes))
            with lock:
                live.append((size, _make(gpu_scenes, size)))
            for k, (_, h) in enumerate(live):
                gpu_scenes.step(h, 3 + k)
            if rng.random() < 0.4:
                with lock:
                    gpu_scenes.destroy(live.pop(0)[1])
            size = int(rng.choice(sizes))
            with lock:
                fresh = _make(gpu_scenes, size)
            gpu_scenes.step(fresh, steps)
            if _state(gpu_scenes, fresh) != alone[size]:
                wrong.append((seed, size))
            with lock:
                gpu_scenes.destroy(fresh)
        with lock:
            for _, h in live:
                gpu_scenes.destroy(h)

    pool = [threading.Thread(target=work, args=(s,)) for s in range(threads)]
    for t in pool:
        t.start()
    for t in pool:
        t.join()
    assert wrong == []


@pytest.mark.parametrize("together", [False, True])
def test_worlds_made_while_the_default_stream_is_busy(gpu_scenes, together):
    steps, sizes = 30, (1, 40, 130, 300)

    def run():
        worlds = [gpu_scenes.create(box2d_amd.SCENE_MIXED_PILE, (n, 1, 77)) for n in sizes]
        ids = (box2d_amd.WorldId * len(worlds))(*[gpu_scenes.world_id(h) for h in worlds])
        if together:
            box2d_amd.step_worlds(ids, steps)
        else:
            for h in worlds:
                gpu_scenes.step(h, steps)
        out = [(_state(gpu_scenes, h), gpu_scenes.counters(h)) for h in worlds]
        for h in worlds:
            gpu_scenes.destroy(h)
        return out

    want = run()
    with EarlierWork(False) as work:
        work.writes((ctypes.c_int * 16)())
        assert run() == want


@pytest.mark.parametrize("rows", [457, 458])  # 104,653 and 105,111 boxes; one readback holds 104,857
def test_transforms_of_many_bodies(gpu_scenes, rows):
    h = gpu_scenes.pyramid(rows)
    try:
        before = gpu_scenes.transforms(h)
        boxes = before[-rows * (rows + 1) // 2:, :2]
        levels, counts = np.unique(np.round(boxes[:, 1], 3), return_counts=True)
        assert counts.tolist() == list(range(rows, 0, -1))
        for y, n in zip(levels, counts):
            x = np.sort(boxes[np.round(boxes[:, 1], 3) == y][:, 0])
            assert np.all(np.diff(x) > 0.5) and x.size == n
    finally:
        gpu_scenes.destroy(h)
