"""The backward kernel's two forms, a world's constraints one per thread (up to 256) and more than
that, against the oracle's float64 reverse mode with the recorded branch pattern held fixed, to the
1e-3 relative of the other adjoint checks."""

import numpy as np
import pytest

from adjoint_ref import WorldRecord
from earlier_work import EarlierWork
from nets import add_circles

pytestmark = pytest.mark.gpu

# rows, whether a step holds more than 256 constraints
SIZES = [(2, False), (13, False), (14, True), (17, True)]


@pytest.mark.parametrize("rows,large", SIZES)
def test_backward_forms_match_fp64_adjoint(rows, large):
    from box2d_amd.adjoint import BODY_STATE, PushWorlds

    rng = np.random.default_rng(rows)
    # fast pushers that hit within six steps, and a sixth of the horizon that the 1e-3 covers in the
    # 10-row world, so that float32 rounding, which grows with the number of steps reversed, stays below
    # it in the larger ones too (after 24 steps the 14-row world's is 1.3e-3)
    params = np.stack([rng.uniform(5, 6, 2), rng.uniform(-0.5, 0.5, 2), rng.uniform(-1, 1, 2), rng.uniform(0.3, 0.9, 2)], 1)
    goals = np.array([[0.5, rows - 1.0], [-0.5, rows - 0.5]])
    steps = 10
    pw = PushWorlds(params, rows=rows)
    try:
        tape = pw.record(steps)
        most = max(int(tape.read_step(w, k)[0]["constraintCount"]) for w in range(2) for k in range(steps))
        assert (most > 256) == large, most
        final = tape.final_states()
        # the loss looks at the box the pusher hits first: the first of the bottom row
        target = [int(b[0]) for b in pw.body_ids]
        fg = np.zeros((2, tape.body_stride), dtype=BODY_STATE)
        for w in range(2):
            fg[w]["center"][target[w]] = 2.0 * (final[w]["center"][target[w]] - goals[w])
        ig, fr, stats = tape.backward(fg)
        assert stats.unsupported == 0 and stats.replayMismatches == 0
        shapes = pw.pusher_shape_ids()
        for w in range(2):
            pusher = int(pw.body_ids[w][-1])
            got = np.array([*ig[w]["linearVelocity"][pusher], ig[w]["angularVelocity"][pusher], fr[w, shapes[w]]], dtype=np.float64)
            rec = WorldRecord.from_tape(tape, w)
            want, _ = rec.push_gradients(rec.slot_of(pusher), shapes[w], rec.slot_of(target[w]), goals[w])
            assert np.linalg.norm(got - want) <= 1e-3 * np.linalg.norm(want), (w, got, want)
    finally:
        pw.destroy()


@pytest.mark.parametrize("blocking", [False, True])
def test_final_gradient_written_by_earlier_work(blocking):
    import ctypes

    from box2d_amd.adjoint import BODY_STATE, PushWorlds

    pw = PushWorlds(np.array([[5.0, 0.1, 0.3, 0.5]]), rows=3)
    try:
        tape = pw.record(8)
        fg = np.zeros((1, tape.body_stride), dtype=BODY_STATE)
        fg["center"] = np.random.default_rng(1).uniform(-1, 1, (1, tape.body_stride, 2))
        want, _, _ = tape.backward(fg)
        assert np.any(want["linearVelocity"] != 0)
        with EarlierWork(blocking) as work:
            got = np.zeros_like(want)
            records = (ctypes.c_byte * fg.nbytes).from_buffer_copy(fg.tobytes())
            assert tape.lib.b2amd_Tape_Backward(tape.handle, work.writes(records), got.ctypes.data_as(ctypes.c_void_p), None, None) == 0
        assert got.tobytes() == want.tobytes()
    finally:
        pw.destroy()


@pytest.mark.parametrize("rows", [1, 5, 14, 17])
def test_friction_gradients_of_all_shapes(rows):
    """The ground's sum, which many constraints of a color share, and the boxes'."""
    from box2d_amd.adjoint import BODY_STATE, PushWorlds

    pw = PushWorlds(np.array([[5.5, 0.2, 0.4, 0.5]]), rows=rows)
    try:
        tape = pw.record(10)
        final = tape.final_states()
        target, pusher = int(pw.body_ids[0][0]), int(pw.body_ids[0][-1])
        goal = np.array([0.5, rows - 1.0])
        fg = np.zeros((1, tape.body_stride), dtype=BODY_STATE)
        fg[0]["center"][target] = 2.0 * (final[0]["center"][target] - goal)
        _, fr, stats = tape.backward(fg)
        assert stats.unsupported == 0 and stats.replayMismatches == 0
        rec = WorldRecord.from_tape(tape, 0)
        _, want = rec.push_gradients(rec.slot_of(pusher), pw.pusher_shape_ids()[0], rec.slot_of(target), goal)
        want = np.asarray(want["grad_friction"])[:fr.shape[1]]
        assert np.count_nonzero(want) > rows
        assert np.linalg.norm(fr[0][:len(want)] - want) <= 1e-3 * np.linalg.norm(want)
    finally:
        pw.destroy()


def test_shapes_without_contacts_cost_nothing():
    """The backward kernel's time does not grow with the world's shapes, only with its contacts."""
    from box2d_amd.adjoint import BODY_STATE, PushWorlds

    def milliseconds(extra):
        pw = PushWorlds(np.array([[5.0, 0.1, 0.3, 0.5]]), rows=10)
        try:
            add_circles(pw.ids[0], extra, 200.0)
            tape = pw.record(10)
            fg = np.zeros((1, tape.body_stride), dtype=BODY_STATE)
            fg["center"] = 1.0
            return min(tape.backward(fg)[2].backwardMs for _ in range(3))
        finally:
            pw.destroy()

    assert milliseconds(5000) < 1.5 * milliseconds(0)
