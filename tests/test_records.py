"""Reading cars, balls and pads from the device and writing controls to it
(csrc/rsg_k_records.hip) against the host's conversion of the downloaded
state: the same bytes, for the smallest batch, ragged ones around a wave's 64
records, arenas without cars, a batch read in one launch and ones read kind by
kind and in several pieces; and controls that take the one way or the other."""
import ctypes as C

import numpy as np
import pytest

from rocketsim_amd.batch import ArenaBatch
from rocketsim_amd.game_events import GameEventTracker
from rocketsim_amd.state import Controls, MODE_HEATSEEKER, MODE_HOOPS, MODE_SOCCAR, MODE_THE_VOID

pytestmark = pytest.mark.gpu


def _batch(per_arena, mode=MODE_SOCCAR, **kw):
    teams = sum(([i % 2 for i in range(k)] for k in per_arena), [])
    return ArenaBatch(list(per_arena), teams, [i % 6 for i in range(len(teams))], mode=mode, seed=7, **kw)


def _records(b):
    return bytes(b.get_cars()), bytes(b.get_balls()), bytes(b.get_pads())


@pytest.mark.parametrize("mode,per_arena", [
    (MODE_SOCCAR, [1]), (MODE_SOCCAR, [0]), (MODE_SOCCAR, [2] * 31 + [3]), (MODE_HOOPS, [0, 6, 1, 3, 2] * 13),
    (MODE_THE_VOID, [1] * 64), (MODE_HEATSEEKER, [8] * 65 + [0]), (MODE_SOCCAR, [4, 2, 6] * 700),
    (MODE_SOCCAR, [8] * 26900),   # more than one piece of cars
], ids=lambda v: str(v) if isinstance(v, int) else f"{len(v)}x{max(v)}")
def test_device_records_equal_the_mirrors(mode, per_arena):
    b = _batch(per_arena, mode, synth_controls=True, auto_reset=True, ball_rotation=True)
    b.step(20 if len(per_arena) > 10000 else 90)
    got = _records(b)
    again = _records(b)
    b.get_goals()               # downloads the mirror, which then serves the getters
    want = _records(b)
    for what, x, y, z in zip(("cars", "balls", "pads"), got, again, want):
        assert x == z, what
        assert y == z, what + " read again"
    b.close()


@pytest.mark.parametrize("arenas", [1, 33, 1500])
def test_controls_on_either_way(arenas):
    def play(mirror):
        b = _batch([2] * arenas)
        rng = np.random.default_rng(3)
        out = []
        for t in range(6):
            ctl = (Controls * b.n_cars)()
            v = np.frombuffer(ctl, dtype=np.dtype(Controls))
            for f in ("throttle", "steer", "pitch", "yaw", "roll"):
                v[f] = rng.uniform(-1, 1, b.n_cars)
            for f in ("jump", "boost", "handbrake"):
                v[f] = rng.integers(0, 3, b.n_cars)
            if mirror:
                b.set_tick_counts(b.get_tick_counts())      # the mirror is the newest now
            b.set_controls(ctl if t % 2 else list(ctl))
            if t == 2:
                b.set_controls(ctl)                         # again before any step
            if t == 3:
                out.append(bytes(b.get_controls()))
            if t == 4:
                b.set_balls(b.get_balls())                  # the mirror takes them over
            b.step(3)
            if t != 1:                                      # once without a read in between
                out += _records(b)
            out.append(bytes(b.get_controls()))
        b.graph_create(2, 2)
        b.set_controls((Controls * b.n_cars)(*[Controls(throttle=1.0)] * b.n_cars))
        b.graph_launch()
        out += _records(b)
        b.close()
        return out

    assert play(False) == play(True)


@pytest.mark.parametrize("arenas", [1, 33, 1500])
def test_what_was_set_is_read_back_after_uploads_without_a_step(arenas):
    """A state set after a read goes to the device by one call that does not
    step, controls set then by another; the getters give what was set."""
    b = _batch([2] * arenas)
    tracker = GameEventTracker(b)
    b.step(30)
    before = _records(b)
    cars, balls, pads = b.get_cars(), b.get_balls(), b.get_pads()
    for c in cars:
        c.boost = 77.0
    for x in balls:
        x.pos[0], x.vel[2] = 123.0, 456.0
    for p in pads:
        p.cooldown, p.is_active = 3.0, 0
    b.set_cars(cars)
    b.set_balls(balls)
    b.set_pads(pads)
    tracker.update(b)               # the set state to the device
    b.set_controls((Controls * b.n_cars)(*[Controls(throttle=1.0)] * b.n_cars))
    tracker.update(b)               # the controls to the device
    got = _records(b)               # the device's are the newer
    b.get_goals()
    want = _records(b)              # the mirror's
    tracker.close()
    b.close()
    for what, x, y, z in zip(("cars", "balls", "pads"), got, want, before):
        assert x == y, what
        assert x != z, what + " as before the set"


@pytest.mark.parametrize("arenas", [3, 1500])
def test_reads_wait_for_replays_of_a_captured_step(arenas):
    """A step that the caller records into a graph of its own and replays on
    another stream: each read gives the state after the replay before it."""
    torch = pytest.importorskip("torch")
    a, b = (_batch([2] * arenas, synth_controls=True, auto_reset=True) for _ in range(2))
    a.step(1)
    b.step(1)
    torch.cuda.synchronize()
    record, replay = torch.cuda.Stream(), torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(record):
        graph.capture_begin()
        b.step(100, stream=record.cuda_stream)      # some 10 ms
        graph.capture_end()
    for _ in range(3):
        a.step(100)
        with torch.cuda.stream(replay):
            graph.replay()
        assert _records(b) == _records(a)
    a.close()
    b.close()
