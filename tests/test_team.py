"""The tick by phases that a team of lanes runs (rocketsim_amd/csrc/rsg_team.h,
the cooperative kernel's) against the tick as one lane runs it (arena_tick):
the same bits in every record after every tick, over the game modes, no cars
to the most a team takes, and with the capacities so low that play overflows
them (manifolds in the local block and past it, solver rows, recorded effects)."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import tick_host
from rocketsim_amd import arena_mesh, native
from rocketsim_amd.state import (ARENA_MODES, BallState, CarState, Controls, MODE_HEATSEEKER, MODE_HOOPS, MODE_SOCCAR,
                                 MODE_THE_VOID, MutatorConfig, NUM_PADS, PadState)

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def build(tmp_path_factory):
    made = {}

    def get(*defines):
        if defines not in made:
            libs = []
            for src in ("tick_host.cpp", "team_host.cpp"):
                out = str(tmp_path_factory.mktemp("team") / (src + ".so"))
                r = subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared",
                                    *["-D" + d for d in defines], "-I" + os.path.join(ROOT, "include"),
                                    os.path.join(HERE, "cpp", src), "-o", out], capture_output=True, text=True)
                assert r.returncode == 0, r.stderr[-3000:]
                libs.append(tick_host.load(out))
            made[defines] = libs
        return made[defines]

    return get


def _rotations(rng, n):
    q = rng.normal(size=(n, 4))
    x, y, z, w = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                     2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                     2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], -1)


def _rollout(L, mode, per_team, ticks, seed, rotate_ball=False, ball_radius=None):
    """Every tick's records of one arena per entry of per_team: cars about the
    ball and anywhere, upright and tumbling, under random controls."""
    rng = np.random.default_rng(seed)
    n = len(per_team)
    total = 2 * sum(per_team)
    teams = sum(([0] * k + [1] * k for k in per_team), [])
    presets = [int(p) for p in rng.integers(0, 7, total)]
    cmfs = [] if mode not in ARENA_MODES else (
        arena_mesh.hoops_cmfs() if mode == MODE_HOOPS else [arena_mesh.soccar_cmf()])
    mut = None
    if ball_radius:
        mut = MutatorConfig()
        native.check(native.lib().rsg_mutator_config_default(mode, C.byref(mut)))
        mut.ball_radius = ball_radius
    h = L.th_create(mode, n, (C.c_int * n)(*[2 * k for k in per_team]), (C.c_uint8 * max(total, 1))(*teams),
                    (C.c_uint8 * max(total, 1))(*presets), *tick_host.mesh_args(cmfs), 120.0,
                    C.byref(mut) if mut is not None else None, None)
    if rotate_ball:
        L.th_set_ball_rotation(h, 1)
    cars, balls, ctl = (CarState * max(total, 1))(), (BallState * n)(), (Controls * max(total, 1))()
    pads, status = (PadState * (n * NUM_PADS))(), (C.c_uint32 * n)()
    L.th_get_balls(h, balls)
    b = np.frombuffer(balls, dtype=np.dtype(BallState))
    b["pos"][:] = rng.uniform([-800, -800, 95], [800, 800, 700], (n, 3))
    b["vel"][:] = rng.normal(0, 700, (n, 3))
    L.th_set_balls(h, balls)
    if total:
        L.th_get_cars(h, cars)
        v = np.frombuffer(cars, dtype=np.dtype(CarState))
        v["pos"][:] = rng.uniform([-3800, -4900, 17], [3800, 4900, 400], (total, 3))
        close = rng.random(total) < 0.5
        v["pos"][close] = rng.uniform([-600, -600, 17], [600, 600, 300], (close.sum(), 3))
        v["vel"][:] = rng.normal(0, 900, (total, 3))
        tumbling = rng.random(total) < 0.5
        v["rot"][:] = np.eye(3).reshape(9)
        v["rot"][tumbling] = _rotations(rng, total)[tumbling]
        v["boost"][:] = rng.uniform(0, 100, total)
        L.th_set_cars(h, cars)
    cv = np.frombuffer(ctl, dtype=np.dtype(Controls))
    trace = []
    for t in range(ticks):
        if t % 20 == 0 and total:
            cv["throttle"] = np.clip(rng.normal(0.6, 0.6, total), -1, 1)
            for f in ("steer", "pitch", "yaw", "roll"):
                cv[f] = rng.uniform(-1, 1, total)
            for f, p in (("jump", .3), ("boost", .5), ("handbrake", .2)):
                cv[f] = rng.random(total) < p
            L.th_set_controls(h, ctl)
        L.th_step(h, 1)
        for get, buf in ((L.th_get_cars, cars), (L.th_get_balls, balls), (L.th_get_pads, pads),
                         (L.th_get_status, status)):
            get(h, buf)
        trace.append(tuple(bytes(x) for x in (cars, balls, pads, status)))
    L.th_destroy(h)
    return trace


def _compare(libs, *args, **kw):
    one, team = (_rollout(L, *args, **kw) for L in libs)
    for t, (x, y) in enumerate(zip(one, team)):
        for what, p, q in zip(("cars", "balls", "pads", "status"), x, y):
            assert p == q, f"{what} differ after tick {t + 1}"
    return np.frombuffer(one[-1][3], np.uint32)


@pytest.mark.parametrize("mode,per_team,ticks,rotate_ball", [
    (MODE_SOCCAR, [0, 1, 2, 3, 4] * 3, 240, False),
    (MODE_SOCCAR, [2, 4], 120, True),
    (MODE_HOOPS, [1, 2, 3] * 3, 180, False),
    (MODE_HEATSEEKER, [1, 2] * 4, 240, True),
    (MODE_THE_VOID, [1, 2] * 3, 180, False),
])
def test_phases_match_the_serial_tick(build, mode, per_team, ticks, rotate_ball):
    assert not _compare(build(), mode, per_team, ticks, 1, rotate_ball=rotate_ball).any()


@pytest.mark.parametrize("mode", [MODE_SOCCAR, MODE_HOOPS])
def test_phases_match_where_the_tree_serves_the_ball(build, mode):
    # a ball whose box the leaf lists do not serve, beside cars that they serve
    assert not _compare(build(), mode, [0, 1, 2] * 5, 240, 5, ball_radius=240.0).any()


@pytest.mark.parametrize("limit", ["RSG_TEST_MAX_MANIFOLDS=1", "RSG_TEST_MAX_MANIFOLDS=2",
                                   "RSG_TEST_MAX_SOLVER_ROWS=2", "RSG_TEST_MAX_SOLVER_ROWS=3",
                                   "RSG_TEST_PAIR_EFFECTS=1", "RSG_SSE_NORMALIZE"])
def test_phases_match_at_the_capacities(build, limit):
    status = _compare(build(limit), MODE_SOCCAR, [1, 2, 3, 4] * 3, 160, 3)
    assert status.any() == ("MAX" in limit)  # the low capacities were reached
