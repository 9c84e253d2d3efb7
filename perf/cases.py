"""Performance cases: the work that programs built on rocketsim_amd have it do,
through its public entry points.

  env    a learner's environment step: set every car's controls, advance the
         batch by a frame skip, read every car, ball and pad back
  sim    a rollout driven by the on-device control process, advanced in
         several calls, then read back once
  events a batch with the game-event tracker: a few ticks, tracker update,
         poll, read back
  pred   ball prediction: every tracker predicts its whole horizon anew
  track  ball prediction following a batch that is being stepped
  air    differentiable air control: rollout and gradients
  shot   differentiable aerial shot: rollout and gradients

Batches are played for a while from the kickoff before they are measured, so
that cars drive, jump, collide and touch the ball as they do in the middle of
a game.  The records of cars, balls, pads and predictions are returned as
their 32-bit words: a tick is a chain of branches on float comparisons
(contacts, friction clamps, penetration tests), in which one rounding changed
becomes another trajectory a few ticks later, so a batch is compared bit for
bit.
"""
import math
import random

import numpy as np
import torch

from rocketsim_amd.adjoint import air_rollout, shot_rollout
from rocketsim_amd.ball_pred import BallPredTracker
from rocketsim_amd.batch import ArenaBatch
from rocketsim_amd.game_events import GameEventTracker
from rocketsim_amd.state import (MODE_HEATSEEKER, MODE_HOOPS, MODE_SOCCAR, MODE_THE_VOID, NUM_PADS, PRED_WORDS,
                                 BallState, Controls)
from rocketsim_amd.workloads import shot_problem

MODES = {"soccar": MODE_SOCCAR, "hoops": MODE_HOOPS, "heatseeker": MODE_HEATSEEKER, "void": MODE_THE_VOID}
PREROLL = 480   # ticks (4 s) played from the kickoff before a case is measured
CAR_BYTES, BALL_BYTES, PAD_BYTES, CONTROLS_BYTES = 312, 104, 12, 24   # public records (include/rsg_state.h)


def listed():
    return [
        # one bot in one match: a frame skip of 8, the smallest call there is
        {"name": "env_1x1v1", "kind": "env", "mode": "soccar", "arenas": 1, "team": 1, "mixed": False, "skip": 8},
        # one learner worker's set of environments
        {"name": "env_64x2v2", "kind": "env", "mode": "soccar", "arenas": 64, "team": 2, "mixed": False, "skip": 8},
        # a full-size learner: thousands of 2v2 matches, every state read each step
        {"name": "env_4096x2v2", "kind": "env", "mode": "soccar", "arenas": 4096, "team": 2, "mixed": False, "skip": 8},
        # the benchmark's batch: 16384 2v2 matches, 8 calls of 8 ticks, then one look at the result
        {"name": "sim_16384x2v2", "kind": "sim", "mode": "soccar", "arenas": 16384, "team": 2, "mixed": False,
         "skip": 8, "calls": 8},
        # the uneven batch: 1v1, 2v2 and 3v3 matches side by side, six hitboxes
        {"name": "sim_32768mixed", "kind": "sim", "mode": "soccar", "arenas": 32768, "team": 3, "mixed": True,
         "skip": 8, "calls": 2},
        # another game mode at an odd size, 3v3, with shots, goals and saves tracked
        {"name": "events_1001x3v3_hoops", "kind": "events", "mode": "hoops", "arenas": 1001, "team": 3,
         "mixed": False, "skip": 4},
        # planning from thousands of imagined ball states, 6 s ahead
        {"name": "pred_4096x720", "kind": "pred", "mode": "soccar", "trackers": 4096, "horizon": 720},
        # bots that ask where the ball will be, every 8 ticks
        {"name": "track_999x240", "kind": "track", "mode": "soccar", "arenas": 999, "team": 1, "horizon": 240,
         "skip": 8},
        # trajectory optimisation of one manoeuvre, few candidates
        {"name": "air_257x45", "kind": "air", "cars": 257, "ticks": 45},
        # ... and of a whole population
        {"name": "air_65536x120", "kind": "air", "cars": 65536, "ticks": 120},
        {"name": "shot_101x60", "kind": "shot", "pairs": 101, "ticks": 60},
        {"name": "shot_16384x90", "kind": "shot", "pairs": 16384, "ticks": 90},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["env", "env", "sim", "sim", "events", "pred", "track", "air", "shot"])
    modes = ["soccar", "soccar", "soccar", "hoops", "heatseeker"]
    if kind == "env":
        return {"kind": kind, "mode": rng.choice(modes + ["void"]), "arenas": _log(rng, 1, 4096),
                "team": rng.randint(1, 4), "mixed": rng.random() < 0.3, "skip": rng.choice([1, 2, 4, 8])}
    if kind == "sim":
        return {"kind": kind, "mode": rng.choice(modes), "arenas": _log(rng, 16, 12000), "team": rng.randint(1, 3),
                "mixed": rng.random() < 0.3, "skip": rng.choice([1, 4, 8]), "calls": rng.randint(1, 8)}
    if kind == "events":
        return {"kind": kind, "mode": rng.choice(["soccar", "hoops"]), "arenas": _log(rng, 1, 4096),
                "team": rng.randint(1, 3), "mixed": False, "skip": rng.choice([1, 4, 8])}
    if kind == "pred":
        return {"kind": kind, "mode": rng.choice(modes), "trackers": _log(rng, 1, 4096),
                "horizon": _log(rng, 60, 720)}
    if kind == "track":
        return {"kind": kind, "mode": rng.choice(modes), "arenas": _log(rng, 1, 4096), "team": rng.randint(1, 2),
                "horizon": _log(rng, 60, 480), "skip": rng.choice([4, 8])}
    if kind == "air":
        return {"kind": kind, "cars": _log(rng, 16, 65536), "ticks": rng.randint(20, 120)}
    return {"kind": kind, "pairs": _log(rng, 16, 16384), "ticks": rng.randint(20, 90)}


# ---------------------------------------------------------------------------
# inputs

def _batch(case, seed, synth):
    rng = random.Random(seed)
    n, team = case["arenas"], case["team"]
    per_team = [team] * n
    if case.get("mixed"):   # 40 % 1v1, 35 % 2v2, 25 % 3v3, in an order of their own for each seed
        per_team = [min(team, 1 + int(i >= 0.4 * n) + int(i >= 0.75 * n)) for i in range(n)]
        rng.shuffle(per_team)
    teams, presets = [], []
    for k in per_team:
        teams += [0] * k + [1] * k
        presets += [rng.randrange(6) if case.get("mixed") else 0 for _ in range(2 * k)]
    b = ArenaBatch([2 * k for k in per_team], teams, presets, mode=MODES[case["mode"]], seed=seed & 0xFFFFFFFF,
                   synth_controls=synth, auto_reset=True)
    return b


def _controls(rng, n_cars):
    """A policy's outputs for every car: throttle mostly forward, steering,
    air control, and the buttons."""
    a = (Controls * n_cars)()
    v = np.frombuffer(a, dtype=np.dtype(Controls))
    v["throttle"] = np.clip(rng.normal(0.6, 0.6, n_cars), -1, 1)
    for f in ("steer", "pitch", "yaw", "roll"):
        v[f] = np.clip(rng.normal(0.0, 0.5, n_cars), -1, 1)
    for f, p in (("jump", 0.15), ("boost", 0.5), ("handbrake", 0.1)):
        v[f] = rng.random(n_cars) < p
    return a


def _ball_states(n, seed):
    """Balls anywhere in the field, moving as they do in play."""
    rng = np.random.default_rng(seed)
    a = (BallState * n)()
    v = np.frombuffer(a, dtype=np.dtype(BallState))
    v["pos"] = rng.uniform([-2700, -3300, 110], [2700, 3300, 1600], (n, 3))
    v["vel"] = rng.normal(0.0, [1200, 1200, 800], (n, 3))
    v["ang_vel"] = rng.normal(0.0, 2.0, (n, 3))
    v["rot"] = np.eye(3).reshape(9)
    return a


class _View:
    """A device array of the library as torch takes it, without a copy; the
    tensor keeps this object, and with it the array's owner."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<i4", "data": (ptr, False), "version": 2,
                                         "strides": None}


def _pred_tensors(tracker):
    v = tracker.view()
    n, t = v.n, v.num_pred_ticks
    traj, head, size = (torch.as_tensor(_View(tracker, p, s), device="cuda")
                        for p, s in ((v.traj, (t, PRED_WORDS, n)), (v.head, (n,)), (v.size, (n,))))
    return traj, head, size


def _words(records, n):
    """n public records as rows of 32-bit words."""
    return np.frombuffer(records, dtype=np.int32).reshape(n, -1)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("env", "sim", "events", "track"):
        b = _batch(case, seed, synth=kind != "env")
        s = {"case": case, "batch": b, "turn": 0}
        if kind == "env":
            rng = np.random.default_rng(seed)
            s["controls"] = [_controls(rng, b.n_cars) for _ in range(4)]
            for t in range(PREROLL // 40):
                b.set_controls(s["controls"][t % 4])
                b.step(40)
        else:
            for _ in range(PREROLL // 8):
                b.step(8)
        if kind == "events":
            s["tracker"] = GameEventTracker(b, capacity=1 << 14)
        if kind == "track":
            s["tracker"] = BallPredTracker(b, case["horizon"])
            s["view"] = _pred_tensors(s["tracker"])
        b.sync()
        return s
    if kind == "pred":
        n = case["trackers"]
        t = BallPredTracker(mode=MODES[case["mode"]], n=n, num_pred_ticks=case["horizon"])
        return {"case": case, "tracker": t, "view": _pred_tensors(t), "balls": _ball_states(n, seed)}
    if kind == "air":
        state0, controls, target = _air_problem(case["cars"], case["ticks"], seed)
    else:
        state0, controls, target = (x.cuda() for x in shot_problem(case["pairs"], case["ticks"], seed,
                                                                   dtype=torch.float32))
    return {"case": case, "state0": state0.requires_grad_(True), "controls": controls.requires_grad_(True),
            "target": target}


def _air_problem(n, ticks, seed):
    """Airborne cars anywhere, any orientation, tumbling; a target pose near by."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    rand = lambda *s: torch.rand(*s, device="cuda", generator=g)     # noqa: E731
    randn = lambda *s: torch.randn(*s, device="cuda", generator=g)   # noqa: E731
    pos = torch.cat([rand(n, 2) * 4000 - 2000, 800 + 1000 * rand(n, 1)], -1)
    quat = torch.nn.functional.normalize(randn(n, 4), dim=-1)
    state0 = torch.cat([pos, quat, randn(n, 3) * 500, randn(n, 3) * 2], -1)
    controls = torch.cat([torch.tanh(randn(ticks, n, 3)), torch.sigmoid(randn(ticks, n, 1))], -1)
    target = torch.cat([torch.nn.functional.normalize(randn(n, 4), dim=-1), pos + 300 * randn(n, 3)], -1)
    return state0, controls, target


# ---------------------------------------------------------------------------
# one pass

def _read(b):
    """Every car, ball and pad, as an agent's observation builder reads them."""
    return {"cars": _words(b.get_cars(), max(b.n_cars, 1)), "balls": _words(b.get_balls(), b.n_arenas),
            "pads": _words(b.get_pads(), b.n_arenas * NUM_PADS)}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "env":
        b = s["batch"]
        b.set_controls(s["controls"][s["turn"] % 4])
        s["turn"] += 1
        b.step(case["skip"])
        return _read(b)
    if kind == "sim":
        b = s["batch"]
        for _ in range(case["calls"]):
            b.step(case["skip"])
        return _read(b)
    if kind == "events":
        b = s["batch"]
        b.step(case["skip"])
        s["tracker"].update(b)
        events = s["tracker"].poll()
        out = _read(b)
        out["events"] = np.array([(e.arena, e.type, e.tick, e.a, e.b) for e in events],
                                 dtype=np.int64).reshape(-1, 5)
        return out
    if kind == "pred":
        s["tracker"].force_update_all_pred(s["balls"])
        return s["view"]
    if kind == "track":
        s["batch"].step(case["skip"])
        s["tracker"].update_pred_from_arena(s["batch"])
        return {"pred": s["view"], "balls": _words(s["batch"].get_balls(), s["batch"].n_arenas)}
    if kind == "air":
        loss, final = air_rollout(s["state0"], s["controls"], s["target"])
        ds0, dctrl = torch.autograd.grad(loss.sum(), [s["state0"], s["controls"]])
        return {"loss": loss, "final": final, "dstate0": ds0, "dcontrols": dctrl}
    loss, final, flags = shot_rollout(s["state0"], s["controls"], s["target"])
    ds0, dctrl = torch.autograd.grad(loss.sum(), [s["state0"], s["controls"]])
    return {"loss": loss, "final": final, "flags": flags, "dstate0": ds0, "dcontrols": dctrl}


# ---------------------------------------------------------------------------
# what a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind in ("env", "sim", "events", "track"):
        n, cars = case["arenas"], 2 * case["team"] * (0.62 if case.get("mixed") and case["team"] > 1 else 1.0)
        ticks = case["skip"] * case.get("calls", 1)
        state = cars * CAR_BYTES + BALL_BYTES + NUM_PADS * PAD_BYTES
        # the state in and out once, the controls in, the records out
        nbytes = n * (2 * state + state + (cars * CONTROLS_BYTES if kind == "env" else 0))
        # a car-tick: 4 wheel rays, suspension and friction of 4 wheels, the
        # car's logic, its body's step; a ball-tick: its body and contact
        flops = n * ticks * (cars * 3000 + 1000)
        if kind == "track":
            nbytes += n * case["skip"] * PRED_WORDS * 4
            flops += n * case["skip"] * 1000
        return {"bytes": float(nbytes), "flops": float(flops)}
    if kind == "pred":
        n, t = case["trackers"], case["horizon"]
        return {"bytes": float(n * (t + 1) * PRED_WORDS * 4), "flops": float(n * t * 1000)}
    words, n = (13, case["cars"]) if kind == "air" else (22, case["pairs"])
    t = case["ticks"]
    target = 7 if kind == "air" else 3
    # controls read and their gradient written, the states, loss and gradients; a tick takes
    # some 300 (air) and 450 (shot) operations forward, and its gradient twice that
    return {"bytes": float(4 * n * (t * 8 + 3 * words + target + 1)),
            "flops": float(n * t * 3 * (300 if kind == "air" else 450))}


def tolerance(case):
    if case["kind"] == "air":
        # 32-bit chains of up to 120 ticks and their adjoint: up to 1e-6 and
        # 3.5e-5 off the 64-bit result over all outputs and seeds tried
        return {"rel": 4e-6, "max": 1.4e-4}
    if case["kind"] == "shot":
        # as above, through the hit: loss and final state are within 1.3e-6, but
        # the gradient of a few grazing hits amplifies roundings, up to 6.8e-3
        # of the whole gradient's norm and 0.9 of its largest element
        return {"rel": 0.02, "max": 0.95, "differ": 1e-3}
    return "exact"


# ---------------------------------------------------------------------------
# 64-bit results of the differentiable rollouts (plain torch).  The tick of a
# batch has none: a whole match's collision detection and solver in 64 bits
# takes other branches than the 32-bit one.

def exact(case, seed):
    if case["kind"] not in ("air", "shot"):
        return None
    state = prepare(case, seed)
    parts = [[], [], [], []]
    n = state["state0"].shape[0]
    step = 65536 if case["kind"] == "air" else 8192
    for i in range(0, n, step):
        s0 = state["state0"].detach()[i:i + step].double().requires_grad_(True)
        c = state["controls"].detach()[:, i:i + step].double().requires_grad_(True)
        t = state["target"].detach()[i:i + step].double()
        loss, final = (_air64 if case["kind"] == "air" else _shot64)(s0, c, t)
        ds0, dc = torch.autograd.grad(loss.sum(), [s0, c])
        for p, x in zip(parts, (loss, final, ds0, dc)):
            p.append(x.detach())
    loss, final, ds0 = (torch.cat(p, 0) for p in parts[:3])
    out = {"loss": loss, "final": final, "dstate0": ds0, "dcontrols": torch.cat(parts[3], 1)}
    if case["kind"] == "shot":
        out["flags"] = None
    return out


BT = 50.0   # uu per Bullet unit
DT = 1.0 / 120.0
F32 = lambda x: float(np.float32(x))   # noqa: E731
TORQUE, DAMPING = (130.0, 95.0, 400.0), (30.0, 20.0, 50.0)   # pitch, yaw, roll
TORQUE_SCALE = 2 * math.pi / (1 << 16) * 1000


def _dot(a, b):
    return (a * b).sum(-1, keepdim=True)


def _cross(a, b):
    return torch.linalg.cross(a, b, dim=-1)


def _basis(q):
    x, y, z, w = q.unbind(-1)
    return (torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y + z * w), 2 * (z * x - w * y)], -1),
            torch.stack([2 * (x * y - w * z), 1 - 2 * (x * x + z * z), 2 * (y * z + w * x)], -1),
            torch.stack([2 * (z * x + y * w), 2 * (y * z - w * x), 1 - 2 * (x * x + y * y)], -1))


def _turn(w, q, dt):
    """q rotated by angular velocity w over dt, normalised."""
    th = w.norm(dim=-1, keepdim=True)
    small = th < 0.001
    ths = torch.where(small, torch.ones_like(th), th)
    a = w * torch.where(small, 0.5 * dt - dt ** 3 / 48.0 * th * th, torch.sin(0.5 * ths * dt) / ths)
    aw, bw = torch.cos(th * dt * 0.5), q[..., 3:]
    b = q[..., :3]
    h = torch.cat([aw * b + bw * a + _cross(a, b), aw * bw - _dot(a, b)], -1)
    return h / h.norm(dim=-1, keepdim=True)


def _cap(v, most):
    n = v.norm(dim=-1, keepdim=True)
    return torch.where(n > most, v * (most / n.clamp(min=1e-30)), v)


def _air_forces(q, v, w, ctrl):
    """The velocity and angular-velocity change of one tick of an airborne car."""
    p, y, r, boost = (c[..., None] for c in ctrl.unbind(-1))
    f, rt, u = _basis(q)
    torque = rt * (-p * TORQUE[0]) + u * (y * TORQUE[1]) + f * (-r * TORQUE[2])
    damp = (u * (DAMPING[1] * (1 - y.abs()) * _dot(u, w)) + rt * (DAMPING[0] * (1 - p.abs()) * _dot(rt, w))
            + f * (DAMPING[2] * _dot(f, w)))
    g = torch.zeros_like(v)
    g[..., 2] = -650.0 / BT
    return (g + f * (boost * (3175.0 / 3.0 / BT))) * DT, (torque - damp) * (TORQUE_SCALE * DT), g * DT, (f, rt, u)


def _air64(state0, controls, target):
    p, q, v, w = state0[:, 0:3] / BT, state0[:, 3:7], state0[:, 7:10] / BT, state0[:, 10:13]
    for c in controls:
        dv, dw, _, _ = _air_forces(q, v, w, c)
        v, w = v + dv, w + dw
        p, q = p + v * DT, _turn(w, q, DT)
        v, w = _cap(v, 2300.0 / BT), _cap(w, 5.5)
    d = (q * target[:, :4]).sum(-1).abs().clamp(max=1 - 1e-6)
    return 2 * torch.acos(d) + 1e-4 * ((p * BT - target[:, 4:]) ** 2).sum(-1), torch.cat([p * BT, q, v * BT, w], -1)


# Octane's hitbox and the ball
_HALF = [F32(h) / BT / 2 for h in (120.507, 86.6994, 38.6591)]
_CORE = [h - 0.04 for h in _HALF]
_MARGIN = min(0.1 * min(_HALF), 0.04)
_OFFSET = [F32(o) / BT for o in (13.8757, 0.0, 20.755)]
_FULL = [h + _MARGIN for h in _CORE]
_INV_I = [3 / (180.0 * (_FULL[a] ** 2 + _FULL[b] ** 2)) for a, b in ((1, 2), (0, 2), (0, 1))]
_CAR_INV_M, _BALL_INV_M = 1 / 180.0, 1 / 30.0
_RADIUS = F32(91.25) / BT
_BALL_INV_I = 1 / (0.4 * 30.0 * _RADIUS ** 2)
_BREAKING = 0.02 * min(math.hypot(*_FULL) + math.hypot(*_OFFSET), _RADIUS + 0.08)
_EXTRA = ((0.0, 0.65), (500.0, 0.65), (2300.0, 0.55), (4600.0, 0.30))


def _curve(x):
    out = torch.full_like(x, _EXTRA[-1][1])
    for (x0, y0), (x1, y1) in reversed(list(zip(_EXTRA[:-1], _EXTRA[1:]))):
        out = torch.where(x < x1, y0 + (y1 - y0) * (x - x0) / (x1 - x0), out)
    return out


def _unit(a):
    n = a.norm(dim=-1, keepdim=True)
    return torch.where(n > 0, a / torch.where(n > 0, n, torch.ones_like(n)), torch.zeros_like(a))


def _shot64(state0, controls, target):
    cp, cq, cv, cw = state0[:, 0:3] / BT, state0[:, 3:7], state0[:, 7:10] / BT, state0[:, 10:13]
    bp, bv, bw = state0[:, 13:16] / BT, state0[:, 16:19] / BT, state0[:, 19:22]
    last = torch.full_like(cp[:, :1], -1000.0)
    for t in range(controls.shape[0]):
        ext_f, ext_t, ext_b, axes = _air_forces(cq, cv, cw, controls[t])
        bv = bv * (1.0 - 0.03) ** DT
        car_v, car_w, ball_v, ball_w, push, last, cache = _hit64(cp, cq, cv, cw, bp, bv, bw, ext_f, ext_t, ext_b,
                                                                 axes, t, last)
        if push is not None:
            hit, a_push, a_turn, b_push = push
            cp = cp + a_push * DT
            cq = torch.where(hit & (a_turn != 0).any(-1, keepdim=True), _turn(a_turn * 0.1, cq, DT), cq)
            bp = bp + b_push * DT
        cp, cq, bp = cp + car_v * DT, _turn(car_w, cq, DT), bp + ball_v * DT
        cv, cw = _cap(car_v, 2300.0 / BT), _cap(car_w, 5.5)
        bv, bw = _cap(ball_v + cache, 6000.0 / BT), _cap(ball_w, 6.0)
    return (bp * BT - target).norm(dim=-1), torch.cat([cp * BT, cq, cv * BT, cw, bp * BT, bv * BT, bw], -1)


def _hit64(cp, cq, cv, cw, bp, bv, bw, ext_f, ext_t, ext_b, axes, tick, last):
    """The velocities after one tick's car-ball contact, if there is one: the
    extra hit impulse, then 10 position and 10 velocity passes over a normal
    and a friction row."""
    f, r, u = axes
    zero = torch.zeros_like(cv)
    box = cp + f * _OFFSET[0] + r * _OFFSET[1] + u * _OFFSET[2]
    d = bp - box
    loc = torch.cat([_dot(f, d), _dot(r, d), _dot(u, d)], -1)
    he = torch.tensor(_CORE, dtype=loc.dtype, device=loc.device)
    inside = (loc.abs() < he).all(-1, keepdim=True)
    q = torch.maximum(torch.minimum(loc, he), -he)
    to_box = (box + f * q[:, 0:1] + r * q[:, 1:2] + u * q[:, 2:3]) - bp
    far = to_box.norm(dim=-1, keepdim=True)
    depth = far - (_MARGIN + _RADIUS)
    hit = ~inside & (depth < _BREAKING) & (far > 0)
    if not bool(hit.any()):
        return cv + ext_f, cw + ext_t, bv + ext_b, bw, None, last, zero
    n = to_box / torch.where(hit, far, torch.ones_like(far))
    pt_b = bp + n * _RADIUS
    rel1, rel2 = pt_b + n * depth - cp, pt_b - bp

    extra = hit & ((tick > last + 1) | (last > tick))
    rel_v = bv * BT - cv * BT
    speed = rel_v.norm(dim=-1, keepdim=True).clamp(max=4600.0)
    way = _unit((bp * BT - cp * BT) * torch.tensor([1.0, 1.0, 0.35], dtype=bp.dtype, device=bp.device))
    way = _unit(way - f * _dot(way, f) * (1 - 0.65))
    cache = torch.where(extra & (speed > 0), way * speed * _curve(speed) / BT, zero)
    last = torch.where(extra, torch.full_like(last, float(tick)), last)

    def inv_i(x):
        return f * (_INV_I[0] * _dot(f, x)) + r * (_INV_I[1] * _dot(r, x)) + u * (_INV_I[2] * _dot(u, x))

    def row(axis):
        j1, j2 = _cross(rel1, axis), _cross(rel2, -axis)
        a, b = inv_i(j1), j2 * _BALL_INV_I
        jac = 1 / ((_CAR_INV_M + _dot(axis, _cross(a, rel1))) + (_BALL_INV_M + _dot(axis, _cross(-b, rel2))))
        return axis, j1, j2, a, b, jac

    def along(x, dv1, dw1, dv2, dw2):
        return _dot(x[0], dv1 - dv2) + _dot(x[1], dw1) + _dot(x[2], dw2)

    def moved(x, m, delta):
        return (m[0] + x[0] * _CAR_INV_M * delta, m[1] + x[3] * delta, m[2] - x[0] * _BALL_INV_M * delta,
                m[3] + x[4] * delta)

    nr = row(n)
    rhs = -along(nr, cv + ext_f, cw + ext_t, bv + ext_b, bw) * nr[5]
    pen = torch.where(depth > 0, torch.zeros_like(depth), -depth * 0.8 / DT) * nr[5]
    vel = ((cv + ext_f) + _cross(cw + ext_t, rel1)) - ((bv + ext_b) + _cross(bw, rel2))
    side = vel - n * _dot(n, vel)
    lat = _dot(side, side)
    slides = lat > 1.1920928955078125e-07
    steep = n[:, 2:].abs() > 0.7071067811865475244
    yz, xy = n[:, 1:2] ** 2 + n[:, 2:] ** 2, n[:, 0:1] ** 2 + n[:, 1:2] ** 2
    k1, k2 = (1 / torch.sqrt(torch.where(a > 0, a, torch.ones_like(a))) for a in (yz, xy))
    flat = torch.zeros_like(k1)
    still = torch.where(steep, torch.cat([flat, -n[:, 2:] * k1, n[:, 1:2] * k1], -1),
                        torch.cat([-n[:, 1:2] * k2, n[:, 0:1] * k2, flat], -1))
    fr = row(torch.where(slides, side / torch.sqrt(torch.where(slides, lat, torch.ones_like(lat))), still))
    f_rhs = -along(fr, cv + ext_f, cw, bv + ext_b, bw) * fr[5]

    m, applied = (zero, zero, zero, zero), torch.zeros_like(depth)
    on = hit & (pen != 0)
    for _ in range(10):
        delta = pen - along(nr, *m) * nr[5]
        total = applied + delta
        delta = torch.where(on, torch.where(total < 0, -applied, delta), torch.zeros_like(delta))
        applied = torch.where(on, total.clamp(min=0), applied)
        m = moved(nr, m, delta)
        on = on & (delta != 0)
    a_push, a_turn, b_push, _ = (torch.where(hit, x, zero) for x in m)

    m, applied, f_applied = (zero, zero, zero, zero), torch.zeros_like(depth), torch.zeros_like(depth)
    for _ in range(10):
        delta = rhs - along(nr, *m) * nr[5]
        total = applied + delta
        delta = torch.where(total < 0, -applied, delta)
        applied = total.clamp(min=0)
        m = moved(nr, m, delta)
        most = 2.0 * applied
        delta = f_rhs - along(fr, *m) * fr[5]
        new = torch.maximum(torch.minimum(f_applied + delta, most), -most)
        new = torch.where(applied > 0, new, f_applied)
        m = moved(fr, m, new - f_applied)
        f_applied = new
    dv1, dw1, dv2, dw2 = (torch.where(hit, x, zero) for x in m)
    return (cv + dv1 + ext_f, cw + dw1 + ext_t, bv + dv2 + ext_b, bw + dw2, (hit, a_push, a_turn, b_push), last,
            cache)
