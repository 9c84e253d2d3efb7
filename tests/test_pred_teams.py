"""The ball-prediction kernel's teams (csrc/rsg_k_pred.hip) against a batch of
arenas without cars stepped one tick at a time by the plain kernel: the same
bits in every predicted record, whatever the trackers per wave (one of 16 lanes
to fifteen of 4, the most a wave's LDS holds; more are run as fifteen), for balls
in flight, rolling along curved walls and resting, at odd counts, in every mode,
fresh and carried on."""
import ctypes as C

import numpy as np
import pytest

from rocketsim_amd.ball_pred import BallPredTracker
from rocketsim_amd.batch import ArenaBatch
from rocketsim_amd.state import BallState, MODE_HEATSEEKER, MODE_HOOPS, MODE_SOCCAR, MODE_THE_VOID

pytestmark = pytest.mark.gpu
KERNEL_SCRATCH = 1


def _balls(n, seed, mode):
    rng = np.random.default_rng(seed)
    a = (BallState * n)()
    v = np.frombuffer(a, dtype=np.dtype(BallState))
    v["pos"] = rng.uniform([-3900, -5000, 93], [3900, 5000, 1900], (n, 3))
    if mode == MODE_HOOPS:
        v["pos"] *= [0.7, 0.6, 0.9]
    v["pos"][::3, 2] = 93.15        # on the floor and along the walls' curves
    v["vel"] = rng.normal(0, [1500, 1500, 700], (n, 3))
    v["vel"][::3, 2] = 0
    v["ang_vel"] = rng.normal(0, 2, (n, 3))
    v["vel"][1] = v["ang_vel"][1] = 0
    v["rot"] = np.eye(3).reshape(9)
    if mode == MODE_HEATSEEKER:
        v["hs_y_target_dir"][::2] = 1
        v["hs_cur_target_speed"][::2] = 2900
    return a


def _key(records):
    v = np.frombuffer(records, dtype=np.dtype(BallState))
    return b"".join(np.ascontiguousarray(v[f]).tobytes() for f in ("pos", "rot", "vel", "ang_vel"))


@pytest.mark.parametrize("mode", [MODE_SOCCAR, MODE_HOOPS, MODE_HEATSEEKER, MODE_THE_VOID])
def test_predictions_are_the_plain_kernels_ticks(mode):
    n, T, more = 67, 130, 7
    balls = _balls(n, 11 + mode, mode)
    b = ArenaBatch([0] * n, [], [], mode=mode)
    b.set_kernel(KERNEL_SCRATCH)
    b.set_balls(balls)
    want = []
    for t in range(T + more):
        want.append(_key(b.get_balls()))
        b.step(1)
    b.close()
    for per_wave in (0, 1, 3, 5, 7, 12, 15, 64):     # 16, 16, 16, 12, 9, 5, 4 and 4 lanes
        tr = BallPredTracker(mode=mode, n=n, num_pred_ticks=T)
        tr.set_launch(per_wave)
        tr.force_update_all_pred(balls)
        preds = [tr.pred_data(i) for i in range(n)]
        assert all(len(p) == T for p in preds)
        for t in range(1, T):   # row 0 is the state as given
            assert _key((BallState * n)(*[p[t] for p in preds])) == want[t], (per_wave, t)
        # the current state `more` ticks on matches: the last ticks are added
        tr.update_pred_manual((BallState * n)(*[p[more] for p in preds]), [more] * n)
        for i in (0, 1, n - 1):
            p = tr.pred_data(i)
            assert len(p) == T and bytes(p[0].pos) == bytes(preds[i][more].pos)
            assert [bytes(x.pos) for x in p[:T - more]] == [bytes(x.pos) for x in preds[i][more:]]
        tr.close()
