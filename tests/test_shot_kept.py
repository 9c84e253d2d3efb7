"""The shot's backward pass over every tick's state (the hand-written adjoint in
flight, tangents on contact ticks) against the one that takes 26 tangents on
every tick of a recomputed segment: the same loss, final state and flags bit
for bit, and gradients within the rounding of their chains, at one and several
pairs a wave, with ragged last waves and tick counts down to one."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ticks", [(1, 1), (65, 33), (1025, 20), (2500, 40), (66000, 3)])
def test_kept_states_give_the_same_gradients(n, ticks):
    from rocketsim_amd import native
    from rocketsim_amd.workloads import shot_problem
    L = native.lib()
    s0, ctrl, tgt = shot_problem(n, ticks, n + ticks, dtype=torch.float32)
    s0, ctrl, tgt = s0.t().contiguous().cuda(), ctrl.permute(0, 2, 1).contiguous().cuda(), tgt.t().contiguous().cuda()
    new = lambda *shape: torch.zeros(*shape, device="cuda")     # noqa: E731
    dl = torch.ones(n, device="cuda")
    out = []
    for every in (16, 1):
        ckpt = new(((ticks + every - 1) // every) * 23 * n)
        final, loss, flags, dc, ds = new(22, n), new(n), new(n).int(), new(ticks, 4, n), new(22, n)
        native.check(L.rsg_shot_rollout(n, ticks, every, 120.0, s0.data_ptr(), ctrl.data_ptr(), tgt.data_ptr(),
                                        final.data_ptr(), loss.data_ptr(), ckpt.data_ptr(), flags.data_ptr(), None))
        native.check(L.rsg_shot_rollout_backward(n, ticks, every, 120.0, ctrl.data_ptr(), tgt.data_ptr(),
                                                 ckpt.data_ptr(), dl.data_ptr(), dc.data_ptr(), ds.data_ptr(), None))
        torch.cuda.synchronize()
        out.append((loss, final, flags, torch.cat([ds, dc.reshape(-1, n)]).t().contiguous()))
    for a, b in zip(out[0][:3], out[1][:3]):
        assert torch.equal(a, b)
    a, b = out[0][3].double(), out[1][3].double()
    # each tick's product rounds some 100 times, half an ulp of the pair's largest term each
    bound = ticks * 100 * 2.0 ** -24
    worst = (a - b).abs().amax(1) / a.abs().amax(1).clamp(min=1e-30)
    assert float(worst.max()) <= bound, float(worst.max())
