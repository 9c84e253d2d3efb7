"""The air rollout over arrays by car, with every tick's state kept, against
the one over arrays by word with checkpoints: the same bits, at tick counts
around the group of loads and the checkpoint distance, for one car, a ragged
wave and several, for inputs that are views at odd offsets or transposed, and
when the caller's tensors change between forward and backward.  And the entry
points by car against those by word at every kind of checkpoint distance (every
tick kept; segments of one group of loads, ragged and whole), with and without
the optional outputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _problem(n, ticks, seed):
    g = torch.Generator().manual_seed(seed)
    s0 = torch.cat([torch.randn(n, 3, generator=g) * 800, torch.nn.functional.normalize(torch.randn(n, 4, generator=g), dim=-1),
                    torch.randn(n, 3, generator=g) * 900, torch.randn(n, 3, generator=g) * 3], -1)
    ctrl = torch.cat([torch.tanh(torch.randn(ticks, n, 3, generator=g)), torch.rand(ticks, n, 1, generator=g)], -1)
    tgt = torch.cat([torch.nn.functional.normalize(torch.randn(n, 4, generator=g), dim=-1),
                     torch.randn(n, 3, generator=g) * 500], -1)
    return s0.cuda(), ctrl.cuda(), tgt.cuda()


def _grads(fn, s0, ctrl, tgt, change=False):
    s0, ctrl = s0.detach().requires_grad_(True), ctrl.detach().requires_grad_(True)
    loss, final = fn(s0, ctrl, tgt)
    if change:
        with torch.no_grad():
            ctrl.zero_()
            tgt.zero_()
    ds0, dctrl = torch.autograd.grad((loss * torch.arange(1, loss.numel() + 1, device="cuda")).sum(), [s0, ctrl])
    return [x.contiguous() for x in (loss, final, ds0, dctrl)]


@pytest.mark.parametrize("n,ticks", [(1, 1), (1, 4), (65, 3), (64, 5), (257, 17), (130, 33)])
def test_by_car_equals_by_word(n, ticks):
    from rocketsim_amd.adjoint import AirRollout, air_rollout
    s0, ctrl, tgt = _problem(n, ticks, n + ticks)
    want = _grads(lambda *a: AirRollout.apply(*a), s0, ctrl, tgt)

    def odd(x):     # the same values at an address off 16 bytes
        return torch.cat([torch.zeros(1, device="cuda"), x.flatten()])[1:].view(x.shape)

    def turned(x):  # ... with the last two dimensions' strides exchanged
        return x.transpose(-1, -2).contiguous().transpose(-1, -2)

    for make in (lambda x: x.clone(), odd, turned):
        for got, w in zip(_grads(air_rollout, make(s0), make(ctrl), make(tgt)), want):
            assert torch.equal(got, w)
    for got, w in zip(_grads(air_rollout, s0.clone(), ctrl.clone(), tgt.clone(), change=True), want):
        assert torch.equal(got, w)


@pytest.mark.parametrize("every", [1, 3, 16, 32])
@pytest.mark.parametrize("n,ticks", [(1, 1), (65, 31), (130, 32), (64, 33), (257, 96)])
def test_entry_points_by_car_equal_those_by_word(n, ticks, every):
    from rocketsim_amd import native
    L = native.lib()
    s0, ctrl, tgt = _problem(n, ticks, 7 * n + ticks)
    by_word = [s0.t().contiguous(), ctrl.permute(0, 2, 1).contiguous(), tgt.t().contiguous()]
    dl = torch.linspace(-1, 2, n, device="cuda")
    new = lambda *shape: torch.full(shape, float("nan"), device="cuda")     # noqa: E731
    words = ((ticks + every - 1) // every) * 13 * n
    check, p = native.check, lambda x: x.data_ptr()                         # noqa: E731

    final, loss, ckpt, dc, ds = new(13, n), new(n), new(words), new(ticks, 4, n), new(13, n)
    check(L.rsg_air_rollout(n, ticks, every, 120.0, *map(p, by_word), p(final), p(loss), p(ckpt), None))
    check(L.rsg_air_rollout_backward(n, ticks, every, 120.0, p(by_word[1]), p(by_word[2]), p(ckpt), p(dl), p(dc), p(ds),
                                     None))
    want = [final.t(), loss, ckpt, dc.permute(0, 2, 1), ds.t()]

    final, loss, ckpt, dc, ds = new(n, 13), new(n), new(words), new(ticks, n, 4), new(n, 13)
    kept, kept_target = new(ticks, n, 4), new(n, 7)
    check(L.rsg_air_rollout_rows(n, ticks, every, 120.0, p(s0), p(ctrl), p(tgt), p(final), p(loss), p(ckpt), p(kept),
                                 p(kept_target), None))
    check(L.rsg_air_rollout_rows_backward(n, ticks, every, 120.0, p(kept), p(kept_target), p(ckpt), p(dl), p(dc), p(ds),
                                          None))
    torch.cuda.synchronize()
    for got, w in zip([final, loss, ckpt, dc, ds, kept, kept_target], want + [ctrl, tgt]):
        assert torch.equal(got, w)
    # outputs left out
    final2, loss2, dc2 = new(n, 13), new(n), new(ticks, n, 4)
    check(L.rsg_air_rollout_rows(n, ticks, every, 120.0, p(s0), p(ctrl), p(tgt), p(final2), p(loss2), None, None, None,
                                 None))
    check(L.rsg_air_rollout_rows_backward(n, ticks, every, 120.0, p(ctrl), p(tgt), p(ckpt), p(dl), p(dc2), None, None))
    torch.cuda.synchronize()
    for got, w in ((final2, final), (loss2, loss), (dc2, dc)):
        assert torch.equal(got, w)
