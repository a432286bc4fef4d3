"""Halo passes over sheared windows (trained stacks and the inverse with scratch) against the float64 oracle: strides that fall as
well as rise around the ring, ranges that do not start at stage 0, last windows of a few groups, every head width."""
import pytest
import torch

from oracle import ncn_oracle as O

pytestmark = pytest.mark.gpu

# batch, groups, E, heads, n_cache, first stage, stages
CASES = [
    (2, 514, 64, 2, 2, 0, 9),        # 2 * 257 groups: strides past 2 wrap to odd multiples of 2, up and down the ring
    (1, 4096, 32, 1, 2, 3, 8),       # from stride 4 on, then closed rings
    (2, 260, 64, 2, 2, 0, 7),        # one group more than a window owns, and a few
    (1, 1030, 16, 2, 2, 0, 8),       # heads of 8 features
    (1, 300, 256, 2, 2, 1, 6),       # heads of 128
    (2, 130, 64, 2, 4, 0, 6),        # 2 * 65 groups of four rows
    (1, 512, 128, 4, 4, 0, 6),
    (2, 66, 64, 2, 4, 0, 5),         # a ring little longer than a window
    (1, 320, 64, 4, 4, 2, 5),        # 5 * 64 groups, from stride 2 on
    (1, 600, 16, 2, 4, 0, 6),        # heads of 8
    (1, 70, 128, 1, 4, 0, 5),        # heads of 128
    (1, 514, 32, 32, 2, 0, 7),       # heads of one feature
    (1, 130, 24, 24, 4, 0, 6),
]


@pytest.mark.parametrize("case", [(64, 32, 64, 2, 4, 0, 6), (64, 32, 32, 32, 4, 1, 6), (64, 64, 64, 2, 2, 0, 7), (64, 64, 32, 32, 2, 2, 7)],
                         ids=lambda c: "_".join(map(str, c)))
def test_many_steps_are_undone_without_drift(case):
    """What the passes reconstruct is off by rounding errors of either sign, not by that of 1/m once for every step.  m is one whose 1/m
    is 5.9e-8 off in float32: 24 or 14 steps would drift by 1.4e-6 or 8e-7 (less what xa makes up for; 3.7e-7 to 9.8e-7 measured).  The
    other constants are off once, by half a unit each (6e-8), four of them in a step: 2.4e-7."""
    from ncn_cuda_amd import ncn_cuda_module as M
    batch, groups, E, C, n, first, L = case
    x, xa, Ws, dy, dya = O.make_inputs(batch, n * groups, E, L, n, seed=sum(case), xa_zero=False)
    m = 0.900225818157196   # a float32
    d = torch.float64
    y, ya = O.net_forward(x.to(d).cuda(), xa.to(d).cuda(), [w.to(d).cuda() for w in Ws], 0.9, n, C, m=m, first_stage=first)
    W = torch.stack([w.reshape(-1) for w in Ws]).cuda()
    back = M.backward_stages(y.float(), ya.float(), dy.cuda(), dya.cuda(), W, 0.9, 0, n, C, first, L, m=m)
    for got, want in ((back[0].cpu().to(d), x.to(d)), (back[1].cpu().to(d), xa.to(d))):
        drift = abs(float(((got - want) * want).sum() / (want * want).sum()))
        assert drift < 2.4e-7


@pytest.mark.parametrize("case", CASES, ids=lambda c: "_".join(map(str, c)))
def test_stack_and_inverse(case):
    from ncn_cuda_amd import ncn_cuda_module as M
    batch, groups, E, C, n, first, L = case
    N, max_range = n * groups, min(L, 26 // n)
    x, xa, Ws, dy, dya = O.make_inputs(batch, N, E, L, n, seed=sum(case), xa_zero=False)
    d = torch.float64
    ref = O.net_autograd(x.to(d), xa.to(d), [w.to(d) for w in Ws], dy.to(d), dya.to(d), 0.9, n, C, first_stage=first)
    W = torch.stack([w.reshape(-1) for w in Ws]).cuda()
    # 1.2e-6 per unit of rounding (the figure of the other stack tests), amplified by 1/m at each step that is undone
    tol = 1.2e-6 * 0.9 ** -(n * max_range)
    plan, y, ya, saves = M.stack_forward(x.cuda(), xa.cuda(), W, 0.9, 0, n, C, first, L, max_range, 8 * x.numel() * L)
    dx, dxa, dW = M.stack_backward(plan, y, ya, saves, dy.cuda(), dya.cuda(), W)
    for name, got, want in (("y", y, ref[0]), ("ya", ya, ref[1]), ("dx", dx, ref[2]), ("dxa", dxa, ref[3]),
                            *(("dW%d" % l, dW[l], ref[4][l].reshape(-1)) for l in range(L))):
        assert O.rel_err(got, want) < tol, name
    rx, rxa = M.inverse_stages(y, ya, W, 0.9, 0, n, C, first, L)
    tol = 1.2e-6 * 0.9 ** -(n * L)
    assert O.rel_err(rx, x) < tol and O.rel_err(rxa, xa) < tol
