"""Halo passes over sheared windows (trained stacks and the inverse with scratch) against the float64 oracle: strides that fall as
well as rise around the ring, ranges that do not start at stage 0, last windows of a few groups, every head width, both types."""
import ctypes

import pytest
import torch

from oracle import ncn_oracle as O

pytestmark = pytest.mark.gpu

# batch, groups, E, heads, n_cache, first stage, stages
CASES = [
    (2, 514, 64, 2, 2, 0, 9),        # 2 * 257 groups: rings of an odd length
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
    (1, 514, 24, 24, 4, 0, 6),
    # from where the strides pass the number of groups and fall
    (2, 514, 64, 2, 2, 10, 5),
    (1, 514, 32, 32, 2, 9, 6),
    (2, 130, 64, 2, 4, 8, 4),
    (1, 130, 64, 64, 4, 8, 4),
    (2, 130, 128, 2, 4, 0, 6),       # heads of 64
    (1, 320, 64, 1, 4, 1, 5),
    (2, 514, 128, 2, 2, 0, 9),
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


def halos(case, max_range, act=0):
    """Halo passes of the inverse (with scratch for two arrays), and of the stack in either direction."""
    from ncn_cuda_amd import _lib
    batch, groups, E, C, n, first, L = case
    shape, buf = _lib.NcnShape(batch, n * groups, E, C, n), (ctypes.c_int32 * 640)()
    found = []
    for backward, longest in ((0, 0), (0, max_range), (1, max_range)):
        k = _lib.load().ncn_plan_sheared_passes(ctypes.byref(shape), first, L, act, backward, longest, L, buf, 64)
        found.append(sum(buf[10 * j + 2] == 1 for j in range(k)))
    return found


def inverse_with_scratch(y, ya, W, act, case):
    from ncn_cuda_amd import _lib
    batch, groups, E, C, n, first, L = case
    x, xa, ws = torch.empty_like(y), torch.empty_like(ya), torch.empty(2 * (y.numel() + 64), device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    shape = _lib.NcnShape(batch, n * groups, E, C, n)
    rc = _lib.load().ncn_inverse_ws(p(y), p(ya), 0, p(x), p(xa), 0, p(W), p(ws), ctypes.c_size_t(ws.numel() * 4), ctypes.byref(shape), first, L,
                                    0.9, 0.9, act, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    return x, xa


def check(case, act, dtype):
    from ncn_cuda_amd import ncn_cuda_module as M
    batch, groups, E, C, n, first, L = case
    N, max_range = n * groups, min(L, 26 // n)
    assert min(halos(case, max_range, act)) >= 1
    x, xa, Ws, dy, dya = O.make_inputs(batch, N, E, L, n, seed=sum(case), xa_zero=False, dtype=dtype)
    d, f32 = torch.float64, dtype == torch.float32
    ref = O.net_autograd(x.to(d), xa.to(d), [w.to(d) for w in Ws], dy.to(d), dya.to(d), 0.9, n, C, activation=act, first_stage=first)
    W = torch.stack([w.reshape(-1) for w in Ws]).cuda()
    # 1.2e-6 per unit of rounding (the figure of the other stack tests), amplified by 1/m at each step that is undone; bfloat16
    # results are rounded once, by at most half a unit of their eight significant bits
    tol = 1.2e-6 * 0.9 ** -(n * max_range) if f32 else 2.0 ** -8
    plan, y, ya, saves = M.stack_forward(x.cuda(), xa.cuda(), W, 0.9, act, n, C, first, L, max_range, 8 * x.numel() * L)
    dx, dxa, dW = M.stack_backward(plan, *((y, ya) if f32 else (None, None)), saves, dy.cuda(), dya.cuda(), W)
    for name, got, want in (("y", y, ref[0]), ("ya", ya, ref[1]), ("dx", dx, ref[2]), ("dxa", dxa, ref[3]),
                            *(("dW%d" % l, dW[l], ref[4][l].reshape(-1)) for l in range(L))):
        assert got.dtype == dtype and O.rel_err(got, want) < tol, name
    if f32:
        tol = 1.2e-6 * 0.9 ** -(n * L)
        for rx, rxa in (M.inverse_stages(y, ya, W, 0.9, act, n, C, first, L), inverse_with_scratch(y, ya, W, act, case)):
            assert O.rel_err(rx, x) < tol and O.rel_err(rxa, xa) < tol


@pytest.mark.parametrize("case", CASES, ids=lambda c: "_".join(map(str, c)))
def test_stack_and_inverse(case):
    check(case, 0, torch.float32)


@pytest.mark.parametrize("act,dtype", [(2, torch.float32), (-1, torch.float32), (0, torch.bfloat16), (2, torch.bfloat16)],
                         ids=["sigmoid", "linear", "bf16", "sigmoid_bf16"])
@pytest.mark.parametrize("case", [(2, 514, 128, 2, 2, 0, 9), (2, 514, 64, 2, 2, 10, 5), (2, 130, 128, 2, 4, 0, 6), (2, 130, 64, 2, 4, 8, 4), (1, 130, 64, 64, 4, 0, 6)],
                         ids=lambda c: "_".join(map(str, c)))
def test_other_activations_and_bfloat16(case, act, dtype):
    check(case, act, dtype)
