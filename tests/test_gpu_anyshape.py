"""Register-tile kernels for group sizes and head widths that are no powers of two (csrc/ncn_anyshape_kernels.h) against
the float64 oracle: every tile of theirs, heads that fill a tile and heads that end inside it, one and several row
lanes, group counts that leave the last wave tile partly empty."""
import pytest
import torch

from oracle import ncn_oracle as O

pytestmark = pytest.mark.gpu

# (n_cache, head width, heads, groups, batch): tile R x F, lanes per row x row lanes (as _tile says)
CASES = [
    (3, 3, 3, 7, 3),     # 3x3, 1x1, a wave tile of 64 groups, three heads
    (1, 5, 2, 70, 2),    # 2x5, 1x1, one row of two that exist
    (5, 1, 5, 1, 2),     # 5x3, 1x1, one feature of three; one group
    (6, 10, 1, 5, 4),    # 3x5, 2x2, one head
    (7, 40, 4, 3, 2),    # 2x5, 8x4, seven rows of eight
    (4, 20, 2, 9, 2),    # 2x5, 4x2, power-of-two rows, nothing padded
    (8, 12, 4, 4, 2),    # 4x3, 4x2
    (9, 7, 2, 3, 2),     # 3x4, 2x4, rows and features padded
    (10, 56, 2, 3, 2),   # 3x4, 16x4
    (13, 16, 2, 3, 2),   # 4x4, 4x4, power-of-two width, 13 rows of 16
    (16, 24, 3, 2, 2),   # 4x3, 8x4, three heads (a wave of the block works on the next tile)
    (20, 56, 1, 2, 2),   # 5x4, 16x4: only a tile of 20 elements holds the group
    (20, 64, 1, 2, 1),   # 5x4, 16x4 exactly
    (48, 12, 1, 2, 1),   # 3x3, 4x16: every lane of the wave in one group
    (2, 46, 1, 5, 2),    # 2x3, 16x1, 46 features of 48
    (2, 7, 3, 41, 2),    # 2x4, 2x1, 32 groups to a wave tile
    (25, 36, 1, 2, 1),   # 4x5, 8x8
    (33, 36, 1, 2, 1),   # 5x5, 8x8: the largest tile, rows and features padded
    (40, 40, 2, 1, 2),   # 5x5, 8x8 exactly
    (24, 64, 1, 2, 1),   # no tile: generic kernels
]
TOL = 1e-5


def _tile(n, ec):
    """The tile that any_tile() (csrc/ncn_launch.h) takes: (R, F, lanes per row, row lanes), or None."""
    best = None
    for r in range(2, 6):
        for f in range(3, 6):
            lf = max(0, (-(-ec // f) - 1).bit_length())
            lr = max(0, (-(-n // r) - 1).bit_length())
            if lf + lr > 6 or lf > 5:
                continue
            cost = ((20 * r * f + 4 * r * lf + 2 * f * lr + 10 * f) << (lf + lr)) * (4 if r * f > 16 else 1)
            if best is None or cost < best[0]:
                best = (cost, (r, f, 1 << lf, 1 << lr))
    return best and best[1]


def test_every_tile_has_a_case():
    tiles = [_tile(n, ec) for n, ec, _, _, _ in CASES]
    assert {t[:2] for t in tiles if t} == {(r, f) for r in range(2, 6) for f in range(3, 6)} and None in tiles


def _tolerance(n):
    """1e-5 up to 16 rows; beyond, the inversion amplifies float32 rounding by (1/m)^n: 1.2e-6 per unit, as measured for
    32 rows and used by the random-shape sweep (gradients)."""
    return max(TOL, 1.2e-6 * 0.9 ** -n)


@pytest.fixture(scope="module")
def M():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ncn_cuda_amd import ncn_cuda_module
    return ncn_cuda_module


def _inputs(case, L=1):
    n, ec, C, groups, batch = case
    return O.make_inputs(batch, n * groups, ec * C, L, n, seed=sum(case), xa_zero=False)


@pytest.mark.parametrize("act", [0, 2])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "n%d_e%d_C%d_g%d_b%d" % c)
def test_stage(M, case, act):
    n, ec, C, groups, batch = case
    x, xa, Ws, dy, dya = _inputs(case)
    d = torch.float64
    for stage in (0, 2):
        ref = O.net_autograd(x.to(d), xa.to(d), [Ws[0].to(d)], dy.to(d), dya.to(d), 0.9, n, C, activation=act, first_stage=stage)
        W = Ws[0].cuda()
        y, ya = M.forward_stages(x.cuda(), xa.cuda(), W, 0.9, act, n, C, stage, 1)
        assert O.rel_err(y, ref[0]) < TOL and O.rel_err(ya, ref[1]) < TOL
        xr, xar, dx, dxa, dW = M.backward_stages(y, ya, dy.cuda(), dya.cuda(), W, 0.9, act, n, C, stage, 1)
        tol = _tolerance(n)
        assert O.rel_err(dx, ref[2]) < tol and O.rel_err(dxa, ref[3]) < tol and O.rel_err(dW[0], ref[4][0]) < tol
        ix, ixa = M.inverse_stages(y, ya, W, 0.9, act, n, C, stage, 1)
        # the float32 outputs are undone: their rounding, amplified by (1/m)^n (6e-6 per unit, the sweep's bound)
        rtol = max(3e-5, 6e-6 * 0.9 ** -n)
        for a, b in ((xr, x), (xar, xa), (ix, x), (ixa, xa)):
            assert O.rel_err(a, b) < rtol


def _with(*shapes):
    return [c for c in CASES if c[:2] in shapes]


# the last one: the generic kernels, with their second launch for the groups that lengths cut and the rows passed through
@pytest.mark.parametrize("case", _with((3, 3), (7, 40), (20, 56), (2, 7), (25, 36), (33, 36), (24, 64)), ids=lambda c: "n%d_e%d_C%d_g%d_b%d" % c)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_table_and_lengths(M, case, dtype):
    """A random table, lengths that cut a group, end between groups, are zero and the whole of N."""
    n, ec, C, groups, batch = case
    batch, N = 4, n * groups
    x, xa, Ws, dy, dya = O.make_inputs(batch, N, ec * C, 1, n, seed=7, xa_zero=False, dtype=dtype)
    table = torch.randperm(N, generator=torch.Generator().manual_seed(3))
    lens = [0, N, n * (groups // 2), N - 1]
    d = torch.float64
    ref = O.net_autograd_indexed(x.to(d), xa.to(d), [Ws[0].to(d)], dy.to(d), dya.to(d), 0.9, n, C, [table], lens)
    kw = dict(group_index=table.to(torch.int32).cuda(), ctx_len=torch.tensor(lens, dtype=torch.int32).cuda())
    W = Ws[0].cuda()
    # bfloat16: what is stored is rounded once, by at most 2^-8 of a value; the float32 copies of y, ya are saved
    stored = lambda tol: tol if dtype == torch.float32 else max(tol, 2.0 ** -8)
    y, ya, sy, sya = M.forward_stages_saving(x.cuda(), xa.cuda(), W, 0.9, 0, n, C, 0, **kw)
    assert O.rel_err(y, ref[0]) < stored(TOL) and O.rel_err(ya, ref[1]) < stored(TOL)
    assert torch.equal(y[0].cpu(), x[0]) and torch.equal(ya[0].cpu(), xa[0])
    xr, xar, dx, dxa, dW = M.backward_stages(sy, sya, dy.cuda(), dya.cuda(), W, 0.9, 0, n, C, 0, 1, **kw)
    tol = _tolerance(n)
    assert dx.dtype == dtype and dW.dtype == torch.float32
    assert O.rel_err(dx, ref[2]) < stored(tol) and O.rel_err(dxa, ref[3]) < stored(tol) and O.rel_err(dW[0], ref[4][0]) < tol
    assert torch.equal(dx[0].cpu(), dy[0]) and torch.equal(xr[0].cpu(), x[0].float())
    # the saved outputs are undone: their float32 rounding, amplified by (1/m)^n
    ix, ixa = M.inverse_stages(sy, sya, W, 0.9, 0, n, C, 0, 1, **kw)
    rtol = max(3e-5, 6e-6 * 0.9 ** -n)
    for a, b in ((xr, x), (xar, xa), (ix, x), (ixa, xa)):
        assert O.rel_err(a, b) < rtol


@pytest.mark.parametrize("n,ec,C,groups", [(7, 24, 3, 5), (8, 20, 2, 17), (12, 56, 2, 3)])
def test_small_m_keeps_the_precision_of_the_plain_formulas(M, n, ec, C, groups):
    """Below m = 0.85 the generic kernels run these shapes: 1.2e-6 of a value per unit of (1/m)^n, the suite's figure for
    gradients, which the register tiles miss up to 17 times over at these scalars (measured: up to 0.77e-6 against 1.5e-6 to
    21e-6)."""
    alpha, m, d = 0.1, 0.7, torch.float64
    for seed in range(3):
        x, xa, Ws, dy, dya = O.make_inputs(2, n * groups, ec * C, 1, n, seed=seed, xa_zero=False)
        ref = O.net_autograd(x.to(d), xa.to(d), [Ws[0].to(d)], dy.to(d), dya.to(d), alpha, n, C, m=m)
        W = Ws[0].cuda()
        y, ya = M.forward_stages(x.cuda(), xa.cuda(), W, alpha, 0, n, C, 0, 1, m=m)
        _, _, dx, dxa, dW = M.backward_stages(y, ya, dy.cuda(), dya.cuda(), W, alpha, 0, n, C, 0, 1, m=m)
        for got, want in ((dx, ref[2]), (dxa, ref[3]), (dW[0], ref[4][0])):
            assert O.rel_err(got, want) < 1.2e-6 * m ** -n


@pytest.mark.parametrize("value", [float("inf"), -float("inf")])
@pytest.mark.parametrize("n,ec,C", [(5, 7, 2), (3, 7, 3), (12, 22, 2), (4, 18, 2)])   # heads that end inside their tile
def test_infinite_inputs(M, n, ec, C, value):
    """An infinite input makes row sums infinite, which saturate tanh: where the oracle's results are finite so are the
    kernel's, although the features that pad a tile see the same sums (zero times them would be NaN)."""
    d, group = torch.float64, slice(0, n)   # stage 0: the group of the infinite value
    for seed in range(40):   # most weights make the sum NaN at once: inf - inf
        x, xa, Ws, _, _ = O.make_inputs(2, n * 4, ec * C, 1, n, seed=seed, xa_zero=False)
        x[:, 2, 1] = value
        ref = O.net_forward(x.to(d), xa.to(d), [Ws[0].to(d)], 0.9, n, C)
        finite = torch.isfinite(ref[1][:, group, :ec])
        if finite.float().mean() > 0.5 and not finite.all():
            break
    assert finite.any() and not finite.all()
    W = Ws[0].cuda()
    y, ya = M.forward_stages(x.cuda(), xa.cuda(), W, 0.9, 0, n, C, 0, 1)
    for a, b in ((y, ref[0]), (ya, ref[1])):
        a, b = a.cpu()[:, group, :ec].to(d), b[:, group, :ec]
        assert torch.equal(torch.isfinite(a), torch.isfinite(b))
        ok = torch.isfinite(b)
        assert (a - b)[ok].norm() < TOL * b[ok].norm()


@pytest.mark.parametrize("case", [CASES[3], CASES[4]], ids=lambda c: "n%d_e%d_C%d_g%d_b%d" % c)
def test_bfloat16(M, case):
    n, ec, C, groups, batch = case
    x, xa, Ws, dy, dya = (t.bfloat16() if isinstance(t, torch.Tensor) else t for t in _inputs(case))
    d = torch.float64
    ref = O.net_autograd(x.to(d), xa.to(d), [Ws[0].to(d)], dy.to(d), dya.to(d), 0.9, n, C)
    W = Ws[0].cuda()
    y, ya, sy, sya = M.forward_stages_saving(x.cuda(), xa.cuda(), W, 0.9, 0, n, C, 0)
    _, _, dx, dxa, dW = M.backward_stages(sy, sya, dy.cuda(), dya.cuda(), W, 0.9, 0, n, C, 0, 1, want_inputs=False)
    for got, want in ((y, ref[0]), (ya, ref[1]), (dx, ref[2]), (dxa, ref[3]), (dW[0], ref[4][0])):
        assert O.rel_err(got, want) < 2e-2


@pytest.mark.parametrize("n,ec,C", [(3, 3, 1), (5, 7, 2), (2, 10, 1)])   # heads that end with a lane, inside one, two lanes of five
def test_more_tiles_than_partial_rows(n, ec, C):
    """The backward then loops over tiles; each half of the batch has a wave for every tile."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ncn_cuda_amd import ncn_cuda_module as M
    batch, E = 16384 + 200, ec * C
    gen = torch.Generator(device="cuda").manual_seed(n)
    x, xa, dy, dya = (torch.randn(batch, n, E, generator=gen, device="cuda") for _ in range(4))
    W = torch.randn(2 * E, generator=gen, device="cuda") / n ** 0.5
    y, ya = M.forward_stages(x, xa, W, 0.9, 0, n, C, 0, 1)
    _, _, dx, dxa, dW = M.backward_stages(y, ya, dy, dya, W, 0.9, 0, n, C, 0, 1, want_inputs=False)
    halves = [M.backward_stages(*(t[s].contiguous() for t in (y, ya, dy, dya)), W, 0.9, 0, n, C, 0, 1, want_inputs=False)
              for s in (slice(0, batch // 2), slice(batch // 2, batch))]
    # the builds with and without the loop round ku rh Wi' differently, by a few units in the last place
    assert O.rel_err(dx, torch.cat([h[2] for h in halves])) < 1e-6 and O.rel_err(dxa, torch.cat([h[3] for h in halves])) < 1e-6
    want = sum(h[4].double() for h in halves)
    assert ((dW.double() - want).norm() / want.norm()) < 1e-5    # sums of some 10^5 products in float32, in other orders
