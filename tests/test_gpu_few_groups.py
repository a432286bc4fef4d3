"""The one-stage kernels for launches with few groups (ncn_split_kernels.h) against the float64 oracle: a group over one to
eight waves, several groups to a wave, a last wave tile and a last workgroup that are partly empty, both storage types, with
and without reconstructed inputs; and the register tiles (ncn_stage_kernels.h), which take over past their largest launch, in every
shape that they are built for, on sizes just above it."""
import ctypes

import pytest
import torch

from conftest import kernels_of
from oracle import ncn_oracle as O

pytestmark = pytest.mark.gpu

# n, head width, heads, groups, batch: waves per group 1, 1, 1, 2, 2, 4, 4, 8, 8; workgroups of 4 or 8 waves
SHAPES = [(2, 4, 3, 3, 1), (4, 8, 1, 19, 2), (8, 32, 3, 1, 1), (8, 64, 3, 5, 1), (16, 32, 3, 3, 3), (32, 32, 1, 7, 1),
          (8, 128, 2, 3, 1), (64, 32, 1, 2, 3), (16, 128, 2, 3, 1)]
# above 2^20 (groups of 8 rows and more) or 2^18 elements, an odd number of groups
ABOVE = [(8, 32, 4, 1025, 1), (16, 32, 4, 171, 3), (32, 32, 3, 115, 3), (4, 32, 4, 171, 3), (2, 8, 3, 1825, 3)]
# every shape of the register tiles (NCN_FOR_EACH_FAST_CONFIG), above the largest launch of the others (split_max_elements): an odd
# number of groups, so that the last wave tile of a batch entry is partly empty wherever it holds several
TILES = [(n, ec, 2, ((1 << (20 if n >= 8 else 18)) // (n * ec * 6) + 1) | 1, 3) for ec in (4, 8, 16, 32, 64, 128)
         for n in (2, 4, 8, 16, 32, 64) if n * ec <= 2048]


@pytest.fixture(scope="module")
def M():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ncn_cuda_amd import ncn_cuda_module
    return ncn_cuda_module


def run(kind, call):
    """call()'s result, and that its stage ran on the kernels of this kind: "split" (few groups) or "stage" (register tiles)."""
    result, ran = kernels_of(call)
    assert {name.split("_")[0] for name in ran} - {"reduce"} == {kind}, ran
    return result


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("shape", SHAPES + ABOVE + TILES, ids=lambda s: "n%d_e%d_C%d_g%d_b%d" % s)
def test_one_stage(M, shape, dtype):
    n, ec, C, groups, batch = shape
    N, stage, kind = n * groups, 2, "split" if shape in SHAPES else "stage"
    x, xa, Ws, dy, dya = O.make_inputs(batch, N, ec * C, 1, n, seed=sum(shape), xa_zero=False)
    x, xa, dy, dya = (t.to(dtype) for t in (x, xa, dy, dya))
    if shape in TILES:   # the oracle's float64 on the GPU
        x, xa, dy, dya, Ws = *(t.cuda() for t in (x, xa, dy, dya)), [Ws[0].cuda()]
    d = torch.float64
    ref = O.net_autograd(x.to(d), xa.to(d), [Ws[0].to(d)], dy.to(d), dya.to(d), 0.9, n, C, first_stage=stage)
    x, xa, dy, dya, W = (t.cuda() for t in (x, xa, dy, dya, Ws[0]))
    y, ya, sy, sya = run(kind, lambda: M.forward_stages_saving(x, xa, W, 0.9, 0, n, C, stage))
    _, _, dx, dxa, dW = run(kind, lambda: M.backward_stages(sy, sya, dy, dya, W, 0.9, 0, n, C, stage, 1, want_inputs=False, grad_dtype=dtype))
    # the tolerances of test_gpu_parity (3e-6 of a value, amplified by 1/m at every step undone, for 32 rows and more) and, for 64
    # rows, of test_gpu_random_shapes (16e-6); two bfloat16 planes keep 2^-18 of a saved value where float32 keeps 2^-24; a
    # bfloat16 result is rounded by at most 2^-8
    bf16 = dtype == torch.bfloat16
    unit = 1.2e-6 if n < 32 else 3e-6 if n < 64 or shape in SHAPES else 16e-6
    tol = max(1e-5, unit * (64 if bf16 else 1) * 0.9 ** -n)
    if n <= 32 or not bf16:   # (64 steps amplify two planes past use)
        for got, want in zip((y, ya, dx, dxa), ref[:4]):
            assert got.dtype == dtype and O.rel_err(got, want) < (max(tol, 2.0 ** -8) if bf16 else tol)
        assert O.rel_err(dW[0], ref[4][0]) < tol
    # float32 outputs, from which the inputs come back
    y32, ya32 = M.forward_stages(x, xa, W, 0.9, 0, n, C, stage, 1, out_dtype=torch.float32)
    assert O.rel_err(y32, ref[0]) < 1e-5 and O.rel_err(ya32, ref[1]) < 1e-5
    back = 12e-6 * 0.9 ** -n   # test_gpu_parity's bound on reconstructed inputs
    if n < 64:
        ix, ixa = run(kind, lambda: M.inverse_stages(y32, ya32, W, 0.9, 0, n, C, stage, 1))
        rx, rxa, dx2, dxa2, dW2 = M.backward_stages(y32, ya32, dy.float(), None, W, 0.9, 0, n, C, stage, 1, want_inputs=True)
        for got, want in ((ix, x), (ixa, xa), (rx, x), (rxa, xa)):
            assert O.rel_err(got, want) < back
        at = ref[0].device
        ref0 = O.net_autograd(x.to(at, d), xa.to(at, d), [Ws[0].to(d)], dy.to(at, d), torch.zeros_like(ref[0]), 0.9, n, C, first_stage=stage)
        f32 = max(1e-5, (3e-6 if n >= 32 else 1.2e-6) * 0.9 ** -n)
        assert O.rel_err(dx2, ref0[2]) < f32 and O.rel_err(dxa2, ref0[3]) < f32 and O.rel_err(dW2[0], ref0[4][0]) < f32


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("shape", [(4, 8, 1, 19, 3), (8, 32, 3, 3, 3), (16, 32, 3, 3, 3), (32, 32, 1, 7, 3), (32, 64, 2, 3, 3)] +
                         [s for s in TILES if s[0] < 64], ids=lambda s: "n%d_e%d_C%d_g%d_b%d" % s)
def test_table_and_lengths(M, shape, dtype):
    n, ec, C, groups, batch = shape
    N, d, kind = n * groups, torch.float64, "stage" if shape in TILES else "split"
    x, xa, Ws, dy, dya = O.make_inputs(batch, N, ec * C, 1, n, seed=sum(shape), xa_zero=False)
    x, xa, dy, dya = (t.to(dtype) for t in (x, xa, dy, dya))
    table = torch.randperm(N, generator=torch.Generator().manual_seed(2))
    lens = [N, n * (groups // 2) + n // 2, 0]   # everything, a group that the length cuts, nothing
    if kind == "stage":
        x, xa, dy, dya, Ws, table = *(t.cuda() for t in (x, xa, dy, dya)), [Ws[0].cuda()], table.cuda()
    ref = O.net_autograd_indexed(x.to(d), xa.to(d), [Ws[0].to(d)], dy.to(d), dya.to(d), 0.9, n, C, [table], lens)
    kw = dict(group_index=table.to(torch.int32).cuda(), ctx_len=torch.tensor(lens, dtype=torch.int32).cuda())
    x, xa, dy, dya, W = (t.cuda() for t in (x, xa, dy, dya, Ws[0]))
    y, ya, sy, sya = run(kind, lambda: M.forward_stages_saving(x, xa, W, 0.9, 0, n, C, 2, **kw))
    _, _, dx, dxa, dW = run(kind, lambda: M.backward_stages(sy, sya, dy, dya, W, 0.9, 0, n, C, 2, 1, want_inputs=False, grad_dtype=dtype, **kw))
    bf16 = dtype == torch.bfloat16
    tol = max(1e-5, (3e-6 if n >= 32 else 1.2e-6) * (64 if bf16 else 1) * 0.9 ** -n)   # as above
    for got, want in zip((y, ya, dx, dxa), ref[:4]):
        assert O.rel_err(got, want) < (max(tol, 2.0 ** -8) if bf16 else tol)
    assert O.rel_err(dW[0], ref[4][0]) < tol
    assert torch.equal(y[2], x[2]) and torch.equal(ya[2], xa[2]) and torch.equal(dx[2], dy[2]) and torch.equal(dxa[2], dya[2])
    y32, ya32 = M.forward_stages(x, xa, W, 0.9, 0, n, C, 2, 1, out_dtype=torch.float32, **kw)
    ix, ixa = run(kind, lambda: M.inverse_stages(y32, ya32, W, 0.9, 0, n, C, 2, 1, **kw))
    rx, rxa, _, _, _ = M.backward_stages(y32, ya32, dy.float(), None, W, 0.9, 0, n, C, 2, 1, want_inputs=True, **kw)
    for got, want in ((ix, x), (ixa, xa), (rx, x), (rxa, xa)):
        assert O.rel_err(got, want) < 12e-6 * 0.9 ** -n


@pytest.mark.parametrize("n,ec,forward,backward", [(8, 16, "split", "stage"), (64, 8, "stage", "stage"), (32, 4, "split", "stage"),
                                                   (16, 32, "split", "split"), (2, 32, "stage", "stage"), (2, 64, "split", "split")])
def test_which_kernels_take_a_launch(M, n, ec, forward, backward):
    """The largest launches of the split kernels depend on direction and width: a million elements for groups of 8 rows and more,
    a quarter of that for groups of two; tables leave the earlier lines aside."""
    elements = 1 << (20 if n >= 8 else 18)
    C, batch = 2, 2
    N = elements // (batch * C * ec)
    x = torch.randn(batch, N, C * ec, device="cuda")
    W = torch.randn(2 * C * ec, device="cuda") / n ** 0.5
    y, ya = run(forward, lambda: M.forward_stages(x, x, W, 0.9, 0, n, C, 1, 1))
    run(forward, lambda: M.inverse_stages(y, ya, W, 0.9, 0, n, C, 1, 1))
    run(backward, lambda: M.backward_stages(y, ya, x, x, W, 0.9, 0, n, C, 1, 1, want_inputs=False))
    kw = dict(group_index=torch.arange(N, dtype=torch.int32, device="cuda"))
    kind = "split" if n >= 8 or ec >= 64 else "stage"
    run(kind, lambda: M.forward_stages(x, x, W, 0.9, 0, n, C, 0, 1, **kw))
    run(kind, lambda: M.backward_stages(y, ya, x, x, W, 0.9, 0, n, C, 0, 1, want_inputs=False, **kw))


@pytest.mark.parametrize("lengths", [False, True], ids=["whole", "lengths"])
def test_more_wave_tiles_than_partial_rows(M, lengths):
    """A wave tile per batch entry and more of them than dW rows: the register tiles, which loop, take the launch."""
    batch, n, E = 16384 + 16, 8, 4
    x, xa, Ws, dy, dya = (t.cuda() if isinstance(t, torch.Tensor) else [t[0].cuda()] for t in O.make_inputs(batch, n, E, 1, n, seed=9, xa_zero=False))
    d, W = torch.float64, Ws[0]
    kw = {}
    if lengths:
        lens = torch.arange(batch, dtype=torch.int32, device="cuda") % (n + 1)
        kw = dict(ctx_len=lens)
        refs = []
        for k in (0, 3, n):   # some entries of each length
            some = (lens == k).nonzero().flatten()[:40]
            pick = lambda *ts: [t[some].to(d) for t in ts]
            refs.append((some, O.net_autograd_indexed(*pick(x, xa), [W.to(d)], *pick(dy, dya), 0.9, n, 1, [torch.arange(n, device="cuda")], [k] * len(some))))
    else:
        refs = [(slice(None), O.net_autograd(x.to(d), xa.to(d), [W.to(d)], dy.to(d), dya.to(d), 0.9, n, 1))]
    y, ya = run("stage", lambda: M.forward_stages(x, xa, W, 0.9, 0, n, 1, 0, 1, **kw))
    _, _, dx, dxa, dW = run("stage", lambda: M.backward_stages(y, ya, dy, dya, W, 0.9, 0, n, 1, 0, 1, want_inputs=False, **kw))
    for rows, ref in refs:
        for got, want in zip((y, ya, dx, dxa), ref[:4]):
            assert O.rel_err(got[rows], want) < 1e-5
    half = batch // 2   # these halves have a dW row for every wave tile
    cut = lambda s: dict(ctx_len=lens[s].contiguous()) if lengths else {}
    parts = [run("split", lambda: M.backward_stages(*(t[s].contiguous() for t in (y, ya, dy, dya)), W, 0.9, 0, n, 1, 0, 1, want_inputs=False,
                                                    **cut(s)))[4] for s in (slice(0, half), slice(half, batch))]
    assert O.rel_err(dW, parts[0].double() + parts[1].double()) < 1e-5
    if not lengths:
        assert O.rel_err(dW[0], refs[0][1][4][0]) < 1e-5


def test_more_wave_tiles_than_rows_of_the_library_scratch(M):
    """ncn_backward_static has 4096 dW rows: past as many wave tiles the register tiles take the launch, as ncn_backward's do at 16384."""
    from ncn_cuda_amd import _lib
    lib = _lib.load()
    n, E = 8, 4
    for batch, kind in ((4096, "split"), (4097, "stage")):
        x, xa, Ws, dy, dya = (t.cuda() if isinstance(t, torch.Tensor) else [t[0].cuda()] for t in O.make_inputs(batch, n, E, 1, n, seed=batch))
        W = Ws[0]
        y, ya = M.forward_stages(x, xa, W, 0.9, 0, n, 1, 0, 1)
        want = run("split", lambda: M.backward_stages(y, ya, dy, dya, W, 0.9, 0, n, 1, 0, 1, want_inputs=False))[2:]
        dx, dxa, dW = torch.empty_like(x), torch.empty_like(x), torch.empty(1, 2 * E, device="cuda")
        shape = _lib.NcnShape(batch, n, E, 1, n)
        rc = run(kind, lambda: lib.ncn_backward_static(y.data_ptr(), ya.data_ptr(), 0, dy.data_ptr(), dya.data_ptr(), 0, dx.data_ptr(), dxa.data_ptr(),
                                                       0, None, None, W.data_ptr(), dW.data_ptr(), ctypes.byref(shape), 0, 1, 0.9, 0.9, 0,
                                                       torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        for a, b in zip((dx, dxa, dW), want):
            assert O.rel_err(a, b) < 1e-5


def test_launches_repeat_bit_for_bit(M):
    n, C, E, N = 32, 4, 128, 256
    x, xa, Ws, dy, dya = (t.cuda() if isinstance(t, torch.Tensor) else [t[0].cuda()] for t in O.make_inputs(4, N, E, 1, n, seed=3))
    first = None
    for _ in range(3):
        y, ya = M.forward_stages(x, xa, Ws[0], 0.9, 0, n, C, 1, 1)
        _, _, dx, dxa, dW = M.backward_stages(y, ya, dy, dya, Ws[0], 0.9, 0, n, C, 1, 1, want_inputs=False)
        got = (y, ya, dx, dxa, dW)
        assert first is None or all(torch.equal(a, b) for a, b in zip(got, first))
        first = got
