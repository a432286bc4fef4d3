"""The one-stage kernels for launches with few groups (ncn_split_kernels.h) against the float64 oracle: a group over one to
eight waves, several groups to a wave, a last wave tile and a last workgroup that are partly empty, both storage types, with
and without reconstructed inputs; and the register tiles, which take over past their largest launch, on sizes just above it."""
import pytest
import torch

from oracle import ncn_oracle as O

pytestmark = pytest.mark.gpu

# n, head width, heads, groups, batch: waves per group 1, 1, 1, 2, 2, 4, 4, 8, 8; workgroups of 4 or 8 waves
SHAPES = [(2, 4, 3, 3, 1), (4, 8, 1, 19, 2), (8, 32, 3, 1, 1), (8, 64, 3, 5, 1), (16, 32, 3, 3, 3), (32, 32, 1, 7, 1),
          (8, 128, 2, 3, 1), (64, 32, 1, 2, 3), (16, 128, 2, 3, 1)]
# above 2^20 (groups of 8 rows and more) or 2^18 elements, an odd number of groups
ABOVE = [(8, 32, 4, 1025, 1), (16, 32, 4, 171, 3), (32, 32, 3, 115, 3), (4, 32, 4, 171, 3), (2, 8, 3, 1825, 3)]


@pytest.fixture(scope="module")
def M():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ncn_cuda_amd import ncn_cuda_module
    return ncn_cuda_module


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("shape", SHAPES + ABOVE, ids=lambda s: "n%d_e%d_C%d_g%d_b%d" % s)
def test_one_stage(M, shape, dtype):
    n, ec, C, groups, batch = shape
    N, stage = n * groups, 2
    x, xa, Ws, dy, dya = O.make_inputs(batch, N, ec * C, 1, n, seed=sum(shape), xa_zero=False)
    x, xa, dy, dya = (t.to(dtype) for t in (x, xa, dy, dya))
    d = torch.float64
    ref = O.net_autograd(x.to(d), xa.to(d), [Ws[0].to(d)], dy.to(d), dya.to(d), 0.9, n, C, first_stage=stage)
    x, xa, dy, dya, W = (t.cuda() for t in (x, xa, dy, dya, Ws[0]))
    y, ya, sy, sya = M.forward_stages_saving(x, xa, W, 0.9, 0, n, C, stage)
    _, _, dx, dxa, dW = M.backward_stages(sy, sya, dy, dya, W, 0.9, 0, n, C, stage, 1, want_inputs=False, grad_dtype=dtype)
    # the tolerances of test_gpu_parity (3e-6 of a value, amplified by 1/m at every step undone, for 32 rows and more); two
    # bfloat16 planes keep 2^-18 of a saved value where float32 keeps 2^-24; a bfloat16 result is rounded by at most 2^-8
    bf16 = dtype == torch.bfloat16
    tol = max(1e-5, (3e-6 if n >= 32 else 1.2e-6) * (64 if bf16 else 1) * 0.9 ** -n)
    if n <= 32 or not bf16:   # (64 steps amplify two planes past use)
        for got, want in zip((y, ya, dx, dxa), ref[:4]):
            assert got.dtype == dtype and O.rel_err(got, want) < (max(tol, 2.0 ** -8) if bf16 else tol)
        assert O.rel_err(dW[0], ref[4][0]) < tol
    # float32 outputs, from which the inputs come back
    y32, ya32 = M.forward_stages(x, xa, W, 0.9, 0, n, C, stage, 1, out_dtype=torch.float32)
    assert O.rel_err(y32, ref[0]) < 1e-5 and O.rel_err(ya32, ref[1]) < 1e-5
    back = 12e-6 * 0.9 ** -n   # test_gpu_parity's bound on reconstructed inputs
    if n < 64:
        ix, ixa = M.inverse_stages(y32, ya32, W, 0.9, 0, n, C, stage, 1)
        rx, rxa, dx2, dxa2, dW2 = M.backward_stages(y32, ya32, dy.float(), None, W, 0.9, 0, n, C, stage, 1, want_inputs=True)
        for got, want in ((ix, x), (ixa, xa), (rx, x), (rxa, xa)):
            assert O.rel_err(got, want) < back
        ref0 = O.net_autograd(x.to(d).cpu(), xa.to(d).cpu(), [Ws[0].to(d)], dy.to(d).cpu(), torch.zeros_like(ref[0]), 0.9, n, C,
                              first_stage=stage)
        f32 = max(1e-5, (3e-6 if n >= 32 else 1.2e-6) * 0.9 ** -n)
        assert O.rel_err(dx2, ref0[2]) < f32 and O.rel_err(dxa2, ref0[3]) < f32 and O.rel_err(dW2[0], ref0[4][0]) < f32


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("shape", [(4, 8, 1, 19, 3), (8, 32, 3, 3, 3), (16, 32, 3, 3, 3), (32, 32, 1, 7, 3), (32, 64, 2, 3, 3)],
                         ids=lambda s: "n%d_e%d_C%d_g%d_b%d" % s)
def test_table_and_lengths(M, shape, dtype):
    n, ec, C, groups, batch = shape
    N, d = n * groups, torch.float64
    x, xa, Ws, dy, dya = O.make_inputs(batch, N, ec * C, 1, n, seed=sum(shape), xa_zero=False)
    x, xa, dy, dya = (t.to(dtype) for t in (x, xa, dy, dya))
    table = torch.randperm(N, generator=torch.Generator().manual_seed(2))
    lens = [N, n * (groups // 2) + n // 2, 0]   # everything, a group that the length cuts, nothing
    ref = O.net_autograd_indexed(x.to(d), xa.to(d), [Ws[0].to(d)], dy.to(d), dya.to(d), 0.9, n, C, [table], lens)
    kw = dict(group_index=table.to(torch.int32).cuda(), ctx_len=torch.tensor(lens, dtype=torch.int32).cuda())
    x, xa, dy, dya, W = (t.cuda() for t in (x, xa, dy, dya, Ws[0]))
    y, ya, sy, sya = M.forward_stages_saving(x, xa, W, 0.9, 0, n, C, 2, **kw)
    _, _, dx, dxa, dW = M.backward_stages(sy, sya, dy, dya, W, 0.9, 0, n, C, 2, 1, want_inputs=False, grad_dtype=dtype, **kw)
    bf16 = dtype == torch.bfloat16
    tol = max(1e-5, (3e-6 if n >= 32 else 1.2e-6) * (64 if bf16 else 1) * 0.9 ** -n)   # as above
    for got, want in zip((y, ya, dx, dxa), ref[:4]):
        assert O.rel_err(got, want) < (max(tol, 2.0 ** -8) if bf16 else tol)
    assert O.rel_err(dW[0], ref[4][0]) < tol
    assert torch.equal(y[2], x[2]) and torch.equal(ya[2], xa[2]) and torch.equal(dx[2], dy[2]) and torch.equal(dxa[2], dya[2])
    y32, ya32 = M.forward_stages(x, xa, W, 0.9, 0, n, C, 2, 1, out_dtype=torch.float32, **kw)
    ix, ixa = M.inverse_stages(y32, ya32, W, 0.9, 0, n, C, 2, 1, **kw)
    rx, rxa, _, _, _ = M.backward_stages(y32, ya32, dy.float(), None, W, 0.9, 0, n, C, 2, 1, want_inputs=True, **kw)
    for got, want in ((ix, x), (ixa, xa), (rx, x), (rxa, xa)):
        assert O.rel_err(got, want) < 12e-6 * 0.9 ** -n


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
