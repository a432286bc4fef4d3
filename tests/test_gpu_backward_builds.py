"""The backward stage kernels for every element type and activation that have no loop over tiles (launches with a wave for
every tile), against the float64 oracle: saved outputs, gradients and results of different types, every activation, with and
without a table and context lengths, tiles of 2 x 4, 4 x 4, 2 x 8 and 4 x 8, a last wave tile that is partly empty.  Small launches
of tanh run on the kernels for few groups (ncn_split_kernels.h), so tanh has a second, larger size of every shape."""
import pytest
import torch

from conftest import kernels_of
from oracle import ncn_oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(2, 8, 4, 33), (4, 64, 2, 5), (8, 32, 4, 3), (16, 32, 4, 3), (16, 64, 1, 3), (32, 8, 4, 2)]   # n, width, heads, groups
F, H = torch.float32, torch.bfloat16
# the same shapes above a million elements (a quarter of that for 2 and 4 rows)
LARGE = [(n, ec, C, ((1 << (20 if n >= 8 else 18)) // (3 * n * ec * C) + 1) | 1) for n, ec, C, _ in SHAPES]
TYPES = [("f32", F, F), ("f32", H, F), ("f32", F, H), ("planes", F, F), ("planes", H, F)]   # saved outputs, dy, dx


@pytest.fixture(scope="module")
def M():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ncn_cuda_amd import ncn_cuda_module
    return ncn_cuda_module


@pytest.mark.parametrize("indexed", [False, True], ids=["stride", "table"])
@pytest.mark.parametrize("types", TYPES, ids=lambda t: "%s-%s-%s" % (t[0], str(t[1])[6:], str(t[2])[6:]))
@pytest.mark.parametrize("shape", LARGE, ids=lambda s: "n%d_e%d_C%d_g%d" % s)
def test_backward_of_tanh_on_the_register_tiles(M, shape, types, indexed):
    test_backward(M, shape, 0, types, indexed, "stage")


@pytest.mark.parametrize("indexed", [False, True], ids=["stride", "table"])
@pytest.mark.parametrize("types", TYPES, ids=lambda t: "%s-%s-%s" % (t[0], str(t[1])[6:], str(t[2])[6:]))
@pytest.mark.parametrize("act", [0, 1, 2, 3, -1])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "n%d_e%d_C%d_g%d" % s)
def test_backward(M, shape, act, types, indexed, kind=None):
    kind = kind or ("split" if act == 0 else "stage")   # the kernels that have to run
    n, ec, C, groups = shape
    saved, g_dtype, out_dtype = types
    batch, N = 3, n * groups
    if act in (1, 3):   # away from the kink, on whose side rounding would decide
        x, xa, Ws, dy, dya = O.make_inputs_signed_regimes(batch, N, ec * C, 1, n, seed=sum(shape))
    else:
        x, xa, Ws, dy, dya = O.make_inputs(batch, N, ec * C, 1, n, seed=sum(shape), xa_zero=False)
    if saved == "planes":
        x, xa = x.to(H), xa.to(H)
    dy, dya = dy.to(g_dtype), dya.to(g_dtype)
    large = shape in LARGE
    if large:   # the oracle's float64 on the GPU
        x, xa, dy, dya, Ws = *(t.cuda() for t in (x, xa, dy, dya)), [Ws[0].cuda()]
    d = torch.float64
    args = (x.to(d), xa.to(d), [Ws[0].to(d)], dy.to(d), dya.to(d), 0.9, n, C)
    kw = {}
    if indexed:
        table = torch.randperm(N, generator=torch.Generator().manual_seed(2))
        lens = [N, n * (groups // 2) + n // 2, 0]
        ref = O.net_autograd_indexed(*args, [table.cuda() if large else table], lens, activation=act)
        kw = dict(group_index=table.to(torch.int32).cuda(), ctx_len=torch.tensor(lens, dtype=torch.int32).cuda())
    else:
        ref = O.net_autograd(*args, activation=act, first_stage=2)
    W = Ws[0].cuda()
    y, ya, sy, sya = M.forward_stages_saving(x.cuda(), xa.cuda(), W, 0.9, act, n, C, 2, **kw)
    (_, _, dx, dxa, dW), ran = kernels_of(lambda: M.backward_stages(sy, sya, dy.cuda(), dya.cuda(), W, 0.9, act, n, C, 2, 1, want_inputs=False,
                                                                    grad_dtype=out_dtype, **kw))
    assert {name.split("_")[0] for name in ran} - {"reduce"} == {kind}, ran
    # float32: 1.2e-6 of a value, amplified by 1/m at every step undone; two planes keep 2^-18 of a saved value where float32
    # keeps 2^-24: 64 times that; a bfloat16 result is rounded once more, by at most 2^-8 of it
    # (the largest of a million errors of 32 steps lies further out: the 3e-6 of test_gpu_few_groups)
    tol = max(1e-5, (3e-6 if large and n >= 32 else 1.2e-6) * (64 if saved == "planes" else 1) * 0.9 ** -n)
    out_tol = tol if out_dtype == F else max(tol, 2.0 ** -8)
    assert dx.dtype == out_dtype and dxa.dtype == out_dtype and dW.dtype == F
    assert O.rel_err(dx, ref[2]) < out_tol and O.rel_err(dxa, ref[3]) < out_tol and O.rel_err(dW[0], ref[4][0]) < tol
    if indexed:
        assert torch.equal(dx[2].cpu(), dy[2].cpu().to(out_dtype)) and torch.equal(dxa[2].cpu(), dya[2].cpu().to(out_dtype))
