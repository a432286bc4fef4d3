"""The multi-level radix kernels (ncn_radix_kernels.h) against the float64 oracle: every head width and group size, passes of two
levels up to the most that a workgroup holds, so that the levels run in registers, after exchanges of register and lane bits and
after the exchange through LDS, windows that are no power of two, every kind of launch; and the kernels that keep rows in LDS
(ncn_fused_kernels.h), which launches with few workgroups take."""
import pytest
import torch

from conftest import kernels_of
from oracle import ncn_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ncn_cuda_amd import ncn_cuda_module
    return ncn_cuda_module


def check(M, batch, N, ec, C, n, first, L, act=0, dtype=torch.float32, forward=None, backward=None):
    """forward, backward: the kernels that the passes have to run on, "radix" (registers) or "fused" (LDS)."""
    E = ec * C
    make = O.make_inputs_signed_regimes if act in (1, 3) else O.make_inputs   # away from the kink
    x, xa, Ws, dy, dya = make(batch, N, E, L, n, seed=N + ec) if act in (1, 3) else make(batch, N, E, L, n, seed=N + ec, xa_zero=False)
    x, xa, dy, dya = (t.to(dtype) for t in (x, xa, dy, dya))
    d = torch.float64
    tables = [O.radix_group_table(N, n, first + l) for l in range(L)]
    ref = O.net_autograd_indexed(x.to(d), xa.to(d), [w.to(d) for w in Ws], dy.to(d), dya.to(d), 0.9, n, C, tables, activation=act)
    W = torch.stack([w.reshape(-1) for w in Ws]).cuda()
    x, xa, dy, dya = (t.cuda() for t in (x, xa, dy, dya))
    args = (W, 0.9, act, n, C, first, L)
    (y, ya), ran = kernels_of(lambda: M.forward_radix(x, xa, *args))
    multi_level = lambda names: {k.split("_")[0] for k in names} & {"radix", "fused"}   # (a last pass of one level has other kernels)
    assert forward is None or multi_level(ran) == {forward}, ran
    (rx, rxa, dx, dxa, dW), ran = kernels_of(lambda: M.backward_radix(y, ya, dy, dya, *args))
    assert backward is None or multi_level(ran) == {backward}, ran
    _, _, dx2, dxa2, dW2 = M.backward_radix(y, ya, dy, dya, *args, want_inputs=False)
    ix, ixa = M.inverse_radix(y, ya, *args)
    # rounding of the sums, amplified by 1/m at every step undone (as in test_gpu_stack); reconstruction as in test_gpu_parity
    tol = max(1e-5, 1.2e-6 * 0.9 ** -(n * L))
    assert O.rel_err(y, ref[0]) < 1e-5 and O.rel_err(ya, ref[1]) < 1e-5
    assert O.rel_err(dx, ref[2]) < tol and O.rel_err(dxa, ref[3]) < tol
    for l in range(L):
        assert O.rel_err(dW[l], ref[4][l].reshape(-1)) < tol, l
    for got, want in ((rx, x), (rxa, xa), (ix, x), (ixa, xa)):
        assert O.rel_err(got, want) < 12e-6 * 0.9 ** -(n * L)
    assert torch.equal(dx, dx2) and torch.equal(dxa, dxa2) and torch.equal(dW, dW2)


@pytest.mark.parametrize("levels", [2, 3, 5, "most"])
@pytest.mark.parametrize("ec", [8, 16, 32, 64, 128])
@pytest.mark.parametrize("n", [2, 4])
def test_levels(M, n, ec, levels):
    most = {2: {8: 10, 16: 9, 32: 8, 64: 7, 128: 6}, 4: {8: 5, 16: 4, 32: 4, 64: 3, 128: 3}}[n][ec]
    L = most if levels == "most" else min(levels, most)
    check(M, 2, 3 * n ** L, ec, 2, n, 0, L)          # three windows of every level
    # workgroups that are full in either direction
    check(M, 1, 3 * 8192 // ec, ec, 2, n, 0, L, forward="radix", backward="radix")


@pytest.mark.parametrize("n,ec,first,L", [(2, 32, 3, 6), (4, 32, 1, 3), (2, 8, 1, 9), (4, 64, 1, 2)])
def test_levels_that_do_not_start_at_the_first(M, n, ec, first, L):
    check(M, 1, 5 * n ** (first + L), ec, 3, n, first, L)


@pytest.mark.parametrize("act", [1, 2, 3, -1])
@pytest.mark.parametrize("n,ec,L", [(2, 32, 7), (4, 32, 3), (2, 128, 5), (4, 16, 4)])
def test_other_activations(M, n, ec, L, act):
    check(M, 2, 3 * n ** L, ec, 2, n, 0, L, act)


# the same on launches that are large enough for the registers
@pytest.mark.parametrize("act", [1, 2, 3, -1])
@pytest.mark.parametrize("n,ec,L,batch,N", [(2, 32, 6, 600, 64), (4, 16, 3, 600, 64), (2, 128, 4, 150, 48), (4, 64, 3, 150, 64), (2, 8, 3, 600, 24)])
def test_other_activations_on_many_workgroups(M, n, ec, L, batch, N, act):
    check(M, batch, N, ec, 2, n, 0, L, act, forward="radix", backward="radix")


@pytest.mark.parametrize("n,ec,batch,N,L,act,backward", [(2, 8, 5, 80, 4, 0, "fused"), (2, 16, 3, 96, 5, 0, "fused"), (2, 32, 3, 96, 5, 0, "radix"),
                                                         (2, 64, 2, 48, 4, 0, "radix"), (2, 128, 2, 24, 3, 0, "radix"), (4, 8, 3, 192, 3, 0, "fused"),
                                                         (4, 32, 2, 48, 2, 0, "fused"), (4, 128, 2, 16, 2, 0, "radix"), (2, 32, 2, 256, 6, 2, "fused"),
                                                         (4, 16, 2, 192, 3, 1, "fused"), (2, 64, 2, 128, 5, -1, "radix"), (2, 1, 3, 48, 4, 0, "fused")])
def test_few_workgroups(M, n, ec, batch, N, L, act, backward):
    check(M, batch, N, ec, 16 if ec == 1 else 2, n, 0, L, act, forward="fused", backward=backward)


@pytest.mark.parametrize("n,ec,N,L,act,below,above", [
    (2, 8, 24, 3, 0, 768, 769), (2, 32, 32, 5, 0, 512, 513), (2, 32, 192, 6, 0, 256, 384), (2, 8, 576, 6, 0, 512, 513), (2, 16, 448, 6, 0, None, 1),
    (2, 32, 256, 7, 0, None, 1), (2, 64, 32, 4, 0, 256, 257), (4, 128, 16, 2, 0, 256, 257), (2, 16, 24, 3, 1, 1024, 1025), (2, 32, 192, 6, 1, 512, 513),
    (4, 8, 64, 3, 2, 512, 513), (2, 64, 64, 5, -1, 256, 257)])
def test_which_kernels_take_a_forward_pass(M, n, ec, N, L, act, below, above):
    """By workgroups (one to a batch entry here): up to as many in LDS, from as many on in registers."""
    W = torch.randn(L, 2 * ec, device="cuda") / n ** 0.5
    for batch, kind in ((below, "fused"), (above, "radix")):
        if batch:
            x = torch.randn(batch, N, ec, device="cuda")
            (y, ya), ran = kernels_of(lambda: M.forward_radix(x, x, W, 0.9, act, n, 1, 0, L))
            assert {k.split("_")[0] for k in ran} == {kind}
            _, ran = kernels_of(lambda: M.inverse_radix(y, ya, W, 0.9, act, n, 1, 0, L))
            assert {k.split("_")[0] for k in ran} == {kind}


@pytest.mark.parametrize("n,E,L,act", [(2, 32, 8, 0), (4, 64, 4, 0), (2, 8, 9, 2), (4, 16, 3, -1)])
def test_heads_of_one_feature(M, n, E, L, act):
    check(M, 2, 3 * n ** L, 1, E, n, 0, L, act)


@pytest.mark.parametrize("n,ec,L", [(2, 32, 8), (4, 32, 4)])
def test_bfloat16_inputs_and_gradients(M, n, ec, L):
    check(M, 2, n ** L, ec, 2, n, 0, L, dtype=torch.bfloat16)


# windows counted through batch entries: several entries to a workgroup, an entry that begins inside one and ends in the next, a
# last workgroup that is not full; levels that do not start at the first; more and fewer windows to an entry than to a workgroup
@pytest.mark.parametrize("batch,N,ec,n,first,L,act,dtype", [
    (259, 4, 8, 2, 0, 2, 0, torch.float32), (213, 8, 32, 2, 0, 3, 0, torch.float32), (215, 80, 32, 2, 0, 4, 0, torch.float32),
    (41, 640, 32, 2, 0, 7, 0, torch.float32), (91, 96, 64, 2, 0, 5, 0, torch.float32), (89, 48, 128, 2, 0, 4, 0, torch.float32),
    (215, 96, 16, 2, 2, 3, 0, torch.float32), (213, 48, 32, 4, 0, 2, 0, torch.float32), (215, 192, 16, 4, 1, 2, 0, torch.bfloat16),
    (239, 64, 8, 4, 0, 3, 2, torch.float32), (379, 48, 32, 2, 0, 4, -1, torch.bfloat16), (819, 56, 1, 2, 0, 3, 0, torch.float32),
    (1123, 16, 1, 4, 0, 2, 2, torch.float32)])
def test_windows_of_several_batch_entries(M, batch, N, ec, n, first, L, act, dtype):
    # (heads of one feature are laid out as one of 16)
    check(M, batch, N, ec, 16 if ec == 1 else 3, n, first, L, act, dtype, forward="radix", backward="radix")


@pytest.mark.parametrize("n,L,rows", [(2, 2, 4), (4, 2, 16)])
def test_millions_of_short_sequences(M, n, L, rows):
    """More windows than a grid holds workgroups: several to a workgroup."""
    batch, C = (1 << 22) * 4 // rows, 4
    gen = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randn(batch * (2 if n == 4 else 1), rows, 8 * C, generator=gen, device="cuda", dtype=torch.bfloat16)
    W = torch.randn(L, 16 * C, generator=gen, device="cuda") / n ** 0.5
    args = (W, 0.9, 0, n, C, 0, L)
    y, ya = M.forward_radix(x, x, *args)
    ix, ixa = M.inverse_radix(y, ya, *args)
    for part in (slice(0, 1000), slice(len(x) // 2 - 500, len(x) // 2 + 500), slice(len(x) - 1001, None)):
        py, pya = M.forward_radix(x[part].contiguous(), x[part].contiguous(), *args)
        assert torch.equal(y[part], py) and torch.equal(ya[part], pya)
        for a, b in zip(M.inverse_radix(py, pya, *args), (ix, ixa)):
            assert torch.equal(a, b[part]) and O.rel_err(a, x[part].float()) < 12e-6 * 0.9 ** -(n * L)


# the windows of an entry fill workgroups, or are counted through the entries
@pytest.mark.parametrize("n,L,batch,N", [(2, 7, 16384 // 7 + 100, 512), (4, 4, 16384 // 4 + 100, 512), (2, 2, 360000, 12)])
def test_more_windows_than_partial_rows(M, n, L, batch, N):
    """The backward then loops over windows; each half of the batch has a workgroup for every window."""
    E = 8
    gen = torch.Generator(device="cuda").manual_seed(0)
    x, xa, dy, dya = (torch.randn(batch, N, E, generator=gen, device="cuda") for _ in range(4))
    W = torch.randn(L, 2 * E, generator=gen, device="cuda") / n ** 0.5
    args = (W, 0.9, 0, n, 1, 0, L)
    y, ya = M.forward_radix(x, xa, *args)
    _, _, dx, dxa, dW = M.backward_radix(y, ya, dy, dya, *args, want_inputs=False)
    halves = [M.backward_radix(*(t[s].contiguous() for t in (y, ya, dy, dya)), *args, want_inputs=False)
              for s in (slice(0, batch // 2), slice(batch // 2, batch))]
    assert torch.equal(dx, torch.cat([h[2] for h in halves])) and torch.equal(dxa, torch.cat([h[3] for h in halves]))
    want = sum(h[4].double() for h in halves)
    # sums of 2^20 products in float32, in other orders
    assert ((dW.double() - want).norm() / want.norm()) < 1e-5
