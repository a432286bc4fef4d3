"""Sum of the dW partial rows: one launch up to 2048 rows, two beyond; row counts around its block of 128 rows and around
the switch, column counts that end inside a block of 8 columns or fill blocks of 32 (numbered for the XCDs)."""
import pytest
import torch

from oracle import ncn_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ncn_cuda_amd import ncn_cuda_module
    return ncn_cuda_module


# (batch entries = wave tiles of a single head = partial rows, E, heads): 2E columns
CASES = [(1, 4, 1), (127, 4, 1), (132, 4, 1), (2048, 4, 1), (2049, 15, 3), (2052, 4, 1), (4096, 4, 1), (4100, 4, 1), (3, 15, 3), (5, 64, 2), (260, 128, 4), (4097, 15, 3)]


@pytest.mark.parametrize("batch,E,C", CASES)
def test_dw_sum(M, batch, E, C):
    n = 2
    x, xa, Ws, dy, dya = O.make_inputs(batch, n, E, 1, n, seed=batch + E, xa_zero=False)
    d = torch.float64
    ref = O.net_autograd(x.to(d), xa.to(d), [Ws[0].to(d)], dy.to(d), dya.to(d), 0.9, n, C)
    y, ya = M.forward_stages(x.cuda(), xa.cuda(), Ws[0].cuda(), 0.9, 0, n, C, 0, 1)
    dW = M.backward_stages(y, ya, dy.cuda(), dya.cuda(), Ws[0].cuda(), 0.9, 0, n, C, 0, 1, want_inputs=False)[4]
    again = M.backward_stages(y, ya, dy.cuda(), dya.cuda(), Ws[0].cuda(), 0.9, 0, n, C, 0, 1, want_inputs=False)[4]
    assert O.rel_err(dW[0], ref[4][0]) < 1e-5
    assert torch.equal(dW, again)   # a fixed order of additions
