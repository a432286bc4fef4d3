"""float32 one-stage launches of heads of 32 on arrays of 2^23 elements and more load their rows with a cache hint: the same bits as the halves of
the batch, which are below that size, in every direction, with plain and gathered groups and with rows past a length."""
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


def inputs(b, N, E, n):
    gen = torch.Generator(device="cuda").manual_seed(b * 7 + n)
    x, xa, dy, dya = (torch.randn(b, N, E, device="cuda", generator=gen) for _ in range(4))
    return x, xa, dy, dya, torch.randn(1, 2 * E, device="cuda", generator=gen) * (0.3 / n ** 0.5)


# at the size itself and beyond, groups of 8 to 32 rows with the hint; tiles of 4 x 8 without
@pytest.mark.parametrize("b,N,E,C,n", [(32, 2048, 128, 4, 8), (34, 2048, 128, 4, 16), (32, 2080, 128, 4, 32), (16, 2080, 256, 2, 16), (16, 2080, 256, 4, 32), (16, 2056, 256, 4, 8)])
def test_halves_of_the_batch(M, b, N, E, C, n):
    x, xa, dy, dya, W = inputs(b, N, E, n)
    assert x.numel() >= 1 << 23 > x.numel() // 2

    def run(s):
        y, ya = M.forward_stages(x[s], xa[s], W, 0.9, 0, n, C, 0, 1)
        back = M.inverse_stages(y, ya, W, 0.9, 0, n, C, 0, 1)
        grads = M.backward_stages(y, ya, dy[s], dya[s], W, 0.9, 0, n, C, 0, 1, want_inputs=False)
        return [y, ya, *back, *[g for g in grads if g is not None and g.dim() == 3]], grads[4]
    whole, dW = run(slice(None))
    a, dWa = run(slice(0, b // 2))
    c, dWc = run(slice(b // 2, None))
    for w, p, q in zip(whole, a, c):
        assert torch.equal(w, torch.cat([p, q]))
    assert O.rel_err(dW, dWa.double() + dWc.double()) < 1e-5   # sums of 2^18 rows and more in another order


def test_table_and_lengths(M):
    from ncn_cuda_amd.chunk_linear import fused_chunk_linear_ncn, radix_group_table
    b, N, E, C, n = 32, 2048, 128, 4, 16
    x, xa, dy, _, W = inputs(b, N, E, n)
    table = radix_group_table(N, n, 1, device="cuda")
    lens = torch.randint(N // 2, N + 1, (b,), device="cuda").to(torch.int32)

    def run(s):
        xr = x[s].clone().requires_grad_(True)
        y, ya = fused_chunk_linear_ncn(xr, xa[s], W[0], table, lens[s], 0.9, "tanh", C, n, 0)
        return [y.detach(), ya.detach(), torch.autograd.grad(y, xr, dy[s])[0]]
    whole, a, c = run(slice(None)), run(slice(0, b // 2)), run(slice(b // 2, None))
    for w, p, q in zip(whole, a, c):
        assert torch.equal(w, torch.cat([p, q]))
