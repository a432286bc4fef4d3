"""bfloat16 weights read, and their gradients written, by the kernels themselves: bit for bit what the same call gives on
the weights converted to float32 (the conversion is exact) and on its float32 dW rounded once."""
import ctypes

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


# (n_cache, E, heads, groups, stages, alpha)
CASES = [(16, 128, 4, 4, 1, 0.9),   # kernels for few groups, a group over two waves
         (4, 128, 2, 6, 1, 0.9),    # .. in part of one
         (16, 256, 4, 3, 1, 0.9),   # .. over four, an odd number of groups
         (16, 128, 4, 173, 1, 0.9), # larger launches: register tiles of 4 x 4
         (4, 128, 2, 173, 1, 0.9),  # 2 x 8
         (2, 32, 4, 1367, 1, 0.9),  # 2 x 4
         (16, 256, 4, 87, 1, 0.9),  # 4 x 8, an odd number of groups
         (8, 32, 32, 4, 1, 0.9),    # heads of one feature
         (5, 30, 2, 5, 1, 0.9),     # no powers of two
         (5, 30, 2, 5, 1, 0.0),     # generic kernels (alpha outside the scaled state)
         (2, 64, 2, 32, 5, 0.9),    # two-row multi-stage passes
         (4, 64, 2, 64, 4, 0.9)]    # multi-stage passes


@pytest.mark.parametrize("case", CASES, ids=lambda c: "n%d_E%d_C%d_g%d_L%d_a%g" % c)
def test_bfloat16_weights(M, case):
    n, E, C, groups, L, alpha = case
    x, xa, Ws, dy, dya = (t.cuda() if isinstance(t, torch.Tensor) else [w.cuda() for w in t]
                          for t in O.make_inputs(3, n * groups, E, L, n, seed=n + E, xa_zero=False))
    W = torch.stack(Ws).bfloat16()
    W32 = W.float()
    y, ya = M.forward_stages(x, xa, W, alpha, 0, n, C, 0, L)
    y32, ya32 = M.forward_stages(x, xa, W32, alpha, 0, n, C, 0, L)
    assert torch.equal(y, y32) and torch.equal(ya, ya32)
    for a, b in zip(M.inverse_stages(y, ya, W, alpha, 0, n, C, 0, L), M.inverse_stages(y, ya, W32, alpha, 0, n, C, 0, L)):
        assert torch.equal(a, b)
    kw = dict(want_inputs=False)
    want = M.backward_stages(y, ya, dy, dya, W32, alpha, 0, n, C, 0, L, **kw)
    got = M.backward_stages(y, ya, dy, dya, W, alpha, 0, n, C, 0, L, dw_dtype=torch.bfloat16, **kw)
    assert torch.equal(got[2], want[2]) and torch.equal(got[3], want[3])
    assert got[4].dtype == torch.bfloat16 and torch.equal(got[4], want[4].bfloat16())
    got = M.backward_stages(y, ya, dy, dya, W, alpha, 0, n, C, 0, L, **kw)   # float32 dW of bfloat16 weights
    assert torch.equal(got[4], want[4])


@pytest.mark.parametrize("types", [(torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)], ids=["bf16-f32", "f32-bf16"])
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("n,E,C,groups", [(16, 128, 4, 5), (16, 256, 4, 3), (4, 64, 4, 7), (8, 32, 32, 3),
                                          (16, 128, 4, 257), (16, 256, 4, 129), (4, 64, 4, 513)])   # register tiles with tanh too
def test_bfloat16_weights_with_mixed_types(M, n, E, C, groups, act, types):
    """The builds for every element type: results of another type than the inputs, with and without a table."""
    first, second = types
    x, xa, Ws, dy, dya = (t.cuda() if isinstance(t, torch.Tensor) else t[0].cuda()
                          for t in O.make_inputs(2, n * groups, E, 1, n, seed=n + E, xa_zero=False))
    W = Ws.bfloat16()
    table = torch.randperm(n * groups, generator=torch.Generator().manual_seed(1)).to(torch.int32).cuda()
    for kw in ({}, dict(group_index=table)):
        def both(f):
            for a, b in zip(f(W), f(W.float())):
                assert (a is None and b is None) or torch.equal(a, b)
        both(lambda w: M.forward_stages(x.to(first), xa.to(first), w, 0.9, act, n, C, 1, 1, out_dtype=second, **kw))
        both(lambda w: M.inverse_stages(x.to(first), xa.to(first), w, 0.9, act, n, C, 1, 1, out_dtype=second, **kw))
        both(lambda w: M.backward_stages(x.to(first), xa.to(first), dy.to(second), dya.to(second), w, 0.9, act, n, C, 1, 1,
                                         grad_dtype=first, **kw))


@pytest.mark.parametrize("case", [CASES[0], CASES[10], CASES[11]], ids=lambda c: "n%d_E%d_C%d_g%d_L%d_a%g" % c)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_one_array_per_stage(M, case, dtype):
    """NCN_W_ARRAYS: the weights of every stage where they are."""
    from ncn_cuda_amd import _lib
    n, E, C, groups, L, alpha = case
    x, xa, Ws, _, _ = (t.cuda() if isinstance(t, torch.Tensor) else [w.cuda().to(dtype) for w in t]
                       for t in O.make_inputs(2, n * groups, E, L, n, seed=n, xa_zero=False))
    want = M.forward_stages(x, xa, torch.stack(Ws), alpha, 0, n, C, 0, L)
    y, ya = torch.empty_like(x), torch.empty_like(x)
    shape = _lib.NcnShape(2, n * groups, E, C, n)
    lib = _lib.load()
    ws = torch.empty(max(16, lib.ncn_workspace_bytes_stages(ctypes.byref(shape), 0, L, 0, 0)), dtype=torch.uint8, device="cuda")
    ptrs = (ctypes.c_void_p * L)(*[w.data_ptr() for w in Ws])
    flags = _lib.NCN_W_ARRAYS | (_lib.NCN_W_BF16 if dtype == torch.bfloat16 else 0)
    args = lambda p: (x.data_ptr(), xa.data_ptr(), _lib.NCN_F32 | flags, y.data_ptr(), ya.data_ptr(), _lib.NCN_F32, None,
                      None, p, ws.data_ptr(), ws.numel(), ctypes.byref(shape), 0, L, alpha, 0.9, 0,
                      torch.cuda.current_stream().cuda_stream)
    array = ctypes.cast(ptrs, ctypes.c_void_p)
    assert lib.ncn_forward(*args(array)) == 0
    assert torch.equal(y, want[0]) and torch.equal(ya, want[1])
    # .. in the inverse and the backward, whose dW is one array
    st = torch.cuda.current_stream().cuda_stream
    want_x = M.inverse_stages(y, ya, torch.stack(Ws), alpha, 0, n, C, 0, L)
    ix, ixa = torch.empty_like(x), torch.empty_like(x)
    assert lib.ncn_inverse_ws(y.data_ptr(), ya.data_ptr(), flags, ix.data_ptr(), ixa.data_ptr(), _lib.NCN_F32, array, ws.data_ptr(),
                              ws.numel(), ctypes.byref(shape), 0, L, alpha, 0.9, 0, st) == 0
    assert torch.equal(ix, want_x[0]) and torch.equal(ixa, want_x[1])
    _, _, want_dx, want_dxa, want_dW = M.backward_stages(y, ya, x, xa, torch.stack(Ws), alpha, 0, n, C, 0, L, want_inputs=False,
                                                         dw_dtype=dtype)
    dx, dxa, dW = torch.empty_like(x), torch.empty_like(x), torch.empty(L, 2 * E, dtype=dtype, device="cuda")
    bws = torch.empty(lib.ncn_workspace_bytes_stages(ctypes.byref(shape), 0, L, 0, 2 if L > 1 else 1), dtype=torch.uint8, device="cuda")
    assert lib.ncn_backward(y.data_ptr(), ya.data_ptr(), flags, x.data_ptr(), xa.data_ptr(), _lib.NCN_F32, dx.data_ptr(),
                            dxa.data_ptr(), _lib.NCN_F32, None, None, array, dW.data_ptr(), bws.data_ptr(), bws.numel(),
                            ctypes.byref(shape), 0, L, alpha, 0.9, 0, st) == 0
    assert torch.equal(dx, want_dx) and torch.equal(dxa, want_dxa) and torch.equal(dW, want_dW)
    ptrs[L - 1] = None
    assert lib.ncn_forward(*args(array)) == -1   # NCN_ERR_NULL, nothing launched
