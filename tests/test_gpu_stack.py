"""ncn_stack_forward / ncn_stack_backward (a trained stack in one call per direction) against the float64 oracle: every
pairing of kept ranges with passes, both element types, group counts without multi-stage passes, heads of one feature."""
import ctypes

import pytest
import torch

from oracle import ncn_oracle as O

pytestmark = pytest.mark.gpu

# batch, N, E, heads, n_cache, stages, max_range, max_saves; ranges expected
CASES = [
    ((2, 1024, 128, 4, 4, 5, 6, 5), None),    # ranges of one and two stages
    ((2, 2048, 64, 2, 4, 6, 6, 1), 1),        # one range: scratch between passes, states handed on inside it
    ((1, 2048, 64, 2, 4, 7, 6, 2), 2),        # two ranges, one of them of several passes
    ((2, 8192, 64, 2, 2, 13, 13, 1), 1),      # three backward passes in one range
    ((1, 8192, 32, 1, 2, 14, 13, 2), 2),
    ((2, 1020, 64, 2, 4, 5, 6, 5), 5),        # an odd number of groups: one launch per stage, every output kept
    ((2, 1018, 64, 2, 2, 4, 13, 1), 1),       # the same with nothing kept between the stages
    ((1, 16, 32, 4, 2, 3, 13, 3), None),      # the smallest rings
    ((1, 512, 64, 64, 2, 7, 13, 7), None),    # heads of one feature
]


@pytest.fixture(scope="module")
def M():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ncn_cuda_amd import ncn_cuda_module
    return ncn_cuda_module


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("case,ranges", CASES, ids=lambda c: "_".join(map(str, c)) if isinstance(c, tuple) else "")
def test_stack(M, case, ranges, dtype):
    batch, N, E, C, n, L, max_range, max_saves = case
    x, xa, Ws, dy, dya = O.make_inputs(batch, N, E, L, n, seed=sum(case), xa_zero=False, dtype=dtype)
    d = torch.float64
    ref = O.net_autograd(x.to(d), xa.to(d), [w.to(d) for w in Ws], dy.to(d), dya.to(d), 0.9, n, C, first_stage=1)
    W = torch.stack([w.reshape(-1) for w in Ws]).cuda()
    plan, y, ya, saves = M.stack_forward(x.cuda(), xa.cuda(), W, 0.9, 0, n, C, 1, L, max_range,
                                         8 * x.numel() * max_saves)
    assert plan.ranges == ranges or (ranges is None and 1 <= plan.ranges <= max_saves)
    f32 = dtype == torch.float32
    kept = (y, ya) if f32 else (None, None)
    # float32: 1.2e-6 per unit of rounding, amplified by 1/m at each of the steps between two kept values (13 stages of
    # groups of two rows at most); bfloat16 results are rounded once, by at most half a unit of their eight significant
    # bits: 2^-8 of a value
    tol = 1.2e-6 * 0.9 ** -(n * min(max_range, L)) if f32 else 2.0 ** -8
    for grad_a in (dya.cuda(), None):
        r = ref if grad_a is not None else O.net_autograd(x.to(d), xa.to(d), [w.to(d) for w in Ws], dy.to(d),
                                                          torch.zeros_like(dya).to(d), 0.9, n, C, first_stage=1)
        dx, dxa, dW = M.stack_backward(plan, *kept, saves, dy.cuda(), grad_a, W)
        for name, got, want in (("y", y, r[0]), ("ya", ya, r[1]), ("dx", dx, r[2]), ("dxa", dxa, r[3])):
            assert got.dtype == dtype
            assert O.rel_err(got, want) < tol, name
        for l in range(L):
            assert dW.dtype == dtype and O.rel_err(dW[l], r[4][l].reshape(-1)) < tol, l


@pytest.mark.parametrize("act", [1, 2, 3, -1])
@pytest.mark.parametrize("case", [CASES[1][0], CASES[3][0], CASES[5][0]], ids=lambda c: "_".join(map(str, c)))
def test_other_activations(M, case, act):
    batch, N, E, C, n, L, max_range, max_saves = case
    make = O.make_inputs_signed_regimes if act in (1, 3) else O.make_inputs   # relu: away from its kink
    x, xa, Ws, dy, dya = make(batch, N, E, L, n, seed=sum(case))
    d = torch.float64
    ref = O.net_autograd(x.to(d), xa.to(d), [w.to(d) for w in Ws], dy.to(d), dya.to(d), 0.9, n, C, activation=act)
    W = torch.stack([w.reshape(-1) for w in Ws]).cuda()
    plan, y, ya, saves = M.stack_forward(x.cuda(), xa.cuda(), W, 0.9, act, n, C, 0, L, max_range, 8 * x.numel() * max_saves)
    dx, dxa, dW = M.stack_backward(plan, y, ya, saves, dy.cuda(), dya.cuda(), W)
    tol = 1.2e-6 * 0.9 ** -(n * min(max_range, L))   # as in test_stack
    for name, got, want in (("y", y, ref[0]), ("ya", ya, ref[1]), ("dx", dx, ref[2]), ("dxa", dxa, ref[3]),
                            *(("dW%d" % l, dW[l], ref[4][l].reshape(-1)) for l in range(L))):
        assert O.rel_err(got, want) < tol, name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("n", [2, 4])
def test_results_depend_on_the_inputs_alone(M, n, dtype):
    """The same bits again whatever the memory holds that scratch, saves and outputs are allocated from (NaN here), and with a
    pass on other inputs in between."""
    from ncn_cuda_amd.modules import fused_ncn_net
    batch, N, E, C, L = 4, 2048, 64, 2, 6

    def inputs(seed):
        x, xa, Ws, dy, _ = O.make_inputs(batch, N, E, L, n, seed=seed, xa_zero=False, dtype=dtype)
        return [t.cuda().requires_grad_() for t in (x, xa, *Ws)], dy.cuda()

    def run(leaves, dy):
        y, ya = fused_ncn_net(leaves[0], leaves[1], leaves[2:], 0.9, 0, n, C)
        return [y, ya, *torch.autograd.grad(y, leaves, dy)]

    leaves, dy = inputs(3)
    first = [t.detach().clone() for t in run(leaves, dy)]
    for again in range(3):
        run(*inputs(4 + again))
        poison = [torch.full((1 << k,), float("nan"), device="cuda") for k in range(6, 24) for _ in range(4)]
        del poison
        for a, b in zip(run(leaves, dy), first):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("batch,N,E,C,n,L", [(16, 2048, 128, 4, 4, 6),     # multi-stage passes
                                             (16, 2046, 128, 4, 2, 13)])   # an odd number of groups: one launch per stage
@pytest.mark.parametrize("how", ["no_grad", "no_leaf"])
def test_no_activations_are_kept_without_gradients(M, batch, N, E, C, n, L, dtype, how):
    """The whole-net node under no_grad, or on tensors that want no gradient: nothing is kept for a backward.  At most a pair
    for the outputs, a float32 pair that the passes end in and one that they run through; the training plan of the second
    shape keeps 13 pairs."""
    from ncn_cuda_amd.modules import fused_ncn_net
    x, xa, Ws, _, _ = O.make_inputs(batch, N, E, L, n, seed=5, xa_zero=False, dtype=dtype)
    ref = O.net_forward(x.double(), xa.double(), [w.double() for w in Ws], 0.9, n, C)
    x, xa, Ws = x.cuda(), xa.cuda(), [w.cuda().requires_grad_(how == "no_grad") for w in Ws]

    def run():
        if how == "no_leaf":
            return fused_ncn_net(x, xa, Ws, 0.9, 0, n, C)
        with torch.no_grad():
            return fused_ncn_net(x, xa, Ws, 0.9, 0, n, C)

    run()
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    y, ya = run()
    peak = torch.cuda.max_memory_allocated() - before
    pair = 2 * x.numel()
    assert peak <= pair * (4 + 4 + (2 if dtype == torch.bfloat16 else 0)) + (1 << 20)
    assert not y.requires_grad and y.dtype == dtype
    # float32: rounding of the sums, 13 stages at most; bfloat16: the outputs are rounded once
    tol = 2e-6 if dtype == torch.float32 else 2.0 ** -8
    assert O.rel_err(y, ref[0]) < tol and O.rel_err(ya, ref[1]) < tol


@pytest.mark.parametrize("why", ["little_left", "allocation_fails"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_fewer_activations_are_kept_where_memory_is_short(M, monkeypatch, dtype, why):
    """A stack that would keep every stage's outputs keeps the fewest when little device memory is left, or when the
    allocation fails; its gradients are as good."""
    batch, N, E, C, n, L = 2, 1018, 64, 2, 2, 13     # 509 groups: one launch per stage
    x, xa, Ws, dy, dya = O.make_inputs(batch, N, E, L, n, seed=1, xa_zero=False, dtype=dtype)
    d = torch.float64
    ref = O.net_autograd(x.to(d), xa.to(d), [w.to(d) for w in Ws], dy.to(d), dya.to(d), 0.9, n, C)
    W = torch.stack([w.reshape(-1) for w in Ws]).cuda()
    x, xa, dy, dya = x.cuda(), xa.cuda(), dy.cuda(), dya.cuda()
    call = lambda: M.stack_forward(x, xa, W, 0.9, 0, n, C, 0, L, 13, 32 << 30)
    assert call()[0].ranges == L
    failed = []
    if why == "little_left":
        monkeypatch.setattr(M, "_SAVES_LOOK_AT_MEMORY", 0)
        total = torch.cuda.get_device_properties(x.device).total_memory
        monkeypatch.setattr(torch.cuda, "memory_allocated", lambda dev=None: total - 16 * x.numel())
    else:
        real = torch.empty

        def empty(*size, **kw):
            if len(size) == 1 and isinstance(size[0], tuple) and len(size[0]) == 5 and size[0][0] > 1:
                failed.append(size[0])
                raise torch.OutOfMemoryError("no memory")
            return real(*size, **kw)

        monkeypatch.setattr(torch, "empty", empty)
    plan, y, ya, saves = call()
    assert plan.ranges == 1 and (saves is None if dtype == torch.float32 else saves.shape[0] == 1)
    assert bool(failed) == (why == "allocation_fails")
    kept = (y, ya) if dtype == torch.float32 else (None, None)
    dx, dxa, dW = M.stack_backward(plan, *kept, saves, dy, dya, W)
    tol = 1.2e-6 * 0.9 ** -(n * L) if dtype == torch.float32 else 2.0 ** -8   # as in test_stack
    for got, want in ((y, ref[0]), (ya, ref[1]), (dx, ref[2]), (dxa, ref[3])):
        assert O.rel_err(got, want) < tol
    for l in range(L):
        assert O.rel_err(dW[l], ref[4][l].reshape(-1)) < tol


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_a_native_node_without_memory_leaves_the_call_to_the_python_node(M, dtype):
    """The native node plans for every activation and runs out of memory; the call is then made with the fewest."""
    from ncn_cuda_amd.modules import fused_ncn_net
    batch, N, E, C, n, L = 64, 1018, 128, 4, 2, 13     # 66 MB a pair of float32 activations, one launch per stage
    gen = torch.Generator(device="cuda").manual_seed(1)
    x, xa, dy, dya = (torch.randn(batch, N, E, generator=gen, device="cuda").to(dtype) for _ in range(4))
    leaves = [x.requires_grad_(), xa.requires_grad_(), *((torch.randn(2 * E, generator=gen, device="cuda") / n ** 0.5).requires_grad_() for _ in range(L))]

    def call():
        y, ya = fused_ncn_net(leaves[0], leaves[1], leaves[2:], 0.9, 0, n, C)
        return type(y.grad_fn).__name__, [y.detach(), ya.detach(), *torch.autograd.grad([y, ya], leaves, [dy, dya])]

    name, want = call()
    assert name != "NCNNetFunctionBackward"
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (600 << 20)) / total)   # the saves alone are 800 MB
    try:
        name, got = call()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert name == "NCNNetFunctionBackward"
    tol = 1.2e-6 * 0.9 ** -(n * L) if dtype == torch.float32 else 2.0 ** -8   # as in test_stack
    for a, b in zip(got, want):
        assert O.rel_err(a, b) < tol


def test_refusals(M):
    """Outputs that are the inputs, a workspace that is too small: refused before any launch."""
    from ncn_cuda_amd import _lib
    x = torch.zeros(1, 64, 32, device="cuda")
    xa, y, W = torch.zeros_like(x), torch.zeros_like(x), torch.zeros(3, 64, device="cuda")
    sh = _lib.NcnShape(1, 64, 32, 1, 2)
    lib = _lib.load()

    def forward(out):
        return lib.ncn_stack_forward(M._ptr(x), M._ptr(xa), 0, M._ptr(out), M._ptr(y), 0, None, M._ptr(W), None,
                                     ctypes.c_size_t(0), ctypes.byref(sh), 0, 3, 13, 1, 0.9, 0.9, 0, M._stream(x.device))

    assert forward(x) == -8 and "call's own inputs" in _lib.error_string(forward(x))   # NCN_ERR_ALIAS
    rc = lib.ncn_stack_backward(M._ptr(y), M._ptr(y), None, M._ptr(x), None, 0, M._ptr(xa), M._ptr(xa), 0, M._ptr(W),
                                M._ptr(W), 0, None, ctypes.c_size_t(0), ctypes.byref(sh), 0, 3, 13, 1, 0.9, 0.9, 0,
                                M._stream(x.device))
    assert "workspace" in _lib.error_string(rc)
