"""The autograd nodes in native code (csrc/ncn_torch.cpp) against the nodes in Python, which run the same kernels: the same bits in
every output and gradient, the same behaviour under hooks, transforms and modes, and the same refusals."""
import pytest
import torch

from oracle import ncn_oracle as O

pytestmark = pytest.mark.gpu

F, H = torch.float32, torch.bfloat16
ALPHA = 0.9


@pytest.fixture(scope="module")
def P():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import ncn_cuda_amd
    from ncn_cuda_amd import _native, chunk_linear, modules
    assert _native.ext().__name__.endswith("_ncn_torch")
    return modules, chunk_linear, ncn_cuda_amd.ncn_cuda_module, _native.ext()


def leaves(n, ec, C, groups, L, dtype, w_dtype, batch=2):
    x, xa, Ws, dy, dya = O.make_inputs(batch, n * groups, ec * C, L, n, seed=n + ec, xa_zero=False)
    x, xa, dy, dya = (t.to(dtype).cuda() for t in (x, xa, dy, dya))
    return x.requires_grad_(), xa.requires_grad_(), [w.to(w_dtype).cuda().requires_grad_() for w in Ws], dy, dya


def kinds(P, kind, n, C):
    """(native, python) callables of (x, xa, Ws) for one kind of node."""
    modules, chunk, M, ext = P
    if kind == "stage":
        return (lambda x, xa, Ws: ext.stage(x, xa, Ws[0], ALPHA, 0, n, C, 2),
                lambda x, xa, Ws: modules.NCNFunction.apply(x, xa, Ws[0], ALPHA, 0, n, C, 2))
    if kind == "stack":
        return (lambda x, xa, Ws: ext.stack(x, xa, Ws, ALPHA, 0, n, C, 0, modules.default_save_every(n), 32 << 30, 1 << 30),
                lambda x, xa, Ws: modules.NCNNetFunction.apply(x, xa, ALPHA, 0, n, C, 0, None, *Ws))
    if kind == "radix":
        return (lambda x, xa, Ws: ext.radix(x, xa, Ws, ALPHA, 0, n, C, 0),
                lambda x, xa, Ws: modules.NCNRadixNetFunction.apply(x, xa, ALPHA, 0, n, C, 0, None, *Ws))
    kept = {}

    def table(N, batch):
        if not kept:
            kept["t"] = torch.randperm(N, generator=torch.Generator().manual_seed(1)).to(torch.int32).cuda()
            kept["l"] = torch.tensor([N - 3, N // 2][:batch], dtype=torch.int32).cuda()
        return kept["t"], kept["l"] if kind == "lengths" else None

    return (lambda x, xa, Ws: ext.table_stage(x, xa, Ws[0], *table(x.shape[1], x.shape[0]), ALPHA, 0, n, C),
            lambda x, xa, Ws: chunk.FusedLinearChunkNCNFunction.apply(x, xa, Ws[0], *table(x.shape[1], x.shape[0]), ALPHA, "tanh", C, n, 0))


# kind, n, head width, heads, groups, stages; the generic kernels (n = 40 rows of 7 features) save float32 copies
CASES = [("stage", 16, 32, 4, 5, 1), ("stage", 40, 7, 2, 3, 1), ("stage", 5, 24, 2, 7, 1), ("stack", 2, 8, 4, 32, 8),
         ("stack", 4, 32, 2, 9, 3), ("radix", 2, 16, 2, 32, 5), ("radix", 3, 8, 2, 9, 2), ("table", 8, 32, 2, 6, 1),
         ("lengths", 8, 16, 2, 6, 1)]


@pytest.mark.parametrize("upstream", ["both", "y", "ya"])
@pytest.mark.parametrize("types", [(F, F), (H, H), (H, F), (F, H)], ids=["f32", "bf16", "bf16_w32", "f32_w16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s_n%d_e%d" % c[:3])
def test_same_bits_as_the_python_node(P, case, types, upstream):
    kind, n, ec, C, groups, L = case
    native, python = kinds(P, kind, n, C)
    x, xa, Ws, dy, dya = leaves(n, ec, C, groups, L, *types)
    got = []
    for f in (native, python):
        y, ya = f(x, xa, Ws)
        outs, grads = {"both": ([y, ya], [dy, dya]), "y": ([y], [dy]), "ya": ([ya], [dya])}[upstream]
        g = torch.autograd.grad(outs, [x, xa, *Ws], grads)
        assert y.dtype == x.dtype and [t.dtype for t in g[2:]] == [w.dtype for w in Ws] and [t.shape for t in g] == [t.shape for t in (x, xa, *Ws)]
        got.append([y.detach(), ya.detach(), *g])
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [F, H], ids=["f32", "bf16"])
def test_without_gradients_the_same_outputs(P, dtype):
    modules = P[0]
    x, xa, Ws, _, _ = leaves(16, 32, 2, 3, 1, dtype, dtype)
    y, ya = modules.fused_ncn_cuda_v2(x, xa, Ws[0], ALPHA, 0, 16, 2, 0)
    with torch.no_grad():
        z, za = modules.fused_ncn_cuda_v2(x, xa, Ws[0], ALPHA, 0, 16, 2, 0)
    assert y.requires_grad and not z.requires_grad and torch.equal(y, z) and torch.equal(ya, za)
    assert z._base is None   # no second plane is held on to


def test_calls_that_are_left_to_the_python_nodes(P):
    modules, _, _, ext = P
    x, xa, Ws, dy, _ = leaves(4, 8, 2, 8, 2, F, F)
    W = Ws[0]
    args = (ALPHA, 0, 4, 2, 0)

    class Sub(torch.Tensor):
        pass

    bad = [(x.cpu(), xa, W), (x, xa.cpu(), W), (x, xa, W.cpu()), (x.transpose(1, 2), xa.transpose(1, 2), W), (x, xa.to(H), W),
           (x.double(), xa.double(), W), (x, xa, W.double()), (x[0], xa[0], W), (x, xa, W[:-4]), (x.as_subclass(Sub), xa, W),
           (x, xa, None), (x[:0], xa[:0], W), (x.detach().reshape(-1)[2:-30].reshape(1, -1, 16)[:, :28], xa[:1, :28], W)]
    for call in bad:
        assert ext.stage(*call, *args) is None
    for scalars in [("0.9", 0, 4, 2, 0), (ALPHA, 9, 4, 2, 0), (ALPHA, 0, 5, 2, 0), (ALPHA, 0, 4, 3, 0), (ALPHA, 0, 4, 2, -1),
                    (ALPHA, 0, 4, 2, 1 << 70), (ALPHA, 0.0, 4, 2, 0), (ALPHA, 0, True, 2, 0)]:
        assert ext.stage(x, xa, W, *scalars) is None
    assert ext.stage(x, xa, W, ALPHA) is None
    assert ext.stack(x, xa, Ws, *args, 6, 32 << 30, 0) is None            # would look at the free memory
    assert ext.stack(x, xa, [Ws[0], Ws[1].to(H)], *args, 6, 32 << 30, 1 << 30) is None
    assert ext.stack(x.detach(), xa.detach(), [w.detach() for w in Ws], *args, 6, 32 << 30, 1 << 30) is None
    assert ext.radix(x, xa, Ws * 2, *args) is None                          # 4^4 does not divide 32
    # the surface still takes what it took, and refuses what it refused
    y, ya = modules.fused_ncn_cuda_v2(x.detach().transpose(1, 2).contiguous().transpose(1, 2), xa, W, ALPHA, 0, 4, 2, 0)
    assert torch.equal(y, modules.fused_ncn_cuda_v2(x, xa, W, ALPHA, 0, 4, 2, 0)[0])
    with pytest.raises(ValueError, match="n_head must divide E"):
        modules.fused_ncn_cuda_v2(x, xa, W, ALPHA, 0, 4, 3, 0)
    with pytest.raises(TypeError, match="float32 or bfloat16"):
        modules.fused_ncn_cuda_v2(x.double(), xa.double(), W, ALPHA, 0, 4, 2, 0)


def test_hooks_transforms_and_modes(P):
    import torch.autograd.forward_ad as fwAD
    modules = P[0]
    x, xa, Ws, dy, _ = leaves(4, 8, 2, 8, 1, F, F)
    call = lambda x, xa: modules.fused_ncn_cuda_v2(x, xa, Ws[0], ALPHA, 0, 4, 2, 0)
    want = torch.autograd.grad(call(x, xa)[0], [x, xa, Ws[0]], dy)
    # saved tensors go through the caller's hooks
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.cuda()):
        y, ya = call(x, xa)
    assert len(packed) == 3
    for a, b in zip(torch.autograd.grad(y, [x, xa, Ws[0]], dy), want):
        assert torch.equal(a, b)
    # checkpointing, which runs the forward twice
    y = torch.utils.checkpoint.checkpoint(lambda a, b: call(a, b)[0], x, xa, use_reentrant=False)
    for a, b in zip(torch.autograd.grad(y, [x, xa, Ws[0]], dy), want):
        assert torch.equal(a, b)
    # gradients that are no contiguous tensors
    y, _ = call(x, xa)
    for a, b in zip(torch.autograd.grad(y, [x, xa, Ws[0]], dy.transpose(1, 2).contiguous().transpose(1, 2)), want):
        assert torch.equal(a, b)
    # a weight that is changed before the backward is noticed
    y, _ = call(x, xa)
    with torch.no_grad():
        Ws[0].mul_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward(dy)
    # what autograd.Function refuses, the native node does not take
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda a: call(a, a)[0])(x.detach().unsqueeze(0))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda a: call(a, a)[0].sum())(x.detach())
    with fwAD.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        call(fwAD.make_dual(x.detach(), dy), xa)
    # a second derivative does not exist, nor did it
    y, _ = call(x, xa)
    g, = torch.autograd.grad(y, [x], dy, create_graph=True)
    assert not g.requires_grad


# what a hook gives back in place of one saved tensor, and what that raises: from y, ya, W on, or (a stack) the kept activations
UNPACKED = [("on the host", lambda t: t.cpu(), RuntimeError), ("half", lambda t: t.half(), (TypeError, ValueError)),
            ("a part", lambda t: t.flatten()[:-4], ValueError), ("transposed", lambda t: t.transpose(0, -1)[..., :1], ValueError)]


@pytest.mark.parametrize("what,unpack,error", UNPACKED, ids=[u[0].replace(" ", "_") for u in UNPACKED])
@pytest.mark.parametrize("kind,n,L,dtype", [("stage", 16, 1, F), ("stage", 16, 1, H), ("stack", 2, 8, F), ("stack", 2, 8, H), ("radix", 2, 5, F),
                                            ("lengths", 8, 1, F)], ids=lambda v: str(v).replace("torch.", ""))
def test_saved_tensors_that_do_not_come_back_as_they_were(P, kind, n, L, dtype, what, unpack, error):
    """Refused by either node before anything is launched: a kernel would read them past their end."""
    for f in kinds(P, kind, n, 4):
        x, xa, Ws, dy, dya = leaves(n, 8, 4, 32, L, dtype, F)
        saved = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: saved.append(t) or t, lambda t: t):
            f(x, xa, Ws)
        for which in range(len(saved)):
            if kind == "stack" and what == "half" and which == 0:
                continue   # a stack reads weights of any type as float32
            count = iter(range(100))
            hooks = torch.autograd.graph.saved_tensors_hooks(lambda t: (next(count), t), lambda k: unpack(k[1]) if k[0] == which else k[1])
            with hooks:
                y, ya = f(x, xa, Ws)
            with pytest.raises(error):
                torch.autograd.grad([y, ya], [x, xa, *Ws], [dy, dya])


@pytest.mark.parametrize("kind,n,L", [("stage", 16, 1), ("radix", 2, 5)])
def test_saved_tensors_kept_as_bfloat16(P, kind, n, L):
    """A hook that packs float32 into bfloat16: both nodes take the outputs in the type they come back in."""
    native, python = kinds(P, kind, n, 4)
    x, xa, Ws, dy, dya = leaves(n, 8, 4, 32, L, F, F)
    got = []
    for f in (native, python):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.to(H), lambda t: t):
            y, ya = f(x, xa, Ws)
        got.append(torch.autograd.grad([y, ya], [x, xa, *Ws], [dy, dya]))
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_table_that_changes_before_the_backward(P):
    """The table and the lengths are the caller's tensors: what they hold by then is read, if the kernels can read it."""
    ext = P[3]
    x, xa, Ws, dy, dya = leaves(8, 8, 4, 6, 1, F, F)
    N = x.shape[1]
    call = lambda table, lens: ext.table_stage(x, xa, Ws[0], table, lens, ALPHA, 0, 8, 4)
    base = lambda: torch.randperm(N, generator=torch.Generator().manual_seed(1)).to(torch.int32).cuda()
    lengths = lambda: torch.tensor([N - 3, N // 2], dtype=torch.int32).cuda()
    want = torch.autograd.grad(call(base(), lengths()), [x, xa, Ws[0]], [dy, dya])
    for change, error in [(lambda t: t.resize_(4 if t.numel() > 4 else 1), ValueError), (lambda t: setattr(t, "data", t.data.cpu()), RuntimeError),
                          (lambda t: setattr(t, "data", t.data.float()), TypeError), (lambda t: setattr(t, "data", t.data.long()), None)]:
        for which in (0, 1):
            args = [base(), lengths()]
            out = call(*args)
            try:
                change(args[which])
            except RuntimeError:   # torch itself refuses: nothing changed
                continue
            if error is None:
                for a, b in zip(torch.autograd.grad(out, [x, xa, Ws[0]], [dy, dya]), want):
                    assert torch.equal(a, b)
            else:
                with pytest.raises(error):
                    torch.autograd.grad(out, [x, xa, Ws[0]], [dy, dya])


def test_streams_and_threads(P):
    import threading
    modules = P[0]
    x, xa, Ws, dy, _ = leaves(16, 32, 4, 16, 2, F, F)

    def run():
        y, ya = x, xa
        for l, W in enumerate(Ws):
            y, ya = modules.fused_ncn_cuda_v2(y, ya, W, ALPHA, 0, 16, 4, l)
        return [y.detach(), *torch.autograd.grad(y, [x, xa, *Ws], dy)]

    want = run()
    torch.cuda.synchronize()
    out = {}

    def work(k):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(5):
                out[k] = run()
        s.synchronize()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    for k in range(3):
        assert all(torch.equal(a, b) for a, b in zip(out[k], want))
