"""Workloads of the NCN layer, from the smallest call to the deepest stack, for timing the framework's public surface.

A case is a plain dict; `listed()` names the fixed ones and `draw()` makes one more of the same ranges.  `prepare()`
builds what a program holds before the call (activations, weights, the net object) and `run()` is one pass of it:

  op = "train"    net(x, xa), then the gradients of y: the reference script's step (yi.backward(dyi)).  Gradients of the
                  inputs and of every stage's weights come back beside y, ya.  fused = False is the drop-in surface
                  (one autograd node per stage), fused = True the whole stack as one node.
  op = "infer"    net(x, xa) without gradients.
  op = "inverse"  the inputs of a whole stack from its outputs (float32, as an invertible net is used).
  op = "table"    stages grouped by tables with one context length per batch entry, trained: fused_chunk_linear_ncn.
  op = "radix"    a net on the radix-n digit grouping, trained.

Sizes are those of bench.py's configurations and of the tests, or lie between them.  alpha = 0.9 and tanh throughout,
x ~ N(0, 1), xa = 0 where a stack starts (the reference script's start), W ~ N(0, 1/n) times the configuration's scale.
"""
import math

import torch

from ncn_cuda_amd import NCNNetTestCuda, ncn_cuda_module
from ncn_cuda_amd.chunk_linear import fused_chunk_linear_ncn, radix_group_table, stride_group_table

ALPHA = 0.9

# Float operations per element and step (an FMA is two, exp2 and reciprocal one each): row sum, z, two for xa, x, and
# the +1 forward; the backward adds the vector-Jacobian product and the weight gradient.
FLOPS_FORWARD = 13.0
FLOPS_BACKWARD = 28.0


def _case(name, op, batch, N, E, heads, n, stages, dtype="f32", fused=False, w_scale=1.0, table="none"):
    case = dict(op=op, batch=batch, N=N, E=E, heads=heads, n=n, stages=stages, dtype=dtype, fused=fused, w_scale=w_scale,
                table=table)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # One sequence of BASELINE's smallest configuration as a stack in one node: launches and host time are all of it.
        _case("train_one_sequence", "train", 1, 256, 32, 4, 2, 8, fused=True),
        # The reference's own script (grad_test_bench.py:22-32) through the drop-in surface: few groups of 32 rows.
        _case("train_script", "train", 4, 256, 128, 4, 32, 3),
        # A layer of medium size with groups of four rows, whole stack in one node.
        _case("train_groups_of_4", "train", 32, 1024, 128, 4, 4, 5, fused=True),
        # Groups of eight rows, float32, drop-in surface, and the inverse of the same stack (the invertible net's use).
        _case("train_groups_of_8", "train", 64, 2048, 128, 4, 8, 4, w_scale=0.1),
        _case("inverse_groups_of_8", "inverse", 64, 2048, 128, 4, 8, 4, w_scale=0.1),
        # The headline workload: bfloat16 activations and weights, groups of 16 rows, drop-in surface.
        _case("train_headline", "train", 128, 4096, 128, 4, 16, 3, dtype="bf16"),
        # The same layer in inference on a serving batch.
        _case("infer_bf16", "infer", 16, 4096, 128, 4, 16, 3, dtype="bf16"),
        # The deep stack: groups of two rows, 13 stages, one node.
        _case("train_deep", "train", 128, 8192, 128, 4, 2, 13, fused=True),
        # bfloat16 activations in a stack of small groups, one node.
        _case("train_bf16_groups_of_4", "train", 64, 2048, 128, 4, 4, 6, dtype="bf16", fused=True),
        # Ragged sequences with a digit table: every batch entry has its own length.
        _case("train_ragged_table", "table", 32, 4096, 128, 4, 16, 3, dtype="bf16", table="radix"),
        # Sizes that are no powers of two anywhere: groups of five rows, an odd number of them, heads of 40 features.
        _case("train_odd_sizes", "train", 16, 1005, 160, 4, 5, 4),
        # The deep stack's tensors (fewer sequences) on the radix-2 digit grouping.
        _case("train_radix_2", "radix", 32, 8192, 128, 4, 2, 13, fused=True),
    ]


# What one pass of a drawn case may hold: elements of an activation tensor, elements x stages, and elements x stages x
# steps.  Below the largest listed cases (1.3e8, 1.7e9, 3.5e9); the odd shapes have a bound of their own on the last.
_MAX_ELEMENTS, _MAX_STAGES, _MAX_STEPS, _MAX_ODD_STEPS = 5.0e7, 4.0e8, 2.0e9, 5.5e7


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the kinds of listed() with sizes spread over the whole range, odd ones among them."""
    while True:
        kind = rng.choice(["fused", "fused", "per_stage", "per_stage", "infer", "inverse", "table", "odd", "radix"])
        dtype = rng.choice(["f32", "bf16"])
        batch = _log_int(rng, 1, 128)
        heads = rng.choice([1, 2, 4, 4, 8])
        ec = rng.choice([8, 16, 32, 32, 64])
        w_scale = rng.choice([0.1, 1.0])
        if kind in ("fused", "per_stage", "infer", "inverse", "table"):
            n = rng.choice([2, 4]) if kind == "fused" else rng.choice([4, 8, 8, 16, 16, 32])
            if n == 32 and ec == 64:
                ec = 32
            groups = _log_int(rng, 8, 8192 // n) if rng.random() < 0.4 else 2 ** rng.randint(3, int(math.log2(8192 // n)))
            stages = rng.randint(3, 12 if n == 2 else 8 if n == 4 else 4)
            if kind == "inverse":
                dtype, n = "f32", min(n, 8)
                stages = min(stages, 4)
            case = _case(None, {"fused": "train", "per_stage": "train"}.get(kind, kind), batch, n * groups, ec * heads, heads,
                         n, stages, dtype, kind == "fused", w_scale, "stride" if kind == "table" else "none")
        elif kind == "odd":
            n = rng.choice([3, 5, 6, 7, 10, 12, 20])
            ec = rng.choice([3, 5, 10, 12, 20, 24, 40, 48, 56])
            case = _case(None, "train", batch, n * _log_int(rng, 8, 4096 // n), ec * heads, heads, n, rng.randint(2, 4), dtype,
                         False, w_scale)
        else:
            n = rng.choice([2, 4])
            levels = rng.randint(4, 12 if n == 2 else 6)
            case = _case(None, "radix", batch, n ** levels * rng.randint(1, 3), ec * heads, heads, n, levels, "f32", True,
                         w_scale)
        elements = case["batch"] * case["N"] * case["E"]
        steps = elements * case["stages"] * case["n"]
        if case["N"] <= 8192 and 8000 <= elements <= _MAX_ELEMENTS and elements * case["stages"] <= _MAX_STAGES and \
                steps <= (_MAX_ODD_STEPS if kind == "odd" else _MAX_STEPS):
            return case


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    shape = (case["batch"], case["N"], case["E"])
    op, n, heads, L = case["op"], case["n"], case["heads"], case["stages"]

    def randn(*size, scale=1.0):
        return (torch.randn(*size, generator=gen, device=dev) * scale).to(dtype)

    state = dict(op=op, n=n, heads=heads, stages=L)
    x = randn(*shape)
    Ws = [randn(2 * case["E"], scale=case["w_scale"] / math.sqrt(n)) for _ in range(L)]
    if op == "inverse":
        # outputs of the stack on inputs as they come from earlier layers: what an invertible net hands back
        state["W"] = torch.stack(Ws)
        state["y"], state["ya"] = ncn_cuda_module.forward_stages(x, randn(*shape), state["W"], ALPHA, 0, n, heads, 0, L)
        return state
    state.update(x=x, xa=torch.zeros(shape, dtype=dtype, device=dev), Ws=Ws)
    if op == "table":
        if case["table"] == "radix":
            levels = 1
            while n ** (levels + 1) <= case["N"] and case["N"] % n ** (levels + 1) == 0:
                levels += 1
            state["tables"] = [radix_group_table(case["N"], n, l % levels, device=dev) for l in range(L)]
        else:
            state["tables"] = [stride_group_table(case["N"], n, l, device=dev) for l in range(L)]
        # lengths between half of the sequence and all of it
        state["lens"] = torch.randint(case["N"] // 2, case["N"] + 1, (case["batch"],), generator=gen, device=dev).to(torch.int32)
    else:
        state["net"] = NCNNetTestCuda(ALPHA, "tanh", n, heads, L, Ws, fuse_stages=case["fused"],
                                      grouping="radix" if op == "radix" else "stride")
    if op != "infer":
        state["dy"] = randn(*shape)
        for t in (state["x"], state["xa"], *Ws):
            t.requires_grad_(True)
    return state


def run(state):
    op = state["op"]
    if op == "inverse":
        return ncn_cuda_module.inverse_stages(state["y"], state["ya"], state["W"], ALPHA, 0, state["n"], state["heads"], 0,
                                              state["stages"])
    x, xa, Ws = state["x"], state["xa"], state["Ws"]
    if op == "infer":
        with torch.no_grad():
            return state["net"](x, xa)
    if op == "table":
        y, ya = x, xa
        for l, (W, table) in enumerate(zip(Ws, state["tables"])):
            y, ya = fused_chunk_linear_ncn(y, ya, W, table, state["lens"], ALPHA, "tanh", state["heads"], state["n"], l)
    else:
        y, ya = state["net"](x, xa)
    grads = torch.autograd.grad(y, [x, xa, *Ws], state["dy"])
    return [y.detach(), ya.detach(), *grads]


def work(case):
    """Bytes: inputs once, outputs once (x, xa -> y, ya, and for training dy -> dx, dxa, and the weights).
    Operations: the recurrence's own."""
    elements = float(case["batch"]) * case["N"] * case["E"]
    size = 2 if case["dtype"] == "bf16" else 4
    train = case["op"] in ("train", "table", "radix")
    weights = 2.0 * case["E"] * case["stages"] * size
    steps = elements * case["stages"] * case["n"]
    return {"bytes": elements * size * (7 if train else 4) + weights * (2 if train else 1),
            "flops": steps * (FLOPS_FORWARD + (FLOPS_BACKWARD if train else 0.0))}


def tolerance(case):
    """About four times the errors measured against float64 over the listed and some drawn cases.  bfloat16: rounding of
    the stored values, once per stage where every stage stores them (worst 3.0e-3), once where a stack is one node
    (1.8e-3).  float32: rounding of the sums (outputs 2.9e-7, gradients 1.0e-6), which the reversible passes amplify by
    1/m = 1/0.9 at every step that they undo without reading a stored value (up to 3.4e-7 per unit, 4.8e-7 for groups of
    32 rows)."""
    if case["dtype"] == "bf16":
        return {"rel": 7.2e-3 if case["fused"] else 1.2e-2}
    if case["op"] == "infer":
        return {"rel": 1.2e-6}
    undone = case["n"] * (case["stages"] if case["op"] == "inverse" else 1)
    if case["fused"]:
        undone = min(26, case["n"] * case["stages"])
    return {"rel": max(4.0e-6, (1.9e-6 if case["n"] > 20 else 1.3e-6) * 0.9 ** -undone)}
