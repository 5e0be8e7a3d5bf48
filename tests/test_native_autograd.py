"""The native autograd nodes (csrc/torch_ops.cpp) on CPU tensors: plain-torch kernels stand in for the HIP ones while a
test runs, so that what autograd sees of the nodes can be checked without a GPU."""

from __future__ import annotations

import math

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx

from flowmatching_lthc_amd import ops
from flowmatching_lthc_amd import ops_branch as OB
from flowmatching_lthc_amd import ops_triangular as OT


def cells(x):
    """[B, 4G, 4G, C] -> [B, G*G, 16, C]."""
    B, H, _, C = x.shape
    G = H // 4
    return x.view(B, G, 4, G, 4, C).permute(0, 1, 3, 2, 4, 5).reshape(B, G * G, 16, C)


def read(x, w):
    return (cells(x) * w.t()).sum(2)


def write(z, w):
    B, M, C = z.shape
    G = math.isqrt(M)
    x = (z[:, :, None] * w.t()).view(B, G, G, 4, 4, C)
    return x.permute(0, 1, 3, 2, 4, 5).reshape(B, 4 * G, 4 * G, C)


def weight_grad(high, low):
    return (cells(high) * low[:, :, None]).sum((0, 1)).t().contiguous()


def all_base_backward(x, grads, alphas, need_x, need_alpha):
    empty = x.new_empty(0)
    gx = sum(map(write, grads, alphas)) if need_x else empty
    return gx, torch.stack([weight_grad(x, g) for g in grads]) if need_alpha else empty


def recur_backward(g, dz, gamma, add=None):
    return gamma * g + (0 if add is None else add), (g * dz).sum((0, 1))


KERNELS = {
    "local_write_traceable": read,
    "local_read_traceable": write,
    "local_read_add_traceable": lambda z, w, x: x + write(z, w),
    "local_weight_grad_traceable": weight_grad,
    "lazy_workspace_update": lambda z, dz, gamma: z + gamma * dz,
    "lazy_workspace_update_backward": recur_backward,
    "lazy_workspace_update_backward_sum": lambda g, b, dz, gamma, add=None: (g + b, *recur_backward(g + b, dz, gamma, add)),
    "all_base_b4_12_split_traceable": lambda x, a: [read(x, w) for w in a],
    "all_base_backward": all_base_backward,
    "final_accumulate_b4_12_traceable": lambda x, *rest: x + sum(map(write, rest[:12], rest[12:])),
    "all_base_b4_12_grad_x": lambda g, a: sum(map(write, g, a)),
    "all_base_b4_12_split_grad_alpha": lambda x, g: torch.stack([weight_grad(x, t) for t in g]),
    "final_accumulate_b4_12_grad_dz_ptr": lambda g, *betas: torch.stack([read(g, b) for b in betas]),
    "final_accumulate_b4_12_grad_beta_ptr": lambda g, *dzs: torch.stack([weight_grad(g, d) for d in dzs]),
    "final_accumulate_list_grad_dz": lambda g, betas: [read(g, b) for b in betas],
    "final_accumulate_list_grad_beta": lambda g, dzs: torch.stack([weight_grad(g, d) for d in dzs]),
    "gate_residual": OB.gate_residual_eager,
    "gate_residual_backward": lambda g, gate, m: ((g * m).sum(1), g * gate.unsqueeze(1)),
}


@pytest.fixture(autouse=True)
def cpu_kernels():
    lib = torch.library.Library("jit_thc", "IMPL")
    for name, fn in KERNELS.items():
        lib.impl(name, fn, "CPU")
    yield
    lib._destroy()


def randn(shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed))


def leaf(shape, seed):
    return randn(shape, seed).requires_grad_()


# ---------------------------------------------------------------------------
# outputs that alias an input or another output
# ---------------------------------------------------------------------------
def open_interface():
    leaves = [leaf((2, 8, 8, 4), 0), leaf((4, 16), 1)]
    return leaves, ops.read_with_residual(*leaves)


def workspace_step(split):
    leaves = [leaf((2, 4, 4), 2), leaf((2, 4, 4), 3), leaf((4,), 4)]
    return leaves, ops.lazy_workspace_step(*leaves, split)


ALIASES = [(open_interface, (), 0), (workspace_step, (False,), 1), *((workspace_step, (True,), i) for i in range(3))]


@pytest.mark.parametrize("node,args,i", ALIASES)
def test_in_place_change_of_an_aliasing_output_is_refused(node, args, i):
    """These outputs share their storage with saved inputs or with each other: autograd has to see a change of one, or
    the backward runs on changed data."""
    leaves, outs = node(*args)
    with pytest.raises(RuntimeError, match="modified inplace"):
        outs[i].mul_(2)
        torch.autograd.grad(sum(o.sum() for o in outs), leaves)


def test_aliases_share_the_version_counter_without_recording():
    x, w, dz = randn((2, 8, 8, 4), 0), randn((4, 16), 1), randn((2, 4, 4), 3)
    version = x._version, dz._version
    xo, _ = ops.read_with_residual(x, w)
    dzo = ops.lazy_workspace_step(randn((2, 4, 4), 2), dz, randn((4,), 4), True)[2]
    xo.mul_(2)
    dzo.mul_(2)
    assert (x._version - version[0], dz._version - version[1]) == (1, 1)


def test_interface_nodes_give_the_gradients_of_the_plain_sequence():
    x, w, dz, gamma = leaf((2, 8, 8, 4), 0), leaf((4, 16), 1), leaf((2, 4, 4), 3), leaf((4,), 4)

    def native(x, w, dz, gamma):
        x, z = ops.read_with_residual(x, w)
        z, branch, d = ops.lazy_workspace_step(z, dz, gamma, split=True)
        return [x, z, branch, d]

    def plain(x, w, dz, gamma):
        z = read(x, w) + gamma * dz
        return [x, z, z, dz]

    got, want = (
        torch.autograd.grad([(o * o).sum() for o in f(x, w, dz, gamma)], [x, w, dz, gamma]) for f in (native, plain)
    )
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5)


# ---------------------------------------------------------------------------
# graphs of the backward
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("C", [8, 2056])  # within the backward kernel's widths, and beyond
def test_second_derivative_of_gate_residual(C):
    """create_graph: the gradients of the gate and m are products of both, as in the plain sequence."""
    leaves = [leaf((2, 4, C), 0), leaf((2, C), 1), leaf((2, 4, C), 2)]
    results = []
    for f in (OB.gate_residual, OB.gate_residual_eager):
        first = torch.autograd.grad(f(*leaves).pow(2).sum(), leaves, create_graph=True)
        results.append([*first, *torch.autograd.grad(sum(g.square().sum() for g in first), leaves)])
    for a, b in zip(*results):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-4)


# ---------------------------------------------------------------------------
# batched gradients
# ---------------------------------------------------------------------------
def bases(want):
    x, alphas = leaf((2, 8, 8, 4), 0), leaf((3, 4, 16), 1)
    return OT.all_base_b4_12_split_traceable(x, alphas), [x, alphas][want]


def materialise(want):
    x, dzs, betas = randn((2, 8, 8, 4), 0), [randn((2, 4, 4), 1 + i) for i in range(12)], [randn((4, 16), 13 + i) for i in range(12)]
    leaves = [t.requires_grad_() for t in (dzs, betas)[want]]
    return [ops.final_accumulate_b4_12_traceable(x, *dzs, *betas)], leaves


def gate(want):
    leaves = [leaf((2, 4, 8), 0), leaf((2, 8), 1), leaf((2, 4, 8), 2)]
    return [OB.gate_residual(*leaves)], leaves[want]


@pytest.mark.parametrize("node,want", [(bases, slice(0, 2)), (bases, slice(0, 1)), (materialise, 0), (materialise, 1), (gate, slice(0, 3))])
def test_batched_gradients_are_those_of_each_sample(node, want):
    outs, leaves = node(want)
    grads = [randn((3, *o.shape), 40 + i) for i, o in enumerate(outs)]
    got = torch.autograd.grad(outs, leaves, grads, is_grads_batched=True, retain_graph=True)
    each = [torch.autograd.grad(outs, leaves, [g[i] for g in grads], retain_graph=True) for i in range(3)]
    vmapped = torch.vmap(lambda *g: torch.autograd.grad(outs, leaves, g, retain_graph=True))(*grads)
    for a, v, b in zip(got, vmapped, zip(*each)):
        torch.testing.assert_close(a, torch.stack(b), rtol=1e-6, atol=1e-5)
        torch.testing.assert_close(v, a, rtol=1e-6, atol=1e-5)


# ---------------------------------------------------------------------------
# devices
# ---------------------------------------------------------------------------
def meta(*shape, dtype=torch.float32):
    return torch.empty(shape, device="meta", dtype=dtype, requires_grad=True)


def meta_cases():
    x, w, z, dz, row, rows = meta(2, 8, 8, 8), meta(8, 16), meta(2, 4, 8), meta(2, 4, 8), meta(8), meta(2, 8)
    qkv, tables = meta(2, 64, 3, 2, 64, dtype=torch.bfloat16), meta(64, 64)
    norm, stack = meta(64), meta(3, 8, 16)
    twelve = [meta(2, 4, 8) for _ in range(12)], [meta(8, 16) for _ in range(12)]
    qk = (qkv, norm, norm, tables.detach(), tables.detach(), 1e-6)
    return {
        "read": (ops.local_write_traceable, (x, w)),
        "write": (ops.local_read_traceable, (z, w)),
        "write_add": (ops.local_read_add_traceable, (z, w, x)),
        "read_with_residual": (ops.read_with_residual, (x, w)),
        "step": (ops.lazy_workspace_step, (z, dz, row, True)),
        "update": (ops.lazy_workspace_update, (z, dz, row)),
        "final_list": (lambda x, d, b: ops.final_accumulate_list(x, [d], [b]), (x, dz, w)),
        "final_12": (lambda x, *rest: ops.final_accumulate_b4_12_traceable(x, *rest), (x, *twelve[0], *twelve[1])),
        "gamma_rounded": (lambda a, b: ops.lazy_gamma_rounded(a, [b], torch.bfloat16), (w, meta(8, 16))),
        "bases": (OT.all_base_b4_12_split_traceable, (x, stack)),
        "tri_list": (lambda z, d, g: OT.triangular_accumulate_list(z, [d], g), (z, dz, meta(1, 8))),
        "tri_12": (OT.triangular_accumulate_b4_12_ptr_traceable, (z, *twelve[0], meta(12, 8))),
        "tri_active": (OT.triangular_accumulate_b4_12_ptr_active_traceable_ops[4], (z, *twelve[0], meta(12, 8))),
        "norm_modulate": (ops.norm_modulate, (z, row, rows, rows, 1e-6)),
        "qk_norm_rope": (OB.qk_norm_rope, qk),
        "attention": (OB.qk_norm_rope_attention, qk),
        "swiglu": (OB.swiglu, (meta(2, 16),)),
        "gate_add_norm_modulate": (OB.gate_add_norm_modulate, (z, dz, rows, row, rows, rows, 1e-6)),
        "gate_residual": (OB.gate_residual, (z, rows, dz)),
    }


@pytest.mark.parametrize("name", meta_cases())
def test_gradients_of_meta_tensors(name):
    """Shapes can be propagated through forward and backward without a device, as through torch's own operators."""
    f, args = meta_cases()[name]
    outs = f(*args)
    outs = [outs] if isinstance(outs, torch.Tensor) else list(outs)
    leaves = list({id(a): a for a in args if isinstance(a, torch.Tensor) and a.requires_grad}.values())
    grads = torch.autograd.grad(outs, leaves, [torch.empty_like(o) for o in outs], allow_unused=True)
    assert any(g is not None for g in grads)
    for g, a in zip(grads, leaves):
        assert g is None or (g.shape, g.dtype, g.device) == (a.shape, a.dtype, a.device)


# ---------------------------------------------------------------------------
# tracing
# ---------------------------------------------------------------------------
def trace(op, tensors, diff, **kw):
    """The graph of op's gradients for its first `diff` operands, traced on fake tensors."""

    def step(grads, *tensors):
        leaves = [t.detach().requires_grad_(i < diff) for i, t in enumerate(tensors)]
        outs = op(*leaves, **kw)
        return torch.autograd.grad(outs, leaves[:diff], grads)

    outs = op(*(t.to("meta") for t in tensors), **kw)
    grads = [torch.zeros(o.shape, dtype=o.dtype) for o in (outs if isinstance(outs, tuple) else (outs,))]
    graph = make_fx(step, tracing_mode="fake")(grads, *tensors).graph
    (out,) = [n for n in graph.nodes if n.op == "output"]
    for got, want in zip(out.args[0], tensors):
        assert got.meta["val"].shape == want.shape and got.meta["val"].dtype == want.dtype
    return [n for n in graph.nodes if n.op == "call_function"]


def traced_cases():
    z, rows, qkv, w = randn((2, 64, 8), 0).bfloat16(), randn((2, 8), 1).bfloat16(), randn((2, 64, 3, 2, 64), 2).bfloat16(), randn((64,), 3)
    table = randn((64, 64), 4)
    return {
        "qk_norm_rope": (OB.qk_norm_rope, (qkv, w, w, table, table), 3, {"eps": 1e-6}),
        "qk_norm_rope_attention": (OB.qk_norm_rope_attention, (qkv, w, w, table, table), 3, {"eps": 1e-6}),
        "swiglu": (OB.swiglu, (randn((4, 32), 5).bfloat16(),), 1, {}),
        "gate_add_norm_modulate": (OB.gate_add_norm_modulate, (z, z, rows, randn((8,), 6), rows, rows), 6, {"eps": 1e-6}),
    }


@pytest.mark.parametrize("name", traced_cases())
def test_traced_branch_backward_is_the_eager_sequence(name):
    """A traced graph holds the plain sequence's gradients, whose intermediates the compiler keeps in fp32, and not the
    backward kernel, which rounds them where eager does.  The attention's products are fp32 ones (scores and output again, and four gradients)."""
    op, tensors, diff, kw = traced_cases()[name]
    nodes = trace(op, tensors, diff, **kw)
    names = {str(n.target) for n in nodes}
    assert f"jit_thc.{name}_backward.default" not in names and {n for n in names if "jit_thc" in n} <= {f"jit_thc.{name}.default"}
    products = [n for n in nodes if n.target in (torch.ops.aten.bmm.default, torch.ops.aten.mm.default)]
    assert len(products) == (6 if name == "qk_norm_rope_attention" else 0)
    assert all(n.meta["val"].dtype == torch.float32 for n in products)


def test_fake_gradients_are_contiguous():
    """The backward kernels return contiguous gradients whatever the strides of their operands; so do their fakes, whose
    strides a compiled graph asserts."""
    z, rows, w = meta(4, 2, 8).transpose(0, 1), meta(2, 8), meta(8)
    x0, qkv = meta(2, 8, 8, 8).permute(0, 2, 1, 3), meta(4, 2, 3, 2, 64).transpose(0, 1)
    q, n, table = meta(2, 4, 2, 64), meta(64), meta(4, 64)
    outs = [
        *OB.qk_norm_rope_backward(q, q, qkv, n, n, table, table, 1e-6),
        *OB.qk_norm_rope_attention_backward(q, qkv, n, n, table, table, 1e-6),
        OB.swiglu_backward(meta(2, 4, 4), z),
        *OB.gate_add_norm_modulate_backward(None, z, z, z, rows, w, rows, 1e-6),
        *OB.gate_residual_backward(z, rows, z),
        *OT.all_base_backward(x0, [z], meta(1, 8, 16), True, True),
    ]
    assert all(o.is_contiguous() for o in outs)
