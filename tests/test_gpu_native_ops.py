"""The native operators (csrc/torch_ops.cpp) where they replace Python dispatch (MI355X only): the stream and the
tensors they launch on, operands they have to copy first, refusals, hooks on saved tensors, graphs of the backward and
gradients that are not asked for."""

from __future__ import annotations

import pytest
import torch

from flowmatching_lthc_amd import ops
from flowmatching_lthc_amd import ops_branch as OB
from flowmatching_lthc_amd import ops_triangular as OT

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def randn(shape, seed, dtype=torch.float32):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(DEV, dtype)


def step(x0, alpha, betas, dzs):
    """The lazy interface in training form: every native node once."""
    x, z = ops.read_with_residual(x0, alpha)
    gammas = ops.lazy_gamma_rounded(alpha, betas, x0.dtype).unbind(0)
    zs, dv = [], []
    for dz, g in zip(dzs, gammas):
        z, zb, d = ops.lazy_workspace_step(z, dz, g, split=True)
        zs.append(zb)
        dv.append(d)
    return [ops.final_accumulate_list(x, dv, betas), *zs]


def inputs(L=3, C=20, G=3):
    x0, alpha = randn((2, 4 * G, 4 * G, C), 0), torch.softmax(randn((C, 16), 1), -1)
    return x0, alpha, [randn((C, 16), 2 + i) for i in range(L)], [randn((2, G * G, C), 9 + i) for i in range(L)]


def leaves(x0, alpha, betas, dzs):
    return [t.detach().requires_grad_() for t in (x0, alpha, *betas, *dzs)]


def run(ls, L=3, **kw):
    outs = step(ls[0], ls[1], ls[2 : 2 + L], ls[2 + L :])
    return outs, torch.autograd.grad([o.square().sum() for o in outs], ls, **kw)


def test_side_stream_and_saved_tensor_hooks():
    print("case native ops: side stream, saved tensor hooks", flush=True)
    data = inputs()
    _, ref = run(leaves(*data))
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _, got = run(leaves(*data))
    side.synchronize()
    for a, b in zip(got, ref):
        assert torch.equal(a, b)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t.cpu(), lambda t: t.to(DEV)):
        outs = step(*(lambda l: (l[0], l[1], l[2:5], l[5:]))(ls := leaves(*data)))
    got = torch.autograd.grad([o.square().sum() for o in outs], ls)
    assert packed
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


def test_operands_that_need_a_copy_and_partial_gradients():
    """Transposed, misaligned and differently typed operands give the plain call's results; a gradient that is not asked
    for changes no other."""
    print("case native ops: strided, misaligned, mixed dtypes", flush=True)
    x0, alpha, betas, dzs = inputs()
    ref = ops.final_accumulate_list(x0, dzs, betas)
    flat = torch.empty(x0.numel() + 1, device=DEV)
    off = flat[1:].view_as(x0).copy_(x0)  # 4 bytes past a 16-byte boundary
    strided = [d.transpose(0, 1).contiguous().transpose(0, 1) for d in dzs]
    assert torch.equal(ops.final_accumulate_list(off, strided, betas), ref)
    mixed = [betas[0].bfloat16(), betas[1], betas[2]]
    assert torch.equal(ops.final_accumulate_list(x0, dzs, mixed), ops.final_accumulate_list(x0, dzs, [mixed[0].float(), *betas[1:]]))
    _, full = run(leaves(x0, alpha, betas, dzs))
    ls = leaves(x0, alpha, betas, dzs)
    ls[0].requires_grad_(False)
    ls[2].requires_grad_(False)
    outs = step(ls[0], ls[1], ls[2:5], ls[5:])
    want = [t for t in ls if t.requires_grad]
    got = torch.autograd.grad([o.square().sum() for o in outs], want)
    for g, t in zip(got, want):
        i = next(j for j, u in enumerate(ls) if u is t)
        assert (g - full[i]).abs().max() <= 1e-5 * full[i].abs().max()


def test_graph_of_the_backward_through_the_read():
    """create_graph: the read's gradient is a write, which is differentiable; its second derivative is the eager one."""
    print("case native ops: create_graph", flush=True)
    x, w = randn((1, 8, 8, 8), 0).requires_grad_(), randn((8, 16), 1)
    cells = lambda t: t.view(1, 2, 4, 2, 4, 8).permute(0, 1, 3, 2, 4, 5).reshape(1, 4, 16, 8)  # noqa: E731
    second = []
    for read in (lambda t: ops.local_write_traceable(t, w), lambda t: (cells(t) * w.t()).sum(2)):
        (g,) = torch.autograd.grad(read(x).pow(3).sum(), x, create_graph=True)
        (h,) = torch.autograd.grad(g.square().sum(), x)
        second.append(h)
    assert (second[0] - second[1]).abs().max() <= 1e-5 * second[1].abs().max()


def batched_cases():
    z, a, m, w = randn((2, 9, 24), 0), randn((2, 9, 24), 1), randn((2, 9, 24), 2), randn((24,), 3)
    gate, shift, scale = (randn((2, 24), 4 + i) for i in range(3))
    qkv, n0, n1, table = randn((2, 6, 3, 2, 64), 7), randn((64,), 8), randn((64,), 9), randn((6, 64), 10)
    x0, alpha, betas, dzs = inputs(12)
    return {
        "norm_modulate": (lambda *t: ops.norm_modulate(*t, 1e-6)[0], (z, w, shift, scale)),
        "gate_add_norm_modulate": (lambda *t: OB.gate_add_norm_modulate(*t, 1e-6), (z, a, gate, w, shift, scale)),
        "gate_residual": (OB.gate_residual, (a, gate, m)),
        "swiglu": (OB.swiglu, (randn((5, 48), 11),)),
        "qk_norm_rope": (lambda *t: OB.qk_norm_rope(*t, table, table, 1e-6), (qkv, n0, n1)),
        "bases": (OT.all_base_b4_12_split_traceable, (x0, torch.stack(betas[:3]))),
        "materialise dz": (lambda *d: ops.final_accumulate_b4_12_traceable(x0, *d, *betas), tuple(dzs)),
        "materialise beta": (lambda *b: ops.final_accumulate_b4_12_traceable(x0, *dzs, *b), tuple(betas)),
        "read": (ops.read_with_residual, (x0, alpha)),
        "step": (lambda *t: ops.lazy_workspace_step(*t, True), (dzs[0], dzs[1], randn((20,), 12))),
    }


@pytest.mark.parametrize("name", ["norm_modulate", "gate_add_norm_modulate", "gate_residual", "swiglu", "qk_norm_rope",
                                  "bases", "materialise dz", "materialise beta", "read", "step"])  # fmt: skip
def test_batched_gradients(name):
    """is_grads_batched gives each sample's own gradients, bit for bit (the same kernels, once per sample)."""
    print(f"case native ops: batched gradients of {name}", flush=True)
    f, tensors = batched_cases()[name]
    ls = [t.detach().requires_grad_() for t in tensors]
    outs = f(*ls)
    outs = [outs] if isinstance(outs, torch.Tensor) else list(outs)
    grads = [randn((3, *o.shape), 20 + i) for i, o in enumerate(outs)]
    got = torch.autograd.grad(outs, ls, grads, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        for a, b in zip(got, torch.autograd.grad(outs, ls, [g[i] for g in grads], retain_graph=True)):
            assert torch.equal(a[i], b)


def test_refusals():
    print("case native ops: refusals", flush=True)
    x, w = randn((1, 8, 8, 8), 0), randn((8, 16), 1)
    bad = [
        (lambda: ops.local_write_traceable(x.cpu(), w), "no CPU fallback"),
        (lambda: ops.local_write_traceable(x, w.cpu()), "all tensors must be on"),
        (lambda: ops.local_write_traceable(x.double(), w), "unsupported dtype"),
        (lambda: ops.local_write_traceable(x[:, :6, :6], w), "cell side"),
        (lambda: ops.local_write_traceable(x, w[:, :8]), r"weight must be \[8,16\]"),
        (lambda: ops.local_read_traceable(randn((1, 5, 8), 2), w), "not a square"),
        (lambda: ops.final_accumulate_list(x, [], []), "expected 1..48"),
        (lambda: ops.lazy_workspace_update(x, x, w[0]), r"gamma must be \[8\]"),
        (lambda: OB.swiglu(randn((2, 24), 3)), "2F with F"),
        (lambda: OB.gate_residual(randn((1, 2, 4), 3), randn((1, 4), 4), randn((1, 2, 4), 5)), "C % 8 == 0"),
        (lambda: OT.triangular_accumulate_list(randn((1, 4, 8), 2), [], w[:1, :8]), "depth 0 outside"),
    ]
    for f, text in bad:
        with pytest.raises(ValueError, match=text):
            f()
    with pytest.raises(RuntimeError):  # functorch over an autograd node, as before
        torch.func.grad(lambda t: OB.swiglu(t).sum())(randn((2, 16), 3))


def test_backward_operators_check_what_they_read():
    print("case native ops: refusals of the backward operators", flush=True)
    z, rows, row = randn((2, 3, 8), 6), randn((2, 8), 7), randn((8,), 8)
    ganm = lambda gate=rows, scale=rows, weight=row: OB.gate_add_norm_modulate_backward(  # noqa: E731
        None, z, z, z, gate, weight, scale, 1e-6
    )
    w, ggamma = randn((8, 16), 1), randn((2, 8), 9)
    bad = [
        (lambda: ganm(gate=rows[:1]), r"gate must be \[2, 8\]"),
        (lambda: ganm(gate=rows.bfloat16()), "gate must be .* Float"),
        (lambda: ganm(scale=rows[:, :4]), r"scale must be \[2, 8\]"),
        (lambda: ganm(scale=rows.double()), "scale must be .* Float"),
        (lambda: ganm(weight=row[:4]), r"weight must be \[8\]"),
        (lambda: ops.norm_modulate_backward(z[:1], z, row, rows, randn((6,), 1)), r"grad must be \[2, 3, 8\]"),
        (lambda: ops.norm_modulate_backward(z, z, row, rows, randn((5,), 1)), "inv must hold 6"),
        (lambda: ops.lazy_gamma_rounded_backward(ggamma, w, [], True, True), "L betas"),
        (lambda: ops.lazy_gamma_rounded_backward(ggamma, w, [w, w[:4]], True, True), "L betas"),
        (lambda: ops.lazy_gamma_rounded_backward(ggamma[:1], w, [w, w], True, True), r"grad must be \[2, 8\]"),
        (lambda: OT.ws_accumulate_backward(z, [z], ggamma, 2, True), "expected 2 dz, got 1"),
        (lambda: OT.ws_accumulate_backward(z, [z, z[:1]], ggamma, 2, True), "does not match grad"),
        (lambda: OT.ws_accumulate_backward(z, [], ggamma[:1], 2, True), r"gamma must be \[>= 2, 8\]"),
        (lambda: OT.ws_accumulate_backward(z, [], ggamma, 25, True), "depth 25 outside"),
    ]
    for f, text in bad:
        with pytest.raises(ValueError, match=text):
            f()
