"""GPU parity of the branch ops' backward kernels (MI355X only): each gradient against autograd of the same function
in float64, no further from it than the eager 16-bit sequence's gradient (x 1.1 for the draw), at the sizes where each
kernel's tiles, lanes and partial rows end."""

from __future__ import annotations

import pytest
import torch
from torch.utils.flop_counter import FlopCounterMode

from flowmatching_lthc_amd import model as M
from flowmatching_lthc_amd import ops
from flowmatching_lthc_amd import ops_branch as OB

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-300)).item()


def qk_exact(x, w, cos, sin):
    n = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w
    rot = torch.stack((-n[..., 1::2], n[..., 0::2]), -1).flatten(-2)
    return n * cos[:, None] + rot * sin[:, None]


# N: one wavefront's queries twice over (64), odd and full numbers of 64-token blocks; H = 1 and odd
@pytest.mark.parametrize("N,H", [(64, 1), (128, 3), (192, 2), (256, 5)])
@pytest.mark.parametrize("dtype,tdt,wdt", [
    (torch.bfloat16, torch.bfloat16, torch.float32),
    (torch.bfloat16, torch.float32, torch.bfloat16),
    (torch.float16, torch.float16, torch.float16),
])  # fmt: skip
def test_attention_backward(N, H, dtype, tdt, wdt):
    print(f"case attention backward N={N} H={H} {dtype} {tdt} {wdt}", flush=True)
    gen = torch.Generator().manual_seed(N + H)
    qkv = (torch.randn((3, N, 3, H, 64), generator=gen) * 2).to(DEV, dtype)
    w0, w1 = ((torch.randn(64, generator=gen) * 0.2 + 1).to(DEV, wdt) for _ in range(2))
    th = torch.rand((N, 64), generator=gen) * 6.2831853
    cos, sin = th.cos().to(DEV, tdt), th.sin().to(DEV, tdt)
    g = (torch.randn((3, N, H, 64), generator=gen) * 0.1).to(DEV, dtype)
    leaves = [t.double().requires_grad_() for t in (qkv, w0, w1)]
    c, s = cos.to(dtype).double(), sin.to(dtype).double()
    q, k = qk_exact(leaves[0][:, :, 0], leaves[1], c, s), qk_exact(leaves[0][:, :, 1], leaves[2], c, s)
    q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, leaves[0][:, :, 2]))
    o = torch.matmul(torch.softmax(torch.matmul(q, k.transpose(-1, -2).contiguous()) / 8, -1), v).transpose(1, 2)
    exact = torch.autograd.grad(o, leaves, g.double())
    got = []
    for fn in (OB.qk_norm_rope_attention, OB.qk_norm_rope_attention_eager):
        leaves = [t.clone().requires_grad_() for t in (qkv, w0, w1)]
        got.append(torch.autograd.grad(fn(*leaves, cos, sin, 1e-6), leaves, g))
    for name, ours, eager, ref in zip(("qkv", "q weight", "k weight"), *got, exact):
        assert ours.dtype == eager.dtype and ours.shape == eager.shape
        assert rel(ours, ref) <= 1.1 * rel(eager, ref), f"{name}: {rel(ours, ref):.2e}, eager {rel(eager, ref):.2e}"
    # a strided gradient, an empty batch, and a batch of gradients under vmap
    leaves = [t.clone().requires_grad_() for t in (qkv, w0, w1)]
    o = OB.qk_norm_rope_attention(*leaves, cos, sin, 1e-6)
    gs = torch.stack((g, g), -1)[..., 0]
    for a, b in zip(torch.autograd.grad(o, leaves, gs, retain_graph=True), got[0]):
        assert torch.equal(a, b)
    (gb,) = torch.autograd.grad(o, leaves[:1], torch.stack((g, 2 * g)), is_grads_batched=True)
    assert rel(gb[1], 2 * exact[0]) <= 1.1 * rel(got[1][0], exact[0])
    e, dw = OB.qk_norm_rope_attention_backward(g[:0], qkv[:0], w0, w1, cos, sin, 1e-6)
    assert e.shape == (0, N, 3, H, 64) and dw.abs().max().item() == 0.0


# RMS-size of one rounding of a result, relative to it: half the unit roundoff
UNIT = {torch.float32: 2.0**-25, torch.bfloat16: 2.0**-9, torch.float16: 2.0**-12}


def check_grads(names, ours, eager, exact, dtype):
    """Each gradient no further from the exact one than eager's (x 1.1) plus one rounding of the result; fp32 sums in
    another order: 1e-6."""
    for name, a, e, x in zip(names, ours, eager, exact):
        assert a.dtype == e.dtype and a.shape == e.shape, name
        bound = 1.1 * rel(e, x) + UNIT[dtype] + (1e-6 if dtype == torch.float32 else 0.0)
        assert rel(a, x) <= bound, f"{name}: {rel(a, x):.2e}, eager {rel(e, x):.2e}"


def grads_of(fn, tensors, outs, dtype=None):
    leaves = [(t.to(dtype) if dtype else t.clone()).detach().requires_grad_() for t in tensors]
    got = fn(*leaves)
    got = got if isinstance(got, tuple) else (got,)
    return torch.autograd.grad(got, leaves, [g.to(o.dtype) for g, o in zip(outs, got)])


def norm_mod_exact(x, w, shift, scale):
    n = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w
    return n * (1 + scale[:, None]) + shift[:, None]


# C: below and past one 256-channel chunk, the 3-chunk form and the widest; N: one token, runs that end inside a block,
# a sample longer than a block's run; B * N large enough for the 16-token runs (1, 8192) and larger (40, 1030); column
# sums of many parts over few columns (1, 8192) and from 12288 columns on (16, 272, 768); one block per CU (8, 520, 1280)
@pytest.mark.parametrize("B,N,C", [(2, 1, 8), (3, 9, 260), (2, 257, 768), (1, 8192, 64), (40, 1030, 128), (2, 33, 1152),
                                   (2, 5, 2048), (16, 272, 768), (8, 520, 1280)])  # fmt: skip
@pytest.mark.parametrize("dtype,wdt", [(torch.float32, torch.float32), (torch.bfloat16, torch.float32), (torch.float16, torch.float16)])
def test_gated_norm_backward(B, N, C, dtype, wdt):
    print(f"case gated norm backward B={B} N={N} C={C} {dtype} {wdt}", flush=True)
    gen = torch.Generator().manual_seed(N + C)
    z, a, m, gd, gy = (torch.randn((B, N, C), generator=gen).to(DEV, dtype) for _ in range(5))
    t6 = (torch.randn((B, 3 * C), generator=gen) * 0.3).to(DEV, dtype)
    gate, shift, scale = t6.chunk(3, -1)  # strided rows, as the model passes them
    w = (torch.randn(C, generator=gen) * 0.1 + 1).to(DEV, wdt)

    def exact(z, a, gate, w, shift, scale):
        d = gate[:, None] * a
        return d, norm_mod_exact(z + d, w, shift, scale)

    tensors, names = (z, a, gate, w, shift, scale), ("z", "a", "gate", "weight", "shift", "scale")
    ours = grads_of(lambda *t: OB.gate_add_norm_modulate(*t, 1e-6), tensors, (gd, gy))
    eager = grads_of(lambda *t: OB.gate_add_norm_modulate_eager(*t, 1e-6), tensors, (gd, gy))
    check_grads(names, ours, eager, grads_of(exact, tensors, (gd, gy), torch.float64), dtype)
    # no gradient of d is a zero gradient of d
    zero = OB.gate_add_norm_modulate_backward(torch.zeros_like(gd), gy, z, a, gate, w, scale, 1e-6)
    for p, q in zip(OB.gate_add_norm_modulate_backward(None, gy, z, a, gate, w, scale, 1e-6), zero):
        assert torch.equal(p, q)

    tensors = (z, w, shift, scale)
    ours = grads_of(lambda *t: ops.norm_modulate(*t, 1e-6)[0], tensors, (gy,))
    eager = grads_of(lambda x, w, sh, sc: OB._rms_norm_eager(x, w, 1e-6) * (1 + sc[:, None]) + sh[:, None], tensors, (gy,))
    check_grads(("x", "weight", "shift", "scale"), ours, eager, grads_of(norm_mod_exact, tensors, (gy,), torch.float64), dtype)

    if C % 8 == 0:
        tensors = (gd, gate, m)
        ours, eager = grads_of(OB.gate_residual, tensors, (gy,)), grads_of(OB.gate_residual_eager, tensors, (gy,))
        check_grads(("d", "gate", "m"), ours, eager, grads_of(OB.gate_residual_eager, tensors, (gy,), torch.float64), dtype)


def test_gate_residual_backward_past_2048_channels():
    print("case gate residual backward C=2056", flush=True)
    gen = torch.Generator().manual_seed(0)
    d, m, g = (torch.randn((2, 3, 2056), generator=gen).to(DEV, torch.bfloat16) for _ in range(3))
    gate = torch.randn((2, 2056), generator=gen).to(DEV, torch.bfloat16)
    ours, eager = grads_of(OB.gate_residual, (d, gate, m), (g,)), grads_of(OB.gate_residual_eager, (d, gate, m), (g,))
    check_grads(("d", "gate", "m"), ours, eager, grads_of(OB.gate_residual_eager, (d, gate, m), (g,), torch.float64), torch.bfloat16)


@pytest.mark.parametrize("rows,F", [(1, 8), (3, 24), (257, 2056)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_swiglu_backward_bits(rows, F, dtype):
    print(f"case swiglu backward rows={rows} F={F} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(F)
    x = (torch.randn((rows, 2 * F), generator=gen) * 3).to(DEV, dtype)
    special = torch.tensor([0.0, -0.0, 88.0, -88.0, 100.0, -100.0, float("inf"), float("nan")], device=DEV, dtype=dtype)
    x[0, :8] = special
    g = torch.randn((rows, F), generator=gen).to(DEV, dtype)
    (ours,), (eager,) = grads_of(OB.swiglu, (x,), (g,)), grads_of(OB.swiglu_eager, (x,), (g,))
    assert torch.equal(ours.isnan(), eager.isnan())
    a, e = ours.nan_to_num().float(), eager.nan_to_num().float()
    if dtype == torch.float16:
        # the kernel rounds the gate's gradient to fp32 and then to fp16; torch's own fp16 kernel may fold its last
        # product and the narrowing into one rounding, so a value next to a tie can differ by one unit: |d| <= 2^-10 |e|
        # (2^-24 below the normal range), in at most 1 of 1000
        assert ((a - e).abs() <= 2.0**-10 * e.abs() + 2.0**-24).all() and (a != e).float().mean().item() <= 1e-3
    else:
        assert torch.equal(a, e)


# vectors: fewer than one block's 32, an odd number, more than the grid takes in one step (B * N * H > 4 CUs x 256)
@pytest.mark.parametrize("B,N,H", [(1, 4, 1), (3, 100, 3), (40, 144, 7)])
@pytest.mark.parametrize("dtype,tdt,wdt", [
    (torch.float32, torch.float32, torch.float32),
    (torch.bfloat16, torch.float32, torch.bfloat16),
    (torch.float16, torch.float16, torch.float32),
])  # fmt: skip
def test_qk_norm_rope_backward(B, N, H, dtype, tdt, wdt):
    print(f"case qk norm rope backward B={B} N={N} H={H} {dtype} {tdt} {wdt}", flush=True)
    gen = torch.Generator().manual_seed(N)
    qkv = (torch.randn((B, N, 3, H, 64), generator=gen) * 2).to(DEV, dtype)
    w0, w1 = ((torch.randn(64, generator=gen) * 0.2 + 1).to(DEV, wdt) for _ in range(2))
    th = torch.rand((N, 64), generator=gen) * 6.2831853
    cos, sin = th.cos().to(DEV, tdt), th.sin().to(DEV, tdt)
    gq, gk = (torch.randn((B, N, H, 64), generator=gen).to(DEV, dtype) for _ in range(2))
    c, s = cos.to(dtype).double(), sin.to(dtype).double()

    def exact(x, a, b):
        return qk_exact(x[:, :, 0], a, c, s), qk_exact(x[:, :, 1], b, c, s)

    tensors = (qkv, w0, w1)
    ours = grads_of(lambda *t: OB.qk_norm_rope(*t, cos, sin, 1e-6), tensors, (gq, gk))
    eager = grads_of(lambda *t: OB.qk_norm_rope_eager(*t, cos, sin, 1e-6), tensors, (gq, gk))
    check_grads(("qkv", "q weight", "k weight"), ours, eager, grads_of(exact, tensors, (gq, gk), torch.float64), dtype)
    assert ours[0][:, :, 2].abs().max().item() == 0.0


# ends of the 256 x 128 tile and of the 32-row stage, one stage, an odd number of stages, parts that end inside a stage;
# one tile per CU, parts long enough for two blocks per CU (16417 rows in 9 parts), more tiles than fit at once (561)
@pytest.mark.parametrize("rows,N,K", [
    (1, 8, 8), (33, 264, 136), (96, 256, 128), (1000, 48, 768), (4097, 520, 392), (600, 4096, 2048),
    (16384 + 33, 2304, 768), (300, 8200, 2056),
])  # fmt: skip
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear_weight_grad(rows, N, K, dtype):
    print(f"case linear weight grad rows={rows} N={N} K={K} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(rows + N)
    g, x = torch.randn((rows, N), generator=gen).to(DEV, dtype), torch.randn((rows, K), generator=gen).to(DEV, dtype)
    gw, gb = OB.linear_weight_grad(g, x, True)
    for got, ref, name in ((gw, g.double().t() @ x.double(), "weight"), (gb, g.double().sum(0), "bias")):
        # one rounding of an fp32 sum, u = 2^-8 (bf16: 8 significant bits) or 2^-11 (fp16: 11):
        # |d| <= u |ref| + 2^-20 sum |terms| (fp32 sums of up to `rows` terms in any order)
        u = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
        terms = g.double().abs().t() @ x.double().abs() if name == "weight" else g.double().abs().sum(0)
        tiny = 2.0**-25 if dtype == torch.float16 else 0.0  # half of fp16's smallest step
        assert ((got.double() - ref).abs() <= u * ref.abs() * (1 + 2.0**-10) + 2.0**-20 * terms + tiny).all(), name
    none = OB.linear_weight_grad(g, x, False)
    assert torch.equal(none[0], gw) and none[1].numel() == 0


def test_linear_layer_routes():
    """The layer's training route against torch's linear: values, gradients under autocast and in 16 bits, without a
    bias, a frozen weight, a graph of the backward, a batch of gradients; and the calls that stay torch's own."""
    print("case linear layer routes", flush=True)
    lin, ref = M.CastLinear(64, 136).to(DEV), torch.nn.Linear(64, 136).to(DEV)
    ref.load_state_dict(lin.state_dict())
    x = torch.randn((4, 200, 64), generator=torch.Generator().manual_seed(0)).to(DEV)
    g = torch.randn((4, 200, 136), generator=torch.Generator().manual_seed(1)).to(DEV)

    def grads(layer, x, g, amp):
        xl = x.clone().requires_grad_()
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
            y = layer(xl)
        return [y, *torch.autograd.grad(y, [xl, *[p for p in layer.parameters() if p.requires_grad]], g.to(y.dtype))]

    def same(a, b):
        for p, q in zip(a, b, strict=True):
            assert p.dtype == q.dtype and p.shape == q.shape and rel(p, q) <= 4e-3

    assert OB.linear(x.bfloat16(), lin.weight.bfloat16(), None) is not None
    same(grads(lin, x, g, True), grads(ref, x, g, True))  # fp32 weights under autocast
    same(grads(lin.bfloat16(), x.bfloat16(), g, False), grads(ref.bfloat16(), x.bfloat16(), g, False))
    xl = x.bfloat16().requires_grad_()
    y = lin(xl)
    (a,) = torch.autograd.grad(y, lin.weight, torch.stack((g, 2 * g)).bfloat16(), is_grads_batched=True, retain_graph=True)
    assert rel(a[1], 2 * a[0]) <= 4e-3
    second = []
    for layer in (lin, ref):  # a graph of the backward
        y = layer(xl)
        (gw,) = torch.autograd.grad(y, layer.weight, g.bfloat16(), create_graph=True)
        second.append(torch.autograd.grad(gw.float().square().sum(), xl)[0])
    assert rel(*second) <= 1e-2
    amp = M.CastLinear(64, 136).to(DEV)
    with torch.autocast("cuda", dtype=torch.bfloat16):  # a parameter is converted once in an autocast region
        nodes = [amp(x).grad_fn for _ in range(2)]
    assert [f for f, _ in nodes[0].next_functions[1:]] == [f for f, _ in nodes[1].next_functions[1:]]
    lin.weight.requires_grad_(False)
    assert OB.linear(xl, lin.weight, lin.bias) is None and lin(xl).requires_grad
    lin.weight.requires_grad_(True)
    wide = torch.zeros((4096, 2048), device=DEV, dtype=torch.bfloat16, requires_grad=True)  # 256 tiles, and 240
    rows = torch.zeros((512, 2048), device=DEV, dtype=torch.bfloat16)
    assert OB.linear(rows, wide, None) is None and OB.linear(rows, wide[:3840], None) is not None
    w = lin.weight.detach()
    assert OB.linear(xl[:1, :100], lin.weight, None) is None and OB.linear(x, lin.weight, None) is None
    out = torch.func.grad(lambda t: torch.nn.functional.linear(t, w).float().sum())(x.bfloat16())
    assert rel(torch.func.grad(lambda t: lin(t).float().sum())(x.bfloat16()), out) <= 1e-6
    with torch.no_grad():
        assert OB.linear(xl, lin.weight, None) is None


class SeenLinear(torch.nn.Parameter):
    """A parameter that notes the calls of torch's linear that it takes part in."""

    seen = 0

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.seen += func is torch.nn.functional.linear
        with torch._C.DisableTorchFunctionSubclass():
            return func(*args, **(kwargs or {}))


class Seen(torch.overrides.TorchFunctionMode):
    seen = 0

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.seen += func is torch.nn.functional.linear
        return func(*args, **(kwargs or {}))


def test_linear_layer_is_torchs_own_to_subclasses_and_modes():
    """What takes torch's linear apart sees it: a parameter subclass, a torch function mode, a flop counter (three
    products of 2 M N K), the TorchScript tracer.  A default device is no such mode."""
    print("case linear layer: subclasses and modes", flush=True)
    lin, x = M.CastLinear(64, 128).to(DEV).bfloat16(), torch.ones((600, 64), device=DEV, dtype=torch.bfloat16)
    x.requires_grad_()
    with FlopCounterMode(display=False) as flops:
        lin(x).sum().backward()
    assert flops.get_total_flops() == 3 * 2 * 600 * 64 * 128
    with Seen() as mode:
        lin(x)
    assert mode.seen == 1
    with torch.device(DEV):
        assert OB.linear(x, lin.weight, lin.bias) is not None
    assert "aten::linear" in str(torch.jit.trace(lin, x).graph)
    lin._parameters["weight"] = torch.Tensor._make_subclass(SeenLinear, lin.weight.detach(), True)
    lin(x)
    assert SeenLinear.seen == 1
