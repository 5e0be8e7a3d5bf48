"""GPU parity of the branch ops' backward kernels (MI355X only): each gradient against autograd of the same function
in float64, no further from it than the eager 16-bit sequence's gradient (x 1.1 for the draw), at the sizes where each
kernel's tiles, lanes and partial rows end."""

from __future__ import annotations

import pytest
import torch

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
