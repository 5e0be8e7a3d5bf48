"""Fused elementwise ops of the LTHC transformer branch (gfx950 HIP kernels).

The reference evaluates these chains as eager PyTorch ops; they have no
``jit_thc`` counterpart there.  Each op here is one HIP pass with the eager
sequence's roundings (fp32 arithmetic, every eager op's result rounded to the
activation dtype), registered as a ``jit_thc`` custom op:

* ``jit_thc::qk_norm_rope``: ``rope(q_norm(q))`` and ``rope(k_norm(k))`` of
  ``WorkspaceAttention.forward`` (local_thc.py:246-249; RMSNorm
  jit_shared_adaln.py:26-30; VisionRotaryEmbeddingFast jit_shared_adaln.py:57-59),
  taking the qkv projection [B, N, 3, H, 64] and returning q and k as
  [B, N, H, 64] (the memory layout of the eager result);
* ``jit_thc::qk_norm_rope_attention``: the same q and k followed by
  ``F.scaled_dot_product_attention`` (local_thc.py:246-251), one matrix-core
  pass from the qkv projection to the attention output [B, N, H, 64];
* ``jit_thc::swiglu``: ``F.silu(x1) * x2`` of ``SwiGLUFFN.forward``
  (local_thc.py:267-269) for the w12 projection [..., 2F];
* ``jit_thc::gate_add_norm_modulate``: ``dz_attn = gate_msa * attn``,
  ``z_tmp = z + dz_attn`` and ``modulate(norm2(z_tmp), ...)`` of
  ``WorkspaceSharedAdaLNBranch.forward`` (local_thc.py:319-322);
* ``jit_thc::gate_residual``: its ``dz_attn + gate_mlp * mlp`` (:322-323);
* ``jit_thc::block_tail`` (inference): that gate_residual, the lazy
  recurrence step ``Z_{l+1} = Z_l + gamma_l * dZ_l`` (local_thc.py:1325-1328)
  and the next block's first pre-norm (:315-317) in one pass, each value
  that of the three separate ops.

Every op but block_tail (inference only) has a backward kernel of its own,
``jit_thc::<op>_backward``, one HIP pass that recomputes what it needs from the
op's inputs and gives the gradients of the eager sequence.  For batched
gradients (is_grads_batched, vmap) torch runs that pass once per sample.  A
traced backward (torch.compile) differentiates the eager sequence in place of
those kernels (gate_residual's apart, which rounds nothing in between): the
compiled graph keeps the chain's intermediates in fp32.
"""

from __future__ import annotations

import torch
import torch.nn.functional as F
from torch import Tensor
from torch.utils._device import DeviceContext

from . import _abi
from .ops import _fake, _refuse

QK_HEAD_DIM = 64


# ---------------------------------------------------------------------------
# eager restatements: what each kernel's values and gradients are compared with
# ---------------------------------------------------------------------------
def _rms_norm_eager(x: Tensor, weight: Tensor, eps: float) -> Tensor:
    xf = x.float()
    return (xf * torch.rsqrt(xf.pow(2).mean(dim=-1, keepdim=True) + eps) * weight).to(x.dtype)


def _rope_eager(x: Tensor, cos: Tensor, sin: Tensor) -> Tensor:
    pairs = x.unflatten(-1, (-1, 2))
    rot = torch.stack((-pairs[..., 1], pairs[..., 0]), dim=-1).flatten(-2)
    return x * cos.to(x.dtype) + rot * sin.to(x.dtype)


def qk_norm_rope_eager(qkv: Tensor, q_weight: Tensor, k_weight: Tensor, cos: Tensor, sin: Tensor, eps: float):
    """The eager sequence on qkv [B, N, 3, H, D]: (q, k) as [B, N, H, D] (cos / sin [N, D] broadcast over heads)."""
    c, s = cos[:, None, :], sin[:, None, :]
    q = _rope_eager(_rms_norm_eager(qkv[:, :, 0], q_weight, eps), c, s)
    k = _rope_eager(_rms_norm_eager(qkv[:, :, 1], k_weight, eps), c, s)
    return q, k


def swiglu_eager(x: Tensor) -> Tensor:
    a, v = x.chunk(2, dim=-1)
    return F.silu(a) * v


# ---------------------------------------------------------------------------
# traced backwards: the eager sequence, differentiated
# ---------------------------------------------------------------------------
def _backward_replay(name: str, eager, leaves: int) -> None:
    """Define jit_thc::<name>_backward_replay(grads, saved, eps) -> the gradients of the first `leaves` of eager's
    arguments (saved; eps).  Composite: the native nodes call it where a backward is traced (csrc/torch_ops.cpp)."""

    def replay(grads: list[Tensor], saved: list[Tensor], eps: float) -> list[Tensor]:
        with torch.enable_grad():
            args = [t.detach().requires_grad_(i < leaves) for i, t in enumerate(saved)]
            outs = eager(args, eps)
            return list(torch.autograd.grad(outs, args[:leaves], grads))

    op = f"jit_thc::{name}_backward_replay"
    torch.library.define(op, "(Tensor[] grads, Tensor[] saved, float eps) -> Tensor[]")
    torch.library.impl(op, "CompositeImplicitAutograd")(replay)


# ---------------------------------------------------------------------------
# jit_thc::qk_norm_rope
# ---------------------------------------------------------------------------
@torch.library.custom_op("jit_thc::qk_norm_rope", mutates_args=())
def qk_norm_rope(qkv: Tensor, q_weight: Tensor, k_weight: Tensor, cos: Tensor, sin: Tensor, eps: float) -> tuple[Tensor, Tensor]:
    """(rope(RMSNorm_q(q)), rope(RMSNorm_k(k))) as [B, N, H, 64] in qkv's dtype, one pass over q and k."""
    _refuse(qkv)


@_fake(qk_norm_rope)
def _(qkv, q_weight, k_weight, cos, sin, eps):
    b, n, _, h, d = qkv.shape
    return qkv.new_empty((b, n, h, d)), qkv.new_empty((b, n, h, d))


@torch.library.custom_op("jit_thc::qk_norm_rope_backward", mutates_args=())
def qk_norm_rope_backward(
    grad_q: Tensor, grad_k: Tensor, qkv: Tensor, q_weight: Tensor, k_weight: Tensor, cos: Tensor, sin: Tensor, eps: float
) -> tuple[Tensor, Tensor]:
    """(gradient of qkv in qkv's dtype, zero for v, and the fp32 [2, 64] gradients of the q and k norm weights) of
    qk_norm_rope, with eager autograd's roundings, one pass."""
    _refuse(qkv)


@_fake(qk_norm_rope_backward)
def _(grad_q, grad_k, qkv, q_weight, k_weight, cos, sin, eps):
    return qkv.new_empty(qkv.shape), qkv.new_empty((2, QK_HEAD_DIM), dtype=torch.float32)


_backward_replay("qk_norm_rope", lambda a, eps: list(qk_norm_rope_eager(*a, eps)), 3)


# ---------------------------------------------------------------------------
# jit_thc::qk_norm_rope_attention
# ---------------------------------------------------------------------------
ATTN_MAX_TOKENS = 256


def attention_supported(qkv: Tensor) -> bool:
    """Whether jit_thc::qk_norm_rope_attention takes qkv [B, N, 3, H, 64]: 16-bit, N a multiple of 64 up to 256."""
    n = qkv.shape[1]
    return (
        qkv.is_cuda
        and qkv.dtype in (torch.bfloat16, torch.float16)
        and qkv.dim() == 5
        and qkv.shape[4] == QK_HEAD_DIM
        and n % 64 == 0
        and 0 < n <= ATTN_MAX_TOKENS
    )


def qk_norm_rope_attention_eager(qkv: Tensor, q_weight: Tensor, k_weight: Tensor, cos: Tensor, sin: Tensor, eps: float):
    """q/k norm + RoPE, then F.scaled_dot_product_attention (default scale, no mask): o as [B, N, H, D]."""
    q, k = qk_norm_rope_eager(qkv, q_weight, k_weight, cos, sin, eps)
    v = qkv[:, :, 2]
    # [B, H, N, D] operands made contiguous (no transposed views in the batched products)
    q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, v))
    o = F.scaled_dot_product_attention(q, k, v)
    return o.transpose(1, 2)


@torch.library.custom_op("jit_thc::qk_norm_rope_attention", mutates_args=())
def qk_norm_rope_attention(qkv: Tensor, q_weight: Tensor, k_weight: Tensor, cos: Tensor, sin: Tensor, eps: float) -> Tensor:
    """softmax(q_n k_n^T / sqrt(64)) v for q_n, k_n = qk_norm_rope(...): o as [B, N, H, 64] in qkv's dtype (bf16 or
    fp16, N a multiple of 64 up to 256), one pass over qkv on the matrix cores."""
    _refuse(qkv)


@_fake(qk_norm_rope_attention)
def _(qkv, q_weight, k_weight, cos, sin, eps):
    b, n, _, h, d = qkv.shape
    return qkv.new_empty((b, n, h, d))


@torch.library.custom_op("jit_thc::qk_norm_rope_attention_backward", mutates_args=())
def qk_norm_rope_attention_backward(
    grad: Tensor, qkv: Tensor, q_weight: Tensor, k_weight: Tensor, cos: Tensor, sin: Tensor, eps: float
) -> tuple[Tensor, Tensor]:
    """(gradient of qkv in qkv's dtype, fp32 [2, 64] gradients of the q and k norm weights) of
    qk_norm_rope_attention for the output gradient `grad` [B, N, H, 64], one matrix-core pass over qkv and grad."""
    _refuse(qkv)


@_fake(qk_norm_rope_attention_backward)
def _(grad, qkv, q_weight, k_weight, cos, sin, eps):
    return qkv.new_empty(qkv.shape), qkv.new_empty((2, QK_HEAD_DIM), dtype=torch.float32)


def _attention_fp32_recompute(qkv: Tensor, q_weight: Tensor, k_weight: Tensor, cos: Tensor, sin: Tensor, eps: float):
    """qk_norm_rope_attention_eager's function with the attention itself in fp32 matrix products and softmax
    (softmax(q k^T / sqrt(64)) v, rounded once to qkv's dtype).  Plain products, not the SDPA kernels: the ROCm
    flash-attention backward returns gradient strides its meta function does not predict, which compiled graphs
    assert on."""
    q, k = qk_norm_rope_eager(qkv, q_weight, k_weight, cos, sin, eps)
    v = qkv[:, :, 2]
    q, k, v = (t.transpose(1, 2).float().contiguous() for t in (q, k, v))
    kt = k.transpose(-1, -2).contiguous()
    p = torch.softmax(torch.matmul(q, kt) * (QK_HEAD_DIM**-0.5), dim=-1)
    return torch.matmul(p, v).to(qkv.dtype).transpose(1, 2)


_backward_replay("qk_norm_rope_attention", lambda a, eps: [_attention_fp32_recompute(*a, eps)], 3)


# ---------------------------------------------------------------------------
# jit_thc::swiglu
# ---------------------------------------------------------------------------
@torch.library.custom_op("jit_thc::swiglu", mutates_args=())
def swiglu(x: Tensor) -> Tensor:
    """silu(x[..., :F]) * x[..., F:] in x's dtype for x [..., 2F], F % 8 == 0."""
    _refuse(x)


@_fake(swiglu)
def _(x):
    return x.new_empty((*x.shape[:-1], x.shape[-1] // 2))


@torch.library.custom_op("jit_thc::swiglu_backward", mutates_args=())
def swiglu_backward(grad: Tensor, x: Tensor) -> Tensor:
    """Gradient of swiglu for x [..., 2F] and the output gradient [..., F], with eager autograd's roundings."""
    _refuse(x)


@_fake(swiglu_backward)
def _(grad, x):
    return x.new_empty(x.shape)


_backward_replay("swiglu", lambda a, eps: [swiglu_eager(*a)], 1)


# ---------------------------------------------------------------------------
# gated residuals of the branch: jit_thc::gate_add_norm_modulate, jit_thc::gate_residual
# (WorkspaceSharedAdaLNBranch.forward, local_thc.py:319-323)
# ---------------------------------------------------------------------------
def gate_add_norm_modulate_eager(z: Tensor, a: Tensor, gate: Tensor, weight: Tensor, shift: Tensor, scale: Tensor, eps: float):
    """(d, y): d = gate * a, y = modulate(RMSNorm(z + d), shift, scale), as the eager branch evaluates them."""
    d = gate.unsqueeze(1) * a
    n = _rms_norm_eager(z + d, weight, eps)
    return d, n * (1 + scale.unsqueeze(1)) + shift.unsqueeze(1)


def gate_residual_eager(d: Tensor, gate: Tensor, m: Tensor) -> Tensor:
    return d + gate.unsqueeze(1) * m


@torch.library.custom_op("jit_thc::gate_add_norm_modulate", mutates_args=())
def gate_add_norm_modulate(
    z: Tensor, a: Tensor, gate: Tensor, weight: Tensor, shift: Tensor, scale: Tensor, eps: float
) -> tuple[Tensor, Tensor]:
    """(gate * a, modulate(RMSNorm(z + gate * a), shift, scale)) in z's dtype, one pass; z, a [B,N,C], the rest [B,C]
    (weight [C])."""
    _refuse(z)


@_fake(gate_add_norm_modulate)
def _(z, a, gate, weight, shift, scale, eps):
    return torch.empty_like(z), torch.empty_like(z)


def _grad_dtype(weight: Tensor) -> torch.dtype:
    """The dtype the kernels write a norm weight's gradient in: the weight's own where it is one of theirs."""
    return weight.dtype if weight.dtype in _abi.DTYPE_CODE else torch.float32


@torch.library.custom_op("jit_thc::gate_add_norm_modulate_backward", mutates_args=())
def gate_add_norm_modulate_backward(
    grad_d: Tensor | None, grad_y: Tensor, z: Tensor, a: Tensor, gate: Tensor, weight: Tensor, scale: Tensor, eps: float
) -> tuple[Tensor, Tensor, Tensor, Tensor, Tensor, Tensor]:
    """Gradients of gate_add_norm_modulate's (z, a, gate, weight, shift, scale) for those of d (None: zero) and y, one
    pass over z, a and the gradients; the weight's in its own dtype, the others in z's."""
    _refuse(z)


@_fake(gate_add_norm_modulate_backward)
def _(grad_d, grad_y, z, a, gate, weight, scale, eps):
    b, _, c = z.shape
    row = lambda: z.new_empty((b, c))  # noqa: E731
    return z.new_empty(z.shape), z.new_empty(z.shape), row(), z.new_empty((c,), dtype=_grad_dtype(weight)), row(), row()


_backward_replay("gate_add_norm_modulate", lambda a, eps: list(gate_add_norm_modulate_eager(*a, eps)), 6)


@torch.library.custom_op("jit_thc::gate_residual", mutates_args=())
def gate_residual(d: Tensor, gate: Tensor, m: Tensor) -> Tensor:
    """d + gate * m in d's dtype for d, m [B,N,C] and a per-sample gate [B,C] (C % 8 == 0)."""
    _refuse(d)


@_fake(gate_residual)
def _(d, gate, m):
    return torch.empty_like(d)


@torch.library.custom_op("jit_thc::gate_residual_backward", mutates_args=())
def gate_residual_backward(grad: Tensor, gate: Tensor, m: Tensor) -> tuple[Tensor, Tensor]:
    """(gradient of gate [B,C], gradient of m [B,N,C]) of gate_residual in grad's dtype, one pass over grad and m."""
    _refuse(grad)


@_fake(gate_residual_backward)
def _(grad, gate, m):
    return grad.new_empty(gate.shape), m.new_empty(m.shape)


# ---------------------------------------------------------------------------
# linear layers in training: weight and bias gradients in one pass over the rows
# ---------------------------------------------------------------------------
# From here the kernel is as fast as torch's product and column sum, or faster, on every layer shape of the models (N x K,
# bf16, us of the kernel / torch's).  512 rows: 4096 x 768 28.5 / 27.1 (the one shape behind, with 768 rows too: 29.1 /
# 27.7), 2304 x 768 21.9 / 28.4, 768 x 2048 20.5 / 26.8, 768 x 768 16.5 / 26.6, 6144 x 1152 30.9 / 34.0, 192 x 192
# 13.2 / 37.2, 128 x 48 12.2 / 18.8.  1024 rows: 30.2 / 31.0, 26.4 / 28.4, 25.2 / 27.0, 19.7 / 26.7.  256 rows: 21.9 /
# 25.0, 18.2 / 23.8, 16.9 / 23.8, 14.9 / 23.7, so the line could lie lower.
LINEAR_MIN_ROWS = 512
# From one 256 x 128 tile of the weight per CU on, torch's tiles are the better ones (rounds of whole tiles; us of the
# kernel / torch's at 512, 4096 and 16384 rows).  216 tiles, 6144 x 1152: 30.9 / 34.0, 82.6 / 93.4, 261 / 289; 256, 4096 x
# 2048: 29.8 / 28.6, 85.0 / 87.4, 272 / 285; 344, 2048 x 5456: 39.2 / 40.2, 133 / 115, 460 / 363; 384, 6144 x 2048: 40.9 /
# 33.1, 135 / 113, 469 / 383; 512, 4096 x 4096: 46.7 / 35.9, 154 / 136, 537 / 482.
LINEAR_MAX_TILES = 256


@torch.library.custom_op("jit_thc::linear_weight_grad", mutates_args=())
def linear_weight_grad(grad: Tensor, x: Tensor, need_bias: bool) -> tuple[Tensor, Tensor]:
    """(grad^T x [N, K], column sums of grad [N] or an empty tensor) for grad [..., N] and x [..., K], bf16 or fp16, N
    and K multiples of 8: fp32 sums in a fixed order, rounded once."""
    _refuse(grad)


@_fake(linear_weight_grad)
def _(grad, x, need_bias):
    n = grad.shape[-1]
    return grad.new_empty((n, x.shape[-1])), grad.new_empty((n if need_bias else 0,))


def linear(x: Tensor, weight: Tensor, bias: Tensor | None) -> Tensor | None:
    """F.linear(x, weight, bias) with the weight and bias gradients of a training step from linear_weight_grad, or None
    where that does not apply and the caller calls F.linear: no gradient of the weight, not 16-bit products (autocast's,
    or the operands' own), few rows, a wide weight, or tracing, functorch and forward-mode transforms, tensor subclasses and torch
    function and dispatch modes (a flop counter, for one), which know torch's linear."""
    if torch.compiler.is_compiling() or torch.jit.is_tracing() or not (
        torch.is_grad_enabled()
        and weight.requires_grad
        and type(x) is Tensor
        and type(weight) in (Tensor, torch.nn.Parameter)
        and type(bias) in (Tensor, torch.nn.Parameter, type(None))
        and x.is_cuda
        and x.dim() >= 2
        and x.is_floating_point()
        and x.numel() >= LINEAR_MIN_ROWS * x.shape[-1] > 0
        and x.shape[-1] % 8 == 0
        and weight.shape[0] % 8 == 0
        and x.shape[-1] == weight.shape[1]
        and -(-weight.shape[0] // 256) * -(-weight.shape[1] // 128) < LINEAR_MAX_TILES
        and torch._C._functorch.peek_interpreter_stack() is None
        and torch.autograd.forward_ad._current_level < 0
        and torch._C._len_torch_dispatch_stack() == 0
        and all(type(m) is DeviceContext for m in map(torch._C._get_function_stack_at, range(torch._C._len_torch_function_stack())))
    ):
        return None
    dt = x.dtype
    operands = (x, weight) if bias is None else (x, weight, bias)
    if torch.is_autocast_enabled("cuda"):
        dt = torch.get_autocast_dtype("cuda")
        if any(t.dtype not in _abi.DTYPE_CODE for t in operands):
            return None
    elif any(t.dtype != dt for t in operands):
        return None
    if dt not in (torch.bfloat16, torch.float16) or weight.device != x.device:
        return None
    return torch.ops.jit_thc.linear(x, weight, bias)


# ---------------------------------------------------------------------------
# block tail (inference): gate_residual + recurrence step + the next block's first pre-norm
# ---------------------------------------------------------------------------
@torch.library.custom_op("jit_thc::block_tail", mutates_args=())
def block_tail(
    z: Tensor, a: Tensor, gate: Tensor, m: Tensor, gamma: Tensor, weight: Tensor, shift: Tensor, scale: Tensor,
    eps: float,
) -> tuple[Tensor, Tensor, Tensor]:
    """(dz, z_next, y) = (a + gate * m, z + gamma * dz, modulate(RMSNorm(z_next), shift, scale)) in z's dtype, one
    pass: gate_residual, lazy_workspace_update and the next block's norm_modulate with the same values.  z, a, m
    [B,N,C]; gate, shift, scale [B,C]; gamma and weight [C].  Forward only (inference)."""
    _refuse(z)


@_fake(block_tail)
def _(z, a, gate, m, gamma, weight, shift, scale, eps):
    return torch.empty_like(z), torch.empty_like(z), torch.empty_like(z)
