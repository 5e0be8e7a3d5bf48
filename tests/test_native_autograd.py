"""The native autograd nodes (csrc/torch_ops.cpp) on CPU tensors: plain-torch kernels stand in for the HIP ones while a
test runs, so that what autograd sees of the nodes can be checked without a GPU."""

from __future__ import annotations

import math

import pytest
import torch

from flowmatching_lthc_amd import ops


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


def recur_backward(g, dz, gamma, add=None):
    return gamma * g + (0 if add is None else add), (g * dz).sum((0, 1))


KERNELS = {
    "local_write_traceable": read,
    "local_read_traceable": write,
    "local_read_add_traceable": lambda z, w, x: x + write(z, w),
    "local_weight_grad_traceable": lambda high, low: (cells(high) * low[:, :, None]).sum((0, 1)).t().contiguous(),
    "lazy_workspace_update": lambda z, dz, gamma: z + gamma * dz,
    "lazy_workspace_update_backward": recur_backward,
    "lazy_workspace_update_backward_sum": lambda g, b, dz, gamma, add=None: (g + b, *recur_backward(g + b, dz, gamma, add)),
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
