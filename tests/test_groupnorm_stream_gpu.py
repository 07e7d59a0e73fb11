"""GroupNorm on tensors past the size from which the operands are read past the caches (128 MiB), at sizes just above that line whose
last workgroups are cut, and the launch that finishes its sums at channel counts off its blocks of 16."""

import pytest
import torch

import scaffold_amd as sa

pytestmark = pytest.mark.gpu
CL = torch.channels_last_3d


@pytest.mark.parametrize("n,c,groups,spatial,dtype", [
    (1, 32, 8, (129, 128, 127), torch.bfloat16),  # 134.2 MB
    (2, 64, 8, (65, 128, 65), torch.float16),     # two samples, cut passes
    (1, 32, 8, (65, 129, 127), torch.float32),    # 136.3 MB
    (2, 24, 3, (9, 30, 31), torch.bfloat16),      # six columns of sums: the finishing launch whatever the size, 24 channels
    (1, 40, 5, (40, 64, 64), torch.float16),
])
def test_against_float64(n, c, groups, spatial, dtype):
    g = torch.Generator(device="cuda").manual_seed(11)
    x = (torch.randn((n, c, *spatial), generator=g, device="cuda") * 3 + 0.5).to(dtype).contiguous(memory_format=CL).requires_grad_()
    gy = torch.randn((n, c, *spatial), generator=g, device="cuda").to(dtype).contiguous(memory_format=CL)
    norm = sa.FastGroupNorm(groups, c, activation="relu", device="cuda")
    with torch.no_grad():
        norm.weight.add_(0.1 * torch.randn(c, generator=g, device="cuda"))
        norm.bias.add_(0.1 * torch.randn(c, generator=g, device="cuda"))
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=dtype is not torch.float32):
        y = norm(x)
    got = (y.detach(), *torch.autograd.grad(y, (x, norm.weight, norm.bias), gy))
    xd, w, b = (t.detach().double().requires_grad_() for t in (x, norm.weight, norm.bias))
    yd = torch.relu(torch.nn.functional.group_norm(xd, groups, w, b, norm.eps))
    want = (yd.detach(), *torch.autograd.grad(yd, (xd, w, b), gy.double()))
    # results: one rounding (2^-9, 2^-12 or 2^-24 relative at most; an element at the ReLU's edge may flip, which 2^-9 covers in fp32
    # too); parameter gradients: fp32 sums of up to two million terms of either sign in trees, a few hundred ulps of their 2-norm at most
    one = {torch.bfloat16: 2 ** -9, torch.float16: 2 ** -12, torch.float32: 1e-5}[dtype]
    for have, ref, tol in zip(got, want, (one, 2 * one, 1e-4, 1e-4)):
        assert torch.linalg.vector_norm(have.double() - ref) <= tol * torch.linalg.vector_norm(ref)


def test_parameter_gradients_of_many_workgroups_meet_in_trees():
    """1024 workgroups of 16 passes of 85 voxels (24 channels) leave a sum each: the first 2^24, the others 1.  fp32 loses up to half an ulp of
    2^24, which is 1, wherever something is added to that first sum: 1024 / 256 - 1 times in its thread, 6 in the wavefront's
    tree, 2 among four wavefronts.  Added one after the other, 1024 / 64 of them in a thread, they would lose 15 there alone."""
    splits, rows, c = 1024, 16 * 85, 24
    x = torch.randn((1, c, splits, 34, 40), device="cuda").to(torch.bfloat16).contiguous(memory_format=CL)
    gy = torch.zeros((1, splits * rows, c), dtype=torch.bfloat16, device="cuda")
    gy[:, ::rows] = 1
    gy[:, 0] = 2.0 ** 24
    gy = gy.view(1, splits, 34, 40, c).permute(0, 4, 1, 2, 3)
    norm = sa.FastGroupNorm(3, c, device="cuda")
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = norm(x.requires_grad_())
    (got,) = torch.autograd.grad(y, norm.bias, gy)
    assert got.dtype is torch.float32 and (got.double() - (2 ** 24 + splits - 1)).abs().max() <= 3 + 6 + 2


@pytest.mark.parametrize("c,groups,spatial", [
    (96, 3, (1024, 16, 21)),  # 1024 sums of 32 channels to a group: a thread's sums are carried over two rounds
    (96, 3, (16, 21, 29)),    # 29 of them, fewer than a round
    (24, 3, (60, 34, 40)),    # 60 of 8 channels
])
def test_group_sums_carried_between_quarters(c, groups, spatial):
    """The group coefficients of a gradient that has a mean and follows x: without a part of them dx is off by a part of itself."""
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((1, c, *spatial), generator=g, device="cuda").to(torch.bfloat16).contiguous(memory_format=CL).requires_grad_()
    gy = (torch.randn((1, c, *spatial), generator=g, device="cuda") + x.detach() + 1).to(torch.bfloat16).contiguous(memory_format=CL)
    norm = sa.FastGroupNorm(groups, c, device="cuda")
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = norm(x)
    got = torch.autograd.grad(y, (x, norm.weight, norm.bias), gy)
    xd, w, b = (t.detach().double().requires_grad_() for t in (x, norm.weight, norm.bias))
    want = torch.autograd.grad(torch.nn.functional.group_norm(xd, groups, w, b, norm.eps), (xd, w, b), gy.double())
    # dx: one rounding, 2^-9 relative; parameter gradients as above
    for have, ref, tol in zip(got, want, (2 ** -8, 1e-4, 1e-4)):
        assert torch.linalg.vector_norm(have.double() - ref) <= tol * torch.linalg.vector_norm(ref)
