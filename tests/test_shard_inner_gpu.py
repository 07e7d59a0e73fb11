"""The data gradient of a depth shard's convolution is computed for the shard's own planes only (the slab's faces are zeros the
module put there): one and several samples, one and two input tensors, and a halo wider than the padded problem's gradient
takes, which is cut out of the slab's gradient."""

import pytest
import torch

from scaffold_amd.modules import FastConv3d

pytestmark = pytest.mark.gpu
CL = torch.channels_last_3d


@pytest.mark.parametrize("batch,channels,padding,spatial", [
    (1, 32, 1, (5, 9, 33)),     # ring kernel, cut tiles
    (1, 64, 2, (4, 8, 17)),     # the widest halo the padded problem takes; brick kernel
    (1, 64, 3, (4, 8, 17)),     # wider: the slab's gradient, cut
    (2, 64, 1, (2, 16, 16)),    # a batch: a shard's planes of several samples; small volumes
    (1, 48, 1, (3, 5, 6)),      # direct kernels
])
def test_shard_gradients_against_float64(batch, channels, padding, spatial):
    g = torch.Generator(device="cuda").manual_seed(3)
    conv = FastConv3d(channels, channels, 3, padding=(padding, 1, 1), bias=False, device="cuda", dtype=torch.bfloat16)
    conv.shard_halo = True
    x = torch.randn((batch, channels, *spatial), generator=g, device="cuda").bfloat16().contiguous(memory_format=CL).requires_grad_()
    y = conv(x)
    gy = torch.randn(y.shape, generator=g, device="cuda").bfloat16()
    y.backward(gy)
    xd, wd = x.detach().cpu().double().requires_grad_(), conv.weight.detach().cpu().double().requires_grad_()
    yd = torch.nn.functional.conv3d(xd, wd, padding=(padding, 1, 1))
    yd.backward(gy.cpu().double())
    assert x.grad.shape == x.shape and x.grad.is_contiguous(memory_format=CL)
    for got, want in ((y, yd), (x.grad, xd.grad), (conv.weight.grad, wd.grad)):
        # one rounding to bf16 (half of 2^-7 relative at most, 1.7e-3 in the mean) of a 32-bit sum
        assert torch.linalg.vector_norm(got.detach().cpu().double() - want.detach()) <= 4e-3 * torch.linalg.vector_norm(want.detach())


@pytest.mark.parametrize("spatial", [(4, 16, 16), (3, 8, 40)])
def test_pair_in_slabs_gets_the_padded_forms_gradients(spatial):
    g = torch.Generator(device="cuda").manual_seed(4)
    conv = FastConv3d(128, 64, 3, padding=1, bias=False, device="cuda", dtype=torch.bfloat16)
    parts, slabs = [], []
    for _ in range(2):
        slab = torch.zeros((1, 64, spatial[0] + 2, *spatial[1:]), device="cuda", dtype=torch.bfloat16).contiguous(memory_format=CL)
        slab[:, :, 1:-1] = torch.randn((1, 64, *spatial), generator=g, device="cuda")
        part = slab[:, :, 1:-1].detach().requires_grad_()
        part._sfh_slab = (slab, 1)
        parts.append(part)
        slabs.append(slab)
    grads = []
    for shard in (False, True):
        conv.shard_halo = shard
        assert conv.takes_pair(*parts)
        y = conv(*parts)
        gy = torch.ones_like(y) / 8 + torch.arange(64, device="cuda", dtype=torch.bfloat16).view(1, 64, 1, 1, 1) / 16
        grads.append(torch.autograd.grad(y, (*parts, conv.weight), gy))
    for a, b in zip(*grads):
        assert torch.equal(a, b)
