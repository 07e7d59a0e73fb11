"""The head's weight gradient in rounds of 128 voxels: whole rounds only, a cut round alone and behind whole ones, ranges of several
workgroups, every wide width, with and without the bias sums."""

import pytest
import torch

import scaffold_amd as sa

CL = torch.channels_last_3d
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("voxels", [1, 100, 128, 129, 256, 511, 512, 513, 1100, 4096 + 7])
@pytest.mark.parametrize("wide,thin", [(32, 11), (64, 6), (128, 32), (32, 1)])
def test_whole_numbers_are_exact(wide, thin, voxels, dtype):
    g = torch.Generator("cuda").manual_seed(voxels)
    x = torch.randint(-1, 2, (1, wide, voxels, 1, 1), generator=g, device="cuda").to(dtype).contiguous(memory_format=CL)
    gy = torch.randint(-1, 2, (1, thin, voxels, 1, 1), generator=g, device="cuda").to(dtype).contiguous(memory_format=CL)
    want = (gy.double().view(thin, voxels) @ x.double().view(wide, voxels).t()).to(dtype)  # sums below 2^24: exact, then one rounding
    assert torch.equal(sa.conv3d_backward_weight(x, (thin, wide, 1, 1, 1), gy, 1, 0).view(thin, wide), want)
    conv = sa.FastConv3d(wide, thin, 1, device="cuda", dtype=dtype)
    conv(x).backward(gy)
    assert torch.equal(conv.weight.grad.view(thin, wide), want)
    assert torch.equal(conv.bias.grad, gy.double().sum((0, 2, 3, 4)).to(dtype))
