"""Bias gradients in fp32 against float64: how often a sum over many voxels is rounded on its way."""

import pytest
import torch

import scaffold_amd as sa
from scaffold_amd import transposed as ct

CL = torch.channels_last_3d
pytestmark = pytest.mark.gpu


def _rms(errors):
    return sum(e * e for e in errors) ** 0.5 / len(errors) ** 0.5


def _gradient(shape, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda").bfloat16().contiguous(memory_format=CL)


def _bound(terms, levels):
    # a rounding to the nearest fp32 is off by 2.7e-8 of the value (rms over mantissas); a partial sum of unit normals has the square
    # root of its count, the sum of magnitudes 0.8 of it: what `levels` roundings at full length come to
    return 2.7e-8 * (levels * terms) ** 0.5 / (0.8 * terms)


@pytest.mark.parametrize("n,wide,thin,spatial", [(1, 32, 6, (32, 32, 32)), (1, 64, 6, (64, 64, 64)), (2, 32, 6, (44, 60, 75))])
def test_head(n, wide, thin, spatial):
    errors = []
    for seed in range(24):
        x, gy = _gradient((n, wide, *spatial), 100 + seed), _gradient((n, thin, *spatial), seed)
        conv = sa.FastConv3d(wide, thin, 1, device="cuda")
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = conv(x)
        y.backward(gy)
        want = gy.double().sum((0, 2, 3, 4))
        errors.append(((conv.bias.grad.double() - want).norm() / gy.double().abs().sum((0, 2, 3, 4)).norm()).item())
    # eight levels over 256 slices and six of the rounds inside a workgroup; chains of 32 slices came to 15 to 26
    assert _rms(errors) <= _bound(n * spatial[0] * spatial[1] * spatial[2], 14)


@pytest.mark.parametrize("n,cin,cout,extents", [(1, 64, 32, (64, 64, 64)), (1, 64, 32, (32, 64, 64)), (1, 128, 64, (48, 40, 56)), (1, 512, 256, (12, 10, 14))])
def test_up_convolution(n, cin, cout, extents):
    errors = []
    x = _gradient((n, cin, *extents), 100)
    for seed in range(12):
        gy = _gradient((n, cout, *(2 * e for e in extents)), seed)
        _, got = ct.conv_transpose3d_backward_weight_bias(x, (cin, cout, 2, 2, 2), gy, 2, grad_dtype=torch.float32)
        errors.append(((got.double() - gy.double().sum((0, 2, 3, 4))).norm() / gy.double().abs().sum((0, 2, 3, 4)).norm()).item())
    # a range's sum is rounded once; eight levels over 256 ranges, and the result's own
    assert _rms(errors) <= _bound(8 * n * extents[0] * extents[1] * extents[2], 10)
