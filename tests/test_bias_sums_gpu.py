"""Bias gradients in fp32 against float64: how often a sum over many voxels is rounded on its way."""

import pytest
import torch

import scaffold_amd as sa

CL = torch.channels_last_3d
pytestmark = pytest.mark.gpu


def _rms(errors):
    return sum(e * e for e in errors) ** 0.5 / len(errors) ** 0.5


def _gradient(shape, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda").bfloat16().contiguous(memory_format=CL)


def _bound(terms, levels):
    # a rounding to the nearest fp32 is off by 2.5e-8 of the value (rms over mantissas); a partial sum of unit normals has the square
    # root of its count, the sum of magnitudes 0.8 of it: what `levels` roundings at full length come to
    return 2.5e-8 * (levels * terms) ** 0.5 / (0.8 * terms)


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
