"""The 2x2x2 weight gradient in fp32 against float64: how often a sum over the voxels is rounded on its way."""

import pytest
import torch

import scaffold_amd as sa

CL = torch.channels_last_3d
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cin,cout,extents", [
    (1, 64, 32, (7, 7, 5)),      # eight ranges of a round
    (2, 128, 64, (6, 8, 5)),
    (1, 256, 128, (4, 8, 8)),
    (1, 512, 256, (4, 5, 6)),    # one range
    (1, 512, 256, (4, 8, 8)),    # 64 tiles: few ranges
    (1, 512, 256, (8, 8, 8)),
])
def test_small_volumes(n, cin, cout, extents):
    d, h, w = extents
    voxels, errors = n * d * h * w, []
    for seed in range(8):
        g = torch.Generator("cuda").manual_seed(seed)
        x = torch.randn((n, cin, d, h, w), generator=g, device="cuda").bfloat16().contiguous(memory_format=CL)
        gy = torch.randn((n, cout, 2 * d, 2 * h, 2 * w), generator=g, device="cuda").bfloat16().contiguous(memory_format=CL)
        got = sa.conv_transpose3d_backward_weight(x, (cin, cout, 2, 2, 2), gy, 2, grad_dtype=torch.float32)
        big = gy.double().reshape(n, cout, d, 2, h, 2, w, 2).permute(0, 2, 4, 6, 3, 5, 7, 1).reshape(voxels, -1)
        want = (x.permute(0, 2, 3, 4, 1).reshape(voxels, cin).double().t() @ big).view(cin, 2, 2, 2, cout).permute(0, 4, 1, 2, 3)
        errors.append(((got.double() - want).norm() / want.norm()).item())
    # The matrix unit's 16 products round hardly at all; a tree over them rounds log2(voxels / 16) times at full length, each time by
    # 2.7e-8 rms (an addition to the nearest). 0.4 for what a short chain or a cut range adds; one chain per parity of step adds 0.5.
    levels = torch.tensor(voxels / 16).log2().item() + 0.4
    assert (sum(e * e for e in errors) / len(errors)) ** 0.5 <= 2.7e-8 * levels ** 0.5
