"""fp32 convolutions over the bricks their launch chooses from: cut bricks, reductions in parts of unequal length."""

import pytest
import torch

import scaffold_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "n,cin,cout,spatial,padding",
    [
        (1, 96, 128, (31, 30, 27), 1),  # 8x8x8, the forward; the data gradient too
        (2, 32, 64, (33, 7, 9), 1),     # 4x4x8
        (2, 48, 64, (9, 41, 9), 1),     # 2x4x16
        (1, 32, 64, (33, 7, 9), 1),     # 2x4x8 in two parts
        (1, 32, 64, (33, 13, 9), 1),    # 2x2x16 in two parts
        (1, 48, 32, (33, 13, 9), 1),    # the same, a chunk in the first part more than in the second
        (1, 32, 32, (5, 7, 7), 1),      # 2x2x8 in four parts, two of them without a chunk
        (1, 160, 32, (5, 3, 9), 1),     # ten chunks in four parts
        (1, 96, 64, (4, 6, 17), 2),
        (1, 64, 32, (6, 5, 11), 0),
    ],
)
def test_bricks(n, cin, cout, spatial, padding):
    """Whole numbers: every sum is exact in fp32 in any order, so the results are the stock convolution's bits."""
    g = torch.Generator().manual_seed(7)
    x = torch.randint(-2, 3, (n, cin, *spatial), generator=g).float()
    w = torch.randint(-2, 3, (cout, cin, 3, 3, 3), generator=g).float()
    bias = torch.randint(-2, 3, (cout,), generator=g).float()
    y = torch.nn.functional.conv3d(x, w, bias, padding=padding)
    gy = torch.randint(-2, 3, y.shape, generator=g).float()
    gx = torch.nn.functional.conv_transpose3d(gy, w, padding=padding)
    cl = torch.channels_last_3d
    xd, wd, gyd = (t.cuda().contiguous(memory_format=cl) for t in (x, w, gy))
    assert torch.equal(sa.conv3d_forward(xd, wd, bias.cuda(), 1, padding).cpu(), y)
    assert torch.equal(sa.conv3d_backward_data(gyd, wd, x.shape, 1, padding).cpu(), gx)
