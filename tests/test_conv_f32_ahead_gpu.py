"""fp32 convolutions at the edges of their pipelines: operands requested ahead, passes dealt to two sets of wavefronts, one slice."""

import pytest
import torch

import scaffold_amd as sa
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "n,cin,cout,spatial,padding",
    [
        (1, 32, 32, (1, 1, 9), (1, 1, 1)),  # two passes, one per set
        (1, 32, 32, (1, 3, 8), (1, 1, 1)),  # three passes over three slices: one set idle
        (1, 64, 32, (5, 6, 17), (1, 1, 1)),  # rows that end inside a pass
        (2, 32, 64, (3, 5, 7), (0, 1, 1)),
        (1, 512, 512, (2, 3, 9), (1, 1, 1)),  # one slice, written in place; 32 chunks requested one ahead of the other
        (1, 96, 32, (4, 5, 6), (2, 2, 2)),
    ],
)
def test_fp32_exact(n, cin, cout, spatial, padding):
    """Whole numbers: every sum is exact in fp32, so the results are the oracle's bits."""
    prob = orc.ConvProblem(n=n, cin=cin, cout=cout, spatial=spatial, padding=padding, dtype=torch.float32)
    g = torch.Generator().manual_seed(5)
    x = torch.randint(-2, 3, prob.input_shape, generator=g).float()
    w = torch.randint(-2, 3, prob.weight_shape, generator=g).float()
    y = torch.nn.functional.conv3d(x.double(), w.double(), padding=padding)
    gy = torch.randint(-2, 3, y.shape, generator=g).float()
    gx_ref = torch.nn.grad.conv3d_input(x.shape, w.double(), gy.double(), padding=padding)
    gw_ref = torch.nn.grad.conv3d_weight(x.double(), w.shape, gy.double(), padding=padding)
    dev, cl = torch.device("cuda"), torch.channels_last_3d
    xd, wd, gyd = (t.to(dev).contiguous(memory_format=cl) for t in (x, w, gy))
    got = (sa.conv3d_forward(xd, wd, None, 1, padding), sa.conv3d_backward_data(gyd, wd, x.shape, 1, padding),
           sa.conv3d_backward_weight(xd, w.shape, gyd, 1, padding))
    for a, b in zip(got, (y, gx_ref, gw_ref)):
        assert torch.equal(a.cpu().double(), b)


def test_fp32_wgrad_leaves_out_what_belongs_to_no_output():
    """Without padding along W the last voxels of a row meet fewer taps: an infinity there must not reach the others as 0 x inf."""
    x = torch.ones((1, 32, 3, 3, 9))
    x[..., 8] = float("inf")  # met by kw = 2 of the last output only
    gy = torch.ones((1, 32, 1, 1, 7))
    ref = torch.nn.grad.conv3d_weight(x.double(), (32, 32, 3, 3, 3), gy.double())
    cl = torch.channels_last_3d
    got = sa.conv3d_backward_weight(x.cuda().contiguous(memory_format=cl), (32, 32, 3, 3, 3), gy.cuda().contiguous(memory_format=cl), 1, 0)
    assert torch.equal(got.cpu().double(), torch.where(torch.tensor([False, False, True]).expand_as(ref), float("inf"), 7.0).double())
