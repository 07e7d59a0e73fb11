"""The small-volume convolution kernel on the launches of few workgroups (one channel block each) and below its plane line: against
float64, on both sides of the line, and the same bits from a depth shard's slab as from the padded volume."""

import pytest
import torch

import scaffold_amd as sa
from scaffold_amd import conv3d as c3

CL = torch.channels_last_3d
pytestmark = pytest.mark.gpu


def _operands(n, cin, cout, spatial, dtype):
    g = torch.Generator("cuda").manual_seed(9)
    x = torch.randn((n, cin, *spatial), generator=g, device="cuda").to(dtype).contiguous(memory_format=CL)
    gy = torch.randn((n, cout, *spatial), generator=g, device="cuda").to(dtype).contiguous(memory_format=CL)
    w = (torch.randn((cout, cin, 3, 3, 3), generator=g, device="cuda") / (27 * cin) ** 0.5).to(dtype).contiguous(memory_format=CL)
    return x, gy, w


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,cin,cout,spatial,kernel", [
    (1, 64, 64, (16, 16, 16), "split"),     # 64 pairs: the first on the line
    (1, 64, 64, (14, 16, 16), "brick"),     # 56
    (1, 64, 64, (15, 13, 15), "split"),     # 64 of cut bricks, one channel block each
    (1, 128, 128, (7, 9, 30), "split"),     # 96
    (1, 192, 128, (13, 9, 12), "split"),    # 84, three rounds of two chunks
    (1, 256, 128, (9, 12, 12), "brick"),    # 60
    (1, 256, 128, (20, 12, 14), "split"),   # 120
    (1, 256, 256, (8, 16, 16), "split"),    # 128: the last with one block each
    (1, 256, 256, (9, 16, 16), "split"),    # 160: two
    (1, 512, 256, (16, 16, 16), "split"),   # 256
])
def test_both_sides_of_the_lines(n, cin, cout, spatial, kernel, dtype):
    x, gy, w = _operands(n, cin, cout, spatial, dtype)
    assert c3.launch_geometry(x.shape, w.shape, 1, 1, 1, dtype, "fwd")["kernel"] == kernel
    # one rounding of the result on top of an fp32 sum of up to 27 * 512 terms
    ulp = 2.0 ** -8 if dtype is torch.bfloat16 else 2.0 ** -11
    for got, want in ((sa.conv3d_forward(x, w, None, 1, 1), torch.nn.functional.conv3d(x.cpu().double(), w.cpu().double(), padding=1)),
                      (sa.conv3d_backward_data(gy, w, x.shape, 1, 1),
                       torch.nn.functional.conv_transpose3d(gy.cpu().double(), w.cpu().double(), padding=1))):
        assert torch.all((got.cpu().double() - want).abs() <= ulp * want.abs() + 1e-5 * want.abs().max())


@pytest.mark.parametrize("cin,cout,spatial", [(64, 64, (16, 16, 16)), (128, 128, (7, 9, 30)), (64, 128, (9, 16, 15)), (256, 256, (8, 16, 16))])
def test_slab_and_padded_volume_agree(cin, cout, spatial):
    x, gy, w = _operands(1, cin, cout, spatial, torch.bfloat16)
    d, h, wd = spatial
    slab = torch.zeros((1, cin, d + 2, h, wd), dtype=x.dtype, device="cuda").contiguous(memory_format=CL)
    slab[:, :, 1:-1] = x
    assert torch.equal(sa.conv3d_forward(slab, w, None, 1, (0, 1, 1)), sa.conv3d_forward(x, w, None, 1, 1))
    assert torch.equal(sa.conv3d_backward_data(gy, w, slab.shape, 1, (0, 1, 1))[:, :, 1:-1], sa.conv3d_backward_data(gy, w, x.shape, 1, 1))
