"""The small-volume convolution kernel on the launches of few workgroups (one channel block each) and below its plane line: against
float64, on both sides of the line, and the same bits from a depth shard's slab as from the padded volume."""

import ctypes

import pytest
import torch

import scaffold_amd as sa
from scaffold_amd import _lib
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


def _conv64(x, w):
    """The 3x3x3 convolution of padding 1 in float64: a matrix product a tap."""
    n, c, d, h, wd = x.shape
    xp = torch.nn.functional.pad(x.double().permute(0, 2, 3, 4, 1), (0, 0, 1, 1, 1, 1, 1, 1))
    w64 = w.double()
    y = torch.zeros((n * d * h * wd, w.shape[0]), dtype=torch.float64, device=x.device)
    for kd in range(3):
        for kh in range(3):
            for kw in range(3):
                rows = xp[:, kd:kd + d, kh:kh + h, kw:kw + wd].reshape(-1, c).contiguous()
                y += rows @ w64[:, :, kd, kh, kw].t().contiguous()
    return y.view(n, d, h, wd, -1).permute(0, 4, 1, 2, 3)


@pytest.mark.parametrize("cin,cout,spatial,fwd,dgrad", [
    (64, 128, (27, 61, 33), "brick", "brick"),   # planes past 32 x 32
    (64, 64, (9, 27, 50), "split", "brick"),     # ... from 240 pairs on
    (64, 64, (8, 27, 50), "brick", "brick"),     # 196
    (64, 128, (14, 13, 6), "split", "brick"),    # few pairs of 128 and more produced channels
    (128, 64, (14, 13, 6), "brick", "split"),    # ... in the gradient
    (128, 128, (9, 12, 8), "split", "split"),    # ... whose four sums are the slices', so that the data gradient comes too
    (128, 128, (4, 6, 12), "brick", "brick"),    # 16 pairs: too few
    (512, 512, (9, 9, 6), "split", "split"),     # a long reduction by the times, two slices
    (256, 256, (5, 8, 14), "split", "split"),    # in the place of eight slices: two rounds, their sums apart
    (256, 256, (3, 16, 12), "split", "split"),   # 72 pairs
    (256, 256, (11, 4, 9), "split", "split"),    # in the place of four: one chain a wavefront
    (128, 64, (33, 57, 50), "wide", "brick"),    # bricks would be sooner, in another order
    (128, 64, (31, 61, 65), "wide", "brick"),
])
def test_lines_that_the_times_draw(cin, cout, spatial, fwd, dgrad):
    x, gy, w = _operands(1, cin, cout, spatial, torch.bfloat16)
    d, h, wd = spatial
    shapes = (((1, cin, d, h, wd), 1), ((1, cin, d + 2, h, wd), (0, 1, 1)))
    geom = {k: [c3.launch_geometry(s, w.shape, 1, p, 1, torch.bfloat16, k) for s, p in shapes] for k in ("fwd", "bwd-data")}
    assert [g["kernel"] for g in geom["fwd"]] == [fwd] * 2 and [g["kernel"] for g in geom["bwd-data"]] == [dgrad] * 2
    slab = torch.zeros(shapes[1][0], dtype=x.dtype, device="cuda").contiguous(memory_format=CL)
    slab[:, :, 1:-1] = x
    for direction, got, from_slab, want in (
            ("fwd", sa.conv3d_forward(x, w, None, 1, 1), sa.conv3d_forward(slab, w, None, 1, (0, 1, 1)), _conv64(x, w)),
            ("bwd-data", sa.conv3d_backward_data(gy, w, x.shape, 1, 1), sa.conv3d_backward_data(gy, w, slab.shape, 1, (0, 1, 1))[:, :, 1:-1],
             _conv64(gy, w.flip(2, 3, 4).transpose(0, 1)))):
        # one rounding of the result on top of an fp32 sum of up to 27 * 512 terms
        for result in (got, from_slab):
            assert torch.all((result.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * want.abs().max())
        if len({g["slices"] for g in geom[direction]}) == 1:  # (slices are cut by a launch's own planes)
            assert torch.equal(got, from_slab)


@pytest.mark.parametrize("n,cin,cout,spatial", [(1, 64, 64, (9, 27, 50)), (1, 64, 128, (14, 13, 6)), (1, 512, 512, (9, 9, 6)), (1, 256, 256, (11, 4, 9)),
                                                (1, 128, 64, (33, 57, 50)), (1, 64, 64, (55, 28, 41)), (1, 512, 512, (12, 10, 14)), (2, 128, 64, (19, 30, 35)),
                                                (1, 32, 32, (11, 75, 97)), (2, 32, 64, (9, 21, 75)), (2, 128, 128, (11, 2, 6))])
@pytest.mark.parametrize("depth_padding", [1, 2])
def test_statistics_change_no_bit(n, cin, cout, spatial, depth_padding):
    """The result is the same bits with GroupNorm records and without, whichever launches estimated times choose for either."""
    x, _, w = _operands(n, cin, cout, spatial, torch.bfloat16)
    padding = (depth_padding, 1, 1)
    y = sa.conv3d_forward(x, w, None, 1, padding, gn_groups=8)
    assert hasattr(y, "_sfh_gn_partials") and torch.equal(y, sa.conv3d_forward(x, w, None, 1, padding))


@pytest.mark.parametrize("n,cin,cout,spatial", [(1, 128, 256, (8, 8, 8)), (1, 128, 128, (4, 6, 20)), (2, 128, 128, (5, 7, 9)),
                                                (1, 256, 256, (5, 8, 14)), (1, 256, 256, (8, 4, 20)), (2, 256, 256, (5, 4, 14)),
                                                (1, 256, 256, (11, 4, 9)), (2, 256, 512, (8, 3, 3)), (1, 64, 128, (14, 13, 6)), (2, 64, 128, (5, 7, 9)),
                                                (1, 64, 512, (7, 3, 6)), (3, 128, 256, (10, 3, 6)),
                                                (1, 512, 512, (9, 9, 6)), (1, 512, 256, (10, 8, 22)), (2, 512, 1024, (5, 4, 4))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_slices_and_their_bits(n, cin, cout, spatial, dtype):
    """A slice to a wavefront, or to a wavefront and round: the launch that leaves GroupNorm records is the bricks' in slices, the one without the small-volume kernel's,
    whose wavefronts (and rounds) add in the slices' order.  Against float64 as well."""
    x, _, w = _operands(n, cin, cout, spatial, dtype)
    assert c3.launch_geometry(x.shape, w.shape, 1, 1, 1, dtype, "fwd")["kernel"] == "split"
    b = torch.randn(cout, device="cuda").to(dtype)
    alone, recorded = sa.conv3d_forward(x, w, b, 1, 1), sa.conv3d_forward(x, w, b, 1, 1, gn_groups=8)
    assert recorded._sfh_gn_partials[1] == -(-cout * spatial[0] * spatial[1] * spatial[2] // 1024)  # of the launch that sums the slices
    assert torch.equal(alone, recorded)
    want = _conv64(x, w) + b.double().view(1, -1, 1, 1, 1)
    half_ulp = 2.0 ** -8 if dtype is torch.bfloat16 else 2.0 ** -11
    assert torch.all((alone.double() - want).abs() <= half_ulp * want.abs() + 1e-5 * want.abs().max())


def test_packed_launch_without_slices_takes_no_workspace():
    """The query has room for the slices behind GroupNorm records; the launch that makes none asks for none."""
    n, cin, cout, spatial = 1, 64, 128, (14, 13, 6)
    x, _, w = _operands(n, cin, cout, spatial, torch.bfloat16)
    packed, _ = c3.pack_weights(w, x.shape, 1, 1, 1)
    prob, lib = c3._Problem(x.shape, w.shape, 1, 1, 1, torch.bfloat16), _lib.lib()
    assert lib.sfh_conv3d_fwd_workspace_bytes(ctypes.byref(prob.desc), prob.code) > packed.numel()
    y = torch.empty_like(sa.conv3d_forward(x, w, None, 1, 1))
    _lib.check(lib.sfh_conv3d_fwd(ctypes.byref(prob.desc), prob.code, x.data_ptr(), packed.data_ptr(), None, None, y.data_ptr(), None, 0,
                                  _lib.SFH_FLAG_WEIGHT_PACKED, torch.cuda.current_stream().cuda_stream), "conv3d forward")
    assert torch.equal(y, sa.conv3d_forward(x, w, None, 1, 1))
