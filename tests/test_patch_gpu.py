"""The 2x2x2 stride-2 kernels where their launch forms change: every register-kept width, several tiles per workgroup with a cut
last tile, fewer tiles than workgroups, and the three ways a weight can lie (packed, channels-last, anything else)."""

import pytest
import torch

import scaffold_amd as sa
from scaffold_amd import conv3d as c3

CL = torch.channels_last_3d
pytestmark = pytest.mark.gpu

#        n, cin, cout, small extents
SHAPES = [
    (1, 64, 32, (33, 36, 36)),      # 1337 tiles on 512 groups, the last one cut
    (1, 64, 96, (5, 6, 7)),         # three blocks: column pairs that reach over two taps
    (2, 128, 64, (17, 31, 33)),     # 1088 tiles, two samples in one tile
    (1, 128, 32, (1, 1, 1)),
    (1, 256, 128, (7, 9, 11)),
    (1, 256, 64, (16, 16, 17)),
    (1, 512, 256, (3, 5, 7)),
    (1, 512, 32, (12, 13, 14)),
    (1, 96, 32, (9, 10, 11)),       # no kept form: general kernels
    (1, 1024, 64, (2, 3, 3)),
]


def _operands(n, cin, cout, extents, dtype):
    g = torch.Generator("cuda").manual_seed(11)
    d, h, w = extents
    x = torch.randn((n, cin, d, h, w), generator=g, device="cuda").to(dtype).contiguous(memory_format=CL)
    gy = torch.randn((n, cout, 2 * d, 2 * h, 2 * w), generator=g, device="cuda").to(dtype).contiguous(memory_format=CL)
    wt = (torch.randn((cin, cout, 2, 2, 2), generator=g, device="cuda") / cin ** 0.5).to(dtype).contiguous(memory_format=CL)
    b = torch.randn(cout, generator=g, device="cuda").to(dtype)
    return x, gy, wt, b


def _close(got, want, dtype):
    # one rounding of the result (2^-9 bf16, 2^-12 fp16, relative to each element) on top of an fp32 sum of a few thousand terms
    ulp = 2.0 ** -8 if dtype is torch.bfloat16 else 2.0 ** -11
    scale = want.abs().max()
    assert torch.all((got.double() - want).abs() <= ulp * want.abs() + 1e-5 * scale)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,cin,cout,extents", SHAPES)
def test_forward(n, cin, cout, extents, dtype):
    x, gy, wt, b = _operands(n, cin, cout, extents, dtype)
    y = sa.conv_transpose3d_forward(x, wt, b, 2)
    rows = x.permute(0, 2, 3, 4, 1).reshape(-1, cin).double() @ wt.double().permute(0, 2, 3, 4, 1).reshape(cin, -1)
    d, h, w = extents
    want = rows.view(n, d, h, w, 2, 2, 2, cout).permute(0, 7, 1, 4, 2, 5, 3, 6).reshape(n, cout, 2 * d, 2 * h, 2 * w)
    _close(y, want + b.double()[None, :, None, None, None], dtype)
    # the same bits whatever the weight's layout: packed, another memory order, off the 16-byte grid
    _, pd = c3.pack_weights(wt, gy.shape, stride=2, padding=0)
    assert torch.equal(sa.conv_transpose3d_forward(x, wt, b, 2, packed_weight=pd), y)
    assert torch.equal(sa.conv_transpose3d_forward(x, wt.contiguous(), b, 2), y)
    flat = torch.empty(wt.numel() + 1, dtype=dtype, device="cuda")[1:]
    off = flat.as_strided(wt.shape, wt.stride())
    off.copy_(wt)
    assert torch.equal(sa.conv_transpose3d_forward(x, off, b, 2), y)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,cin,cout,extents,odd", [
    (1, 64, 32, (33, 36, 36), 0),     # tiles of 64 voxels, several per workgroup, the last one cut
    (1, 64, 32, (20, 20, 20), 1),     # 8000 voxels, under the rule's line; a big volume with a plane no window covers
    (1, 64, 32, (8, 32, 32), 1),      # 8192, on it
    (2, 128, 64, (17, 31, 33), 1),
    (1, 128, 64, (8, 17, 31), 0),
    (1, 256, 128, (13, 13, 13), 0),   # the reduction in two parts
    (1, 256, 128, (2, 32, 32), 1),
    (1, 512, 256, (9, 11, 13), 1),    # in four
    (1, 192, 32, (20, 21, 22), 0),    # three groups of two blocks
    (1, 64, 64, (16, 17, 18), 0),     # no kept form for this pair
])
def test_backward_data(n, cin, cout, extents, odd, dtype):
    _, _, wt, _ = _operands(n, cin, cout, (1, 1, 1), dtype)
    g = torch.Generator("cuda").manual_seed(5)
    d, h, w = extents
    big = torch.randn((n, cout, 2 * d + odd, 2 * h + odd, 2 * w + odd), generator=g, device="cuda").to(dtype).contiguous(memory_format=CL)
    b = torch.randn(cin, generator=g, device="cuda").to(dtype)
    y = sa.conv3d_forward(big, wt, b, 2, 0)
    rows = big[:, :, :2 * d, :2 * h, :2 * w].double().reshape(n, cout, d, 2, h, 2, w, 2).permute(0, 2, 4, 6, 3, 5, 7, 1).reshape(n * d * h * w, -1)
    want = rows @ wt.double().permute(2, 3, 4, 1, 0).reshape(-1, cin) + b.double()
    _close(y.permute(0, 2, 3, 4, 1).reshape(-1, cin), want, dtype)
    pf, _ = c3.pack_weights(wt, big.shape, stride=2, padding=0)
    assert torch.equal(sa.conv3d_forward(big, wt, b, 2, 0, packed_weight=pf), y)
    assert torch.equal(sa.conv3d_forward(big, wt.contiguous(), b, 2, 0), y)
    if not odd:
        gx = sa.conv_transpose3d_backward_data(big, wt, (n, cin, d, h, w), 2)
        _close(gx.permute(0, 2, 3, 4, 1).reshape(-1, cin), want - b.double(), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,cin,cout,extents", [
    (1, 64, 32, (1, 1, 1)),           # one voxel: one split, one half idle
    (1, 64, 32, (3, 3, 5)),           # 45: a cut round in the second half
    (1, 128, 96, (9, 10, 11)),        # six tiles
    (2, 128, 64, (11, 15, 18)),       # a range of voxels per XCD, the last one short
    (1, 512, 256, (4, 8, 8)),         # 64 tiles, one split
    (1, 512, 256, (5, 9, 9)),         # two splits
    (1, 64, 32, (33, 36, 36)),
    (1, 1024, 1056, (2, 2, 2)),       # more tiles than compute units
])
def test_backward_weight(n, cin, cout, extents, dtype):
    from scaffold_amd import transposed as ct

    x, gy, wt, _ = _operands(n, cin, cout, extents, dtype)
    d, h, w = extents
    big = gy.double().reshape(n, cout, d, 2, h, 2, w, 2).permute(0, 2, 4, 6, 3, 5, 7, 1).reshape(n * d * h * w, -1)
    want = (x.permute(0, 2, 3, 4, 1).reshape(-1, cin).double().t() @ big).view(cin, 2, 2, 2, cout).permute(0, 4, 1, 2, 3)
    gw = sa.conv_transpose3d_backward_weight(x, wt.shape, gy, 2)
    _close(gw, want, dtype)
    fw, fb = ct.conv_transpose3d_backward_weight_bias(x, wt.shape, gy, 2, grad_dtype=torch.float32)
    # fp32 sums of unit-variance products: 1e-6 of the largest entry covers their round-off at these counts
    assert (fw.double() - want).abs().max() <= 1e-6 * want.abs().max()
    bias = gy.double().sum((0, 2, 3, 4))
    assert (fb.double() - bias).abs().max() <= 1e-6 * gy.double().abs().sum((0, 2, 3, 4)).max()
    bw, _ = ct.conv_transpose3d_backward_weight_bias(x, wt.shape, gy, 2)
    assert torch.equal(bw, gw)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("odd", [0, 1])
@pytest.mark.parametrize("n,cin,cout,extents", [
    (1, 64, 32, (2, 3, 5)),           # a round that is cut
    (2, 64, 32, (3, 5, 7)),           # the step of a walk is longer than a row, than a plane, and reaches over samples
    (1, 64, 32, (12, 12, 12)),        # a range per round
    (1, 64, 32, (16, 17, 30)),        # 255 rounds: the last of one half
    (1, 64, 32, (17, 17, 29)),        # 262: two
    (2, 128, 64, (9, 10, 11)),        # 62 rounds of four tiles
    (1, 512, 256, (3, 5, 6)),         # three rounds of 64
    (1, 512, 256, (5, 5, 5)),         # four: two halves
    (2, 128, 64, (11, 15, 18)),
])
def test_weight_gradient_of_small_and_odd_volumes(n, cin, cout, extents, odd, dtype):
    """The stride-2 convolution's weight gradient is the same kernel with the roles turned; with an odd big extent a walk over the small
    voxels skips the plane, row or voxel that no window covers."""
    g = torch.Generator("cuda").manual_seed(3)
    d, h, w = extents
    small = torch.randint(-2, 3, (n, cin, d, h, w), generator=g, device="cuda").to(dtype).contiguous(memory_format=CL)
    big = torch.randint(-2, 3, (n, cout, 2 * d + odd, 2 * h + odd, 2 * w + odd), generator=g, device="cuda").to(dtype).contiguous(memory_format=CL)
    got = sa.conv3d_backward_weight(big, (cin, cout, 2, 2, 2), small, 2, 0, grad_dtype=torch.float32)
    rows = big[:, :, :2 * d, :2 * h, :2 * w].double().reshape(n, cout, d, 2, h, 2, w, 2).permute(0, 2, 4, 6, 3, 5, 7, 1).reshape(n * d * h * w, -1)
    want = (small.permute(0, 2, 3, 4, 1).reshape(-1, cin).double().t() @ rows).view(cin, 2, 2, 2, cout).permute(0, 4, 1, 2, 3)
    assert torch.equal(got.double(), want)  # whole numbers whose sums stay far below 2^24
