"""The few-channel 3x3x3 stem on the matrix cores (1 to 4 input channels, 32 or 64 output channels), through the C ABI.

Integer draws whose sums are exactly representable, bit for bit against the fp64 oracle and against the direct kernels, at
the sizes where its tiles can go wrong: one voxel, a tile and one more along each axis, cut tiles on all three, several
tiles per workgroup, two samples, the three padding forms of a depth shard."""

import pytest
import torch

import scaffold_amd as sa
from oracle import oracle as orc
from tests.test_conv_gpu import check_exact
from tests.test_gn_partials_gpu import check_records

pytestmark = pytest.mark.gpu
CL = torch.channels_last_3d

SHAPES = [
    # (n, cin, cout, spatial, padding, bias)
    (1, 1, 32, (1, 1, 1), (1, 1, 1), True),
    (1, 3, 64, (4, 4, 32), (1, 1, 1), False),       # one whole tile of the forward, two of the weight gradient
    (1, 3, 32, (5, 5, 33), (1, 1, 1), True),        # one voxel past the tile on every axis
    (2, 3, 64, (6, 9, 40), (0, 1, 1), False),       # shard form, two samples
    (1, 2, 32, (3, 7, 31), (1, 1, 1), False),
    (1, 4, 64, (7, 6, 35), (2, 0, 1), True),
    (2, 1, 64, (9, 10, 65), (0, 1, 1), False),
    (1, 3, 32, (33, 70, 66), (1, 1, 1), False),     # more tiles than workgroups: a workgroup walks several
    (1, 1, 32, (34, 66, 65), (1, 1, 1), False),
]


@pytest.mark.parametrize("direction", ("fwd", "bwd-weight"))
@pytest.mark.parametrize("n,cin,cout,spatial,padding,bias", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_stem_exact(device, dtype, n, cin, cout, spatial, padding, bias, direction):
    prob = orc.ConvProblem(n=n, cin=cin, cout=cout, spatial=spatial, padding=padding, bias=bias, dtype=dtype)
    got = check_exact(prob, direction, device)
    assert torch.equal(got, check_exact(prob, direction, device, force_generic=True))


@pytest.mark.parametrize("n,cin,cout,spatial,padding,groups", [
    (1, 3, 64, (5, 6, 40), (1, 1, 1), 8),
    (2, 3, 32, (37, 40, 66), (0, 1, 1), 8),         # two samples, several tiles per workgroup
    (1, 4, 32, (4, 4, 5), (1, 1, 1), 1),
    (1, 1, 32, (33, 65, 64), (1, 1, 1), 4),
])
def test_stem_leaves_the_moments_of_its_output(device, n, cin, cout, spatial, padding, groups):
    g = torch.Generator().manual_seed(11)
    x = torch.randn((n, cin, *spatial), generator=g).to(torch.bfloat16).to(device).contiguous(memory_format=CL)
    w = (torch.randn((cout, cin, 3, 3, 3), generator=g) / 5).to(torch.bfloat16).to(device).contiguous(memory_format=CL)
    plain = sa.conv3d_forward(x, w, None, 1, padding)
    y = sa.conv3d_forward(x, w, None, 1, padding, gn_groups=groups)
    assert torch.equal(plain, y)
    check_records(y, groups, y._sfh_gn_partials)


@pytest.mark.parametrize("cin", [1, 3])
def test_stem_keeps_nan_and_inf_to_their_windows(device, cin):
    """The contraction is padded to whole k-steps with zero weights; a NaN times a zero weight would be a NaN."""
    x = torch.zeros((1, cin, 9, 9, 40), dtype=torch.bfloat16, device=device).contiguous(memory_format=CL)
    w = torch.ones((32, cin, 3, 3, 3), dtype=torch.bfloat16, device=device).contiguous(memory_format=CL)
    x[0, 0, 4, 4, 20] = float("nan")
    x[0, cin - 1, 0, 8, 39] = float("inf")
    y = sa.conv3d_forward(x, w, None, 1, 1).float().cpu()
    nan, inf = torch.zeros(9, 9, 40, dtype=torch.bool), torch.zeros(9, 9, 40, dtype=torch.bool)
    nan[3:6, 3:6, 19:22] = True
    inf[:2, 7:, 38:] = True
    assert torch.equal(torch.isnan(y[0]), nan.expand(32, -1, -1, -1)) and torch.equal(torch.isinf(y[0]), inf.expand(32, -1, -1, -1))
    assert (y[0][:, ~(nan | inf)] == 0).all()


def test_stem_weight_gradient_in_fp32_rounds_to_the_16_bit_one(device):
    g = torch.Generator().manual_seed(12)
    x = torch.randn((1, 3, 6, 7, 37), generator=g).to(torch.bfloat16).to(device).contiguous(memory_format=CL)
    gy = torch.randn((1, 64, 6, 7, 37), generator=g).to(torch.bfloat16).to(device).contiguous(memory_format=CL)
    g16 = sa.conv3d_backward_weight(x, (64, 3, 3, 3, 3), gy, 1, 1)
    g32 = sa.conv3d_backward_weight(x, (64, 3, 3, 3, 3), gy, 1, 1, grad_dtype=torch.float32)
    assert g32.dtype is torch.float32 and torch.equal(g32.to(torch.bfloat16), g16)


@pytest.mark.parametrize("cin", [1, 3])
@pytest.mark.parametrize("spatial,padding", [((3, 6, 40), (1, 1, 1)), ((2, 4, 33), (1, 1, 1)), ((5, 7, 17), (0, 1, 1)), ((3, 5, 66), (2, 0, 0)),
                                             ((4, 4, 47), (1, 2, 2))])
def test_stem_weight_gradient_keeps_nan_and_inf_to_their_taps(device, cin, spatial, padding):
    """A tile reaches past the output: a voxel there has no gradient, and an infinity that only its taps would meet (0 x
    infinity) stays out.  One infinity or NaN at a corner or edge of the input: exactly the taps that some output reads it
    through are not finite, the others are the sums without it."""
    shape = (32, cin, 3, 3, 3)
    g = torch.Generator().manual_seed(13)
    x = torch.randint(-2, 3, (1, cin, *spatial), generator=g).to(torch.bfloat16)
    out = [s + 2 * p - 2 for s, p in zip(spatial, padding)]
    gy = torch.randint(-1, 2, (1, 32, *out), generator=g).to(torch.bfloat16)
    gy[gy == 0] = 2
    d, h, w = (s - 1 for s in spatial)
    for at, value in (((d, h, w), "inf"), ((0, 0, w), "nan"), ((d, 0, 0), "inf"), ((d // 2, h, w), "inf"), ((0, h, w // 2), "nan")):
        clean, dirty = x.clone(), x.clone()
        clean[(0, cin - 1, *at)], dirty[(0, cin - 1, *at)] = 0, float(value)
        want = torch.nn.grad.conv3d_weight(clean.double(), shape, gy.double(), 1, padding)
        met = torch.zeros(cin, 3, 3, 3, dtype=torch.bool)
        for tap in torch.cartesian_prod(*[torch.arange(3)] * 3).tolist():
            met[(cin - 1, *tap)] = all(0 <= a + p - t < o for a, p, t, o in zip(at, padding, tap, out))
        got = sa.conv3d_backward_weight(dirty.to(device).contiguous(memory_format=CL), shape, gy.to(device).contiguous(memory_format=CL), 1,
                                        padding, grad_dtype=torch.float32).cpu()
        assert torch.equal(~torch.isfinite(got), met.expand(32, -1, -1, -1, -1)), (at, value)
        assert torch.equal(got[:, ~met].double(), want[:, ~met])
