"""The fp32 weight gradient's steps of 64 voxels: rows of either segment width with cut ends, row tiles that end inside a plane, one range
and many, every padding, operands off the 16-byte grid, and infinities next to voxels that no output uses."""

import pytest
import torch

import scaffold_amd as sa

CL = torch.channels_last_3d
pytestmark = pytest.mark.gpu


def _reference(x, shape, gy, padding):
    return torch.nn.grad.conv3d_weight(x.cpu().double(), shape, gy.cpu().double(), padding=padding)


def _close(got, want):
    # fp32 sums of up to a few thousand unit-variance products: their round-off is within 2e-6 of the largest entry
    assert (got.cpu().double() - want).abs().max() <= 2e-6 * want.abs().max()


@pytest.mark.parametrize("padding", [(1, 1, 1), (0, 1, 1), (0, 0, 0), (2, 2, 2)])
@pytest.mark.parametrize("n,cin,cout,spatial", [
    (1, 32, 32, (3, 5, 8)),       # rows of 8
    (2, 32, 64, (4, 9, 7)),       # an odd row: its last pair has one voxel
    (1, 64, 32, (3, 4, 16)),      # one whole segment
    (1, 32, 32, (5, 7, 17)),      # a segment of one voxel
    (1, 32, 32, (9, 6, 33)),
    (1, 32, 32, (16, 24, 20)),    # more steps than workgroups
    (1, 320, 320, (3, 3, 3)),     # more blocks than compute units: one range each
])
def test_weight_gradient(n, cin, cout, spatial, padding):
    g = torch.Generator("cuda").manual_seed(2)
    x = torch.randn((n, cin, *spatial), generator=g, device="cuda").contiguous(memory_format=CL)
    out = [s + 2 * p - 2 for s, p in zip(spatial, padding)]
    gy = torch.randn((n, cout, *out), generator=g, device="cuda").contiguous(memory_format=CL)
    shape = (cout, cin, 3, 3, 3)
    got = sa.conv3d_backward_weight(x, shape, gy, 1, padding)
    _close(got, _reference(x, shape, gy, padding))
    # the same bits from views 4 bytes off the grid
    views = []
    for t in (x, gy):
        flat = torch.empty(t.numel() + 1, device="cuda")[1:].as_strided(t.shape, t.stride())
        flat.copy_(t)
        views.append(flat)
    assert torch.equal(sa.conv3d_backward_weight(views[0], shape, views[1], 1, padding), got)


@pytest.mark.parametrize("width", [9, 15, 19])
def test_infinities_that_no_output_meets(width):
    """With padding 0 the first outputs of a row do not exist for some taps: an infinity in x may reach only the taps that use it."""
    g = torch.Generator("cuda").manual_seed(4)
    x = torch.randn((1, 32, 4, 5, width), generator=g, device="cuda").contiguous(memory_format=CL)
    x[:, :, :, :, -1] = float("inf")  # met by kw = 2 of the last output only
    gy = torch.randn((1, 32, 2, 3, width - 2), generator=g, device="cuda").contiguous(memory_format=CL)
    got = sa.conv3d_backward_weight(x, (32, 32, 3, 3, 3), gy, 1, 0)
    assert torch.isfinite(got[..., :2]).all() and not torch.isfinite(got[..., 2]).any()


def test_a_row_of_two_gibibytes():
    """Offsets past 2^31 bytes inside a row, in the first, a middle and the last step: whole numbers, so the sums are exact."""
    width = 16_800_000
    g = torch.Generator("cuda").manual_seed(6)
    x = torch.randint(-1, 2, (width, 32), generator=g, device="cuda", dtype=torch.int8).float()
    gy = torch.randint(-1, 2, (width, 32), generator=g, device="cuda", dtype=torch.int8).float()
    as_volume = lambda t: t.view(1, 1, 1, width, 32).permute(0, 4, 1, 2, 3)
    got = sa.conv3d_backward_weight(as_volume(x), (32, 32, 3, 3, 3), as_volume(gy), 1, 1)
    want = torch.zeros_like(got, dtype=torch.float64)
    for kw in range(3):
        lo, hi = max(0, 1 - kw), min(width, width + 1 - kw)  # outputs whose voxel at this tap exists
        for part in range(lo, hi, 1 << 21):
            end = min(hi, part + (1 << 21))
            want[:, :, 1, 1, kw] += gy[part:end].double().t() @ x[part + kw - 1:end + kw - 1].double()
    assert torch.equal(got.double(), want)
