"""The brick kernel's row classes beyond the row length's own, and where it takes the wide kernel's place: results against float64 at
volumes that leave every brick cut, GroupNorm records, pairs of tensors, and the same bits from a depth shard's slab."""

import pytest
import torch

import scaffold_amd as sa
from scaffold_amd import conv3d as c3

CL = torch.channels_last_3d
pytestmark = pytest.mark.gpu


def _tensor(shape, seed, dtype=torch.bfloat16, scale=1.0):
    g = torch.Generator("cuda").manual_seed(seed)
    return (torch.randn(shape, generator=g, device="cuda") * scale).to(dtype).contiguous(memory_format=CL)


def _planes(x, w, planes):
    """Output planes of the padded convolution in float64, on the GPU (two-dimensional convolutions per depth tap)."""
    out = []
    for d in planes:
        acc = 0.0
        for k in range(3):
            if 0 <= d + k - 1 < x.shape[2]:
                acc = acc + torch.nn.functional.conv2d(x[:, :, d + k - 1].double(), w[:, :, k].double(), padding=1)
        out.append(acc)
    return torch.stack(out, 2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,cin,cout,spatial,kernel", [
    (1, 64, 64, (60, 72, 48), "brick"),     # rows of 16
    (2, 64, 64, (22, 30, 37), "brick"),     # half bricks of 8 x 8
    (1, 64, 64, (50, 49, 81), "brick"),
    (1, 64, 32, (24, 50, 70), "brick"),     # one block
    (1, 96, 96, (33, 41, 50), "brick"),     # three blocks of one
    (1, 128, 64, (65, 77, 90), "brick"),    # in the wide kernel's place: 9 x 20 x 3 of its bricks
    (1, 128, 64, (48, 64, 60), "wide"),     # two rounds of them or fewer stay
    (10, 128, 64, (64, 28, 28), "brick"),   # planes that the small-volume kernel would take
])
def test_planes_match_float64(n, cin, cout, spatial, kernel, dtype):
    x, w = _tensor((n, cin, *spatial), 1, dtype), _tensor((cout, cin, 3, 3, 3), 2, dtype, (27 * cin) ** -0.5)
    assert c3.launch_geometry(x.shape, w.shape, 1, 1, 1, dtype, "fwd")["kernel"] == kernel
    y = sa.conv3d_forward(x, w, None, 1, 1, gn_groups=8)
    planes = sorted({0, 1, spatial[0] // 2, spatial[0] - 2, spatial[0] - 1})
    want = _planes(x, w, planes)
    ulp = 2.0 ** -8 if dtype is torch.bfloat16 else 2.0 ** -11  # one rounding, on top of an fp32 sum
    assert torch.all((y[:, :, planes].double() - want).abs() <= ulp * want.abs() + 1e-5 * want.abs().max())
    # the statistics a GroupNorm takes from the launch are those of what it wrote
    norm = sa.FastGroupNorm(8, cout, activation="relu", device="cuda")
    with torch.autocast("cuda", dtype=dtype):
        assert torch.allclose(norm(y).float(), norm(y.clone()).float(), atol=2e-2)
    # the data gradient is the same kernel on the flipped weight
    gy = _tensor(y.shape, 3, dtype)
    gx = sa.conv3d_backward_data(gy, w, x.shape, 1, 1)
    want = _planes(gy, w.transpose(0, 1).flip(2, 3, 4), planes)
    assert torch.all((gx[:, :, planes].double() - want).abs() <= ulp * want.abs() + 1e-5 * want.abs().max())


@pytest.mark.parametrize("spatial", [(65, 77, 90), (49, 80, 112)])
def test_pairs_and_slabs(spatial):
    x, w = _tensor((1, 128, *spatial), 4), _tensor((64, 128, 3, 3, 3), 5, scale=0.02)
    y = sa.conv3d_forward(x, w, None, 1, 1)
    a, b = (x[:, s].contiguous(memory_format=CL) for s in (slice(0, 64), slice(64, 128)))
    assert torch.equal(c3.conv3d_forward_pair(a, b, w, None, 1, 1, 1), y)
    # unequal cuts stay refused, whichever kernel serves the volume
    c, d = (x[:, s].contiguous(memory_format=CL) for s in (slice(0, 32), slice(32, 128)))
    assert not c3.is_supported_pair(c, d, w, None, 1, 1, 1)
    slab = torch.zeros((1, 128, spatial[0] + 2, *spatial[1:]), dtype=x.dtype, device="cuda").contiguous(memory_format=CL)
    slab[:, :, 1:-1] = x
    assert torch.equal(sa.conv3d_forward(slab, w, None, 1, (0, 1, 1)), y)
    w2 = _tensor((128, 64, 3, 3, 3), 6, scale=0.02)
    small, gy = (1, 64, *spatial), _tensor((1, 128, *spatial), 7)
    padded = sa.conv3d_backward_data(gy, w2, small, 1, 1)
    shard = sa.conv3d_backward_data(gy, w2, (1, 64, spatial[0] + 2, *spatial[1:]), 1, (0, 1, 1))
    assert torch.equal(shard[:, :, 1:-1], padded)
