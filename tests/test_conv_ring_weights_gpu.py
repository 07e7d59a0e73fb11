"""Convolutions of 32 reduction channels read a channels-last weight where it lies and pack any other: the same bits either way.
Rows of more than 16 voxels and shorter ones have kernels of their own."""

import pytest
import torch

import scaffold_amd as sa

pytestmark = pytest.mark.gpu


def _placed(w, layout):
    if layout == "first":
        return w.contiguous()
    room = torch.empty(w.numel() + 1, device=w.device, dtype=w.dtype)[1:]  # channels-last, 2 bytes off the 16-byte grid
    o, i = w.shape[:2]
    return room.as_strided(w.shape, (27 * i, 1, 9 * i, 3 * i, i)).copy_(w)


def _weight(g, cout, cin, dtype):
    return torch.randn(cout, cin, 3, 3, 3, generator=g, device="cuda").to(dtype).contiguous(memory_format=torch.channels_last_3d)


@pytest.mark.parametrize("layout", ["first", "shifted"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,wide,spatial", [(1, 32, (4, 8, 32)), (1, 96, (5, 9, 33)), (2, 64, (3, 7, 17)), (1, 32, (40, 24, 65)), (1, 32, (4, 8, 16)),
                                            (1, 96, (33, 9, 13)), (2, 64, (3, 5, 7)), (1, 32, (40, 41, 8))])
def test_forms_of_a_weight(n, wide, spatial, dtype, layout):
    g = torch.Generator(device="cuda").manual_seed(5)
    cl = torch.channels_last_3d
    narrow = torch.randn(n, 32, *spatial, generator=g, device="cuda").to(dtype).contiguous(memory_format=cl)
    bias = torch.randn(wide, generator=g, device="cuda").to(dtype)
    w = _weight(g, wide, 32, dtype)
    other = _placed(w, layout)
    for b in (None, bias):
        assert torch.equal(sa.conv3d_forward(narrow, w, b, 1, 1), sa.conv3d_forward(narrow, other, b, 1, 1))
    y, packed = (sa.conv3d_forward(narrow, v, None, 1, 1, gn_groups=8) for v in (w, other))
    assert torch.equal(y, packed)
    if hasattr(packed, "_sfh_gn_partials"):
        assert torch.equal(y._sfh_gn_partials[0], packed._sfh_gn_partials[0])
    w = _weight(g, 32, wide, dtype)
    shape = (n, wide, *spatial)
    assert torch.equal(sa.conv3d_backward_data(narrow, w, shape, 1, 1), sa.conv3d_backward_data(narrow, _placed(w, layout), shape, 1, 1))
