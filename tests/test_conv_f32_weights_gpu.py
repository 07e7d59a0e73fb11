"""fp32 convolutions read a channels-last weight where it lies and pack any other: the same bits either way."""

import pytest
import torch

import scaffold_amd as sa

pytestmark = pytest.mark.gpu


def _placed(w, layout):
    if layout == "first":
        return w.contiguous()
    if layout == "shifted":  # channels-last, 4 bytes off the 16-byte grid
        room = torch.empty(w.numel() + 1, device=w.device)[1:]
        o, i = w.shape[:2]
        out = room.as_strided(w.shape, (27 * i, 1, 9 * i, 3 * i, i))
        assert out.data_ptr() % 16 == 4
        return out.copy_(w)
    return w.permute(0, 1, 4, 3, 2).contiguous(memory_format=torch.channels_last_3d).permute(0, 1, 4, 3, 2)  # kd innermost of the taps


@pytest.mark.parametrize("layout", ["first", "shifted", "turned"])
@pytest.mark.parametrize(
    "n,cin,cout,spatial",
    [
        (1, 32, 32, (31, 30, 27)),  # 4x4x8
        (1, 96, 128, (31, 30, 27)), # 8x8x8, four sub-tiles
        (1, 48, 32, (33, 13, 9)),   # 2x2x16 in two parts of unequal length; the data gradient's 48 channels run elsewhere
        (2, 32, 64, (9, 41, 9)),    # 2x4x16
        (1, 32, 64, (33, 7, 9)),    # 2x4x8 in two parts
        (1, 32, 32, (5, 7, 7)),     # 2x2x8 in four parts, two of them without a chunk
        (1, 160, 32, (5, 3, 9)),    # ten chunks in four parts
        (1, 64, 64, (63, 9, 30)),   # a data gradient past the line up to which it reads the weight where it lies
        (2, 64, 32, (20, 33, 41)),  # a forward past its line
    ],
)
def test_forms_of_a_weight(n, cin, cout, spatial, layout):
    g = torch.Generator(device="cuda").manual_seed(5)
    cl = torch.channels_last_3d
    x = torch.randn(n, cin, *spatial, generator=g, device="cuda").contiguous(memory_format=cl)
    gy = torch.randn(n, cout, *spatial, generator=g, device="cuda").contiguous(memory_format=cl)
    w = torch.randn(cout, cin, 3, 3, 3, generator=g, device="cuda").contiguous(memory_format=cl)
    other = _placed(w, layout)
    assert torch.equal(sa.conv3d_forward(x, w, None, 1, 1), sa.conv3d_forward(x, other, None, 1, 1))
    assert torch.equal(sa.conv3d_backward_data(gy, w, x.shape, 1, 1), sa.conv3d_backward_data(gy, other, x.shape, 1, 1))
