"""Packing a dense channels-last weight in tiles of 32 x 32 channels against the piece-by-piece packing of any other layout: the same
bytes for both forms, either alone, every tap count, fp32 masters, more weights than one launch's table holds."""

import pytest
import torch

from scaffold_amd import conv3d as c3

CL = torch.channels_last_3d
pytestmark = pytest.mark.gpu


def _pack(w, k, **kw):
    return c3.pack_weights(w, (1, w.shape[1], 8, 8, 8), stride=2 if k == 2 else 1, padding=0 if k == 2 else 1, **kw)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cout,cin,k", [(32, 32, 3), (64, 32, 3), (32, 96, 3), (160, 64, 3), (64, 128, 2), (32, 32, 2)])
def test_tiles_equal_pieces(cout, cin, k, dtype):
    w = torch.randn((cout, cin, k, k, k), generator=torch.Generator("cuda").manual_seed(3), device="cuda").to(dtype)
    dense = w.contiguous(memory_format=CL)
    rows, cols = _pack(dense, k)
    other = w.contiguous()  # [c0][c1][tap]: piece by piece
    off = torch.empty(w.numel() + 1, dtype=dtype, device="cuda")[1:].as_strided(dense.shape, dense.stride())
    off.copy_(dense)        # the dense order off the 16-byte grid
    for source in (other, off):
        r, c = _pack(source, k)
        assert torch.equal(r.view(torch.int16), rows.view(torch.int16)) and torch.equal(c.view(torch.int16), cols.view(torch.int16))
    r, none = _pack(dense, k, backward_data=False)
    assert none is None and torch.equal(r.view(torch.int16), rows.view(torch.int16))
    none, c = _pack(dense, k, forward=False)
    assert none is None and torch.equal(c.view(torch.int16), cols.view(torch.int16))
