"""Packing a dense channels-last weight in tiles of 32 x 32 channels against the piece-by-piece packing of any other layout: the same
bytes for both forms, either alone, every tap count, off the 16-byte grid, and more weights than one launch's table holds."""

import ctypes

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


def _launches(graph):
    """Nodes of a captured graph, from the HIP runtime that torch has loaded."""
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64.so" in line)
    count = ctypes.c_size_t()
    assert ctypes.CDLL(path).hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(count)) == 0
    return count.value


@pytest.mark.parametrize("dense,other,launches", [
    (72, 0, 1),      # both forms of a full table
    (73, 0, 2),
    (0, 24, 1),      # 48 jobs of the piece-by-piece table
    (0, 25, 2),
    (80, 60, None),  # both tables overflow, in turn
])
def test_more_weights_than_a_table_holds(dense, other, launches):
    g = torch.Generator("cuda").manual_seed(8)
    packs = []
    for i in range(dense + other):
        cout, cin = (32, 64)[i % 2], (32, 96)[i % 3 == 0]
        w = torch.randn((cout, cin, 3, 3, 3), generator=g, device="cuda").bfloat16()
        take_dense = i * dense // (dense + other) != (i + 1) * dense // (dense + other)  # spread over the list
        packs.append(c3.PackedWeights(w.contiguous(memory_format=CL) if take_dense else w.contiguous(), (1, cin, 8, 8, 8), 1, 1, 1))
    want = [(e.fwd.clone(), e.dgrad.clone()) for e in packs]
    for e in packs:
        e.fwd.zero_(), e.dgrad.zero_()
    plan = c3.pack_weights_batch(packs)
    for e, (pf, pd) in zip(packs, want):
        assert torch.equal(e.fwd.view(torch.int16), pf.view(torch.int16)) and torch.equal(e.dgrad.view(torch.int16), pd.view(torch.int16))
    if launches is not None:
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            c3.pack_weights_batch(plan)
        assert _launches(graph) == launches
