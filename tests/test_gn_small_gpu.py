"""GroupNorm of small groups (one launch each way): the edges of its range against the fp64 oracle."""
import pytest
import torch

import scaffold_amd as sa
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# (n, channels, groups, spatial, dtype): one piece; a part of a wavefront; 2 and 4 pieces per thread with a ragged last row;
# the largest of each row width; one voxel more (two launches); rows of 16 pieces and of 32 (two launches); two samples
CASES = [
    (1, 64, 8, (1, 1, 1), torch.bfloat16), (1, 16, 2, (1, 3, 5), torch.bfloat16), (1, 128, 8, (3, 19, 23), torch.bfloat16),
    (1, 64, 8, (8, 16, 16), torch.bfloat16), (1, 64, 8, (3, 683, 1), torch.bfloat16), (1, 512, 8, (8, 8, 8), torch.bfloat16),
    (1, 512, 8, (3, 171, 1), torch.bfloat16), (1, 1024, 8, (5, 7, 7), torch.float16),
    (1, 512, 2, (3, 5, 7), torch.float16), (2, 256, 8, (5, 7, 9), torch.bfloat16), (1, 128, 8, (5, 9, 11), torch.float32),
    (1, 32, 8, (16, 16, 8), torch.float32), (3, 512, 8, (4, 8, 8), torch.float32),
]


@pytest.mark.parametrize("n,c,groups,spatial,dtype", CASES)
@pytest.mark.parametrize("relu", [True, False])
def test_small_groups(n, c, groups, spatial, dtype, relu):
    g = torch.Generator().manual_seed(c + spatial[0])
    x = (torch.randn((n, c, *spatial), generator=g) * 3 + 40).to(dtype).contiguous(memory_format=torch.channels_last_3d)
    w, b = (1 + 0.1 * torch.randn(c, generator=g)).to(dtype), (0.1 * torch.randn(c, generator=g)).to(dtype)
    dy = torch.randn(x.shape, generator=g).to(dtype).contiguous(memory_format=torch.channels_last_3d)
    xd, wd, bd = (t.cuda().requires_grad_() for t in (x, w, b))
    y = sa.group_norm(xd, groups, wd, bd, 1e-5, "relu" if relu else None)
    y.backward(dy.cuda())
    for name, got, ref in zip(("y", "dx", "dw", "db"), (y, xd.grad, wd.grad, bd.grad),
                              orc.group_norm_reference(x, groups, w, b, 1e-5, relu, dy)):
        assert orc.gn_rel_error(got, ref) <= orc.GN_TOLERANCE[dtype], name


def test_small_groups_into_a_slab_and_with_nan():
    x = torch.randn((1, 128, 4, 8, 8), device="cuda").to(torch.bfloat16).contiguous(memory_format=torch.channels_last_3d)
    plain = sa.group_norm(x, 8, None, None, 1e-5, "relu")
    y = sa.group_norm(x, 8, None, None, 1e-5, "relu", out_halo=1)
    slab, halo = y._sfh_slab
    assert halo == 1 and torch.equal(y, plain) and not slab[:, :, 0].any() and not slab[:, :, -1].any()
    x[0, 3, 1, 2, 3] = float("nan")
    y = sa.group_norm(x, 8, None, None, 1e-5, "relu")
    assert y[:, :16].isnan().all() and not y[:, 16:].isnan().any()
