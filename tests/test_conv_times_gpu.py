"""Where the kernels' launch times decide which of them serves a problem: both sides of the lines, exact against the oracle, alone
and from a pair of tensors, with the GroupNorm records of the kernel that serves."""
import pytest
import torch

import scaffold_amd as sa
from oracle import oracle as orc
from scaffold_amd import conv3d as c3

pytestmark = pytest.mark.gpu
CL = torch.channels_last_3d

CASES = [
    # n, cin, cout, spatial, kernel, voxels
    (1, 64, 64, (9, 27, 50), "split", 64),      # a plane past 32 x 32, 245 pairs
    (1, 64, 64, (8, 27, 50), "brick", 256),     # 196: the reduction sliced
    (1, 128, 128, (10, 28, 56), "split", 64),
    (1, 64, 128, (14, 13, 6), "split", 64),     # 56 pairs under 128 channels
    (1, 128, 128, (4, 6, 20), "split", 64),     # 24: the fewest
    (1, 128, 128, (4, 6, 12), "brick", 256),    # 16
    (1, 256, 256, (3, 8, 14), "brick", 256),    # 32
    (1, 256, 256, (5, 8, 14), "split", 64),     # 48
    (1, 512, 512, (9, 9, 6), "split", 64),      # 120 pairs of a long reduction on cut bricks
    (2, 128, 64, (19, 30, 35), "brick", None),  # a round and a bit of the wide kernel's workgroups would be two
    (1, 256, 256, (32, 32, 8), "split", 64),
    (2, 128, 128, (10, 5, 30), "split", 64),    # bricks of 2 x 2 x 16, a workgroup of one channel block each
    (2, 128, 512, (6, 9, 29), "split", 64),     # ... two
    (2, 192, 128, (10, 5, 30), "split", 64),    # ... two chunks a round
    (2, 192, 256, (10, 5, 30), "split", 64),    # ... two blocks
    (1, 128, 256, (7, 11, 12), "split", 64),    # bricks of 4 x 4 x 4, cut on two axes, one block
    (1, 192, 512, (7, 11, 12), "split", 64),    # ... two blocks, two chunks a round
    (1, 64, 64, (55, 28, 41), "brick", 256),    # 4 x 8 x 8 with one block in the place of 4 x 4 x 32
]


@pytest.mark.parametrize("n,cin,cout,spatial,kernel,voxels", CASES)
def test_both_sides_of_the_lines(device, n, cin, cout, spatial, kernel, voxels):
    dtype = torch.bfloat16
    prob = orc.ConvProblem(n=n, cin=cin, cout=cout, spatial=spatial, padding=(1, 1, 1), dtype=dtype)
    geom = c3.launch_geometry(prob.input_shape, prob.weight_shape, 1, 1, 1, dtype, "fwd")
    assert geom["kernel"] == kernel and voxels in (None, geom["voxels"]), geom
    ops = orc.make_inputs(prob, seed=cin + spatial[2], exact=True, density=0.02)
    x, w, gy = (ops[k].to(device) for k in ("input", "weight", "grad_output"))
    y = sa.conv3d_forward(x, w, None, 1, 1, 1, gn_groups=8)
    assert torch.equal(y.cpu().double(), orc.conv_reference(prob, ops, "fwd").to(dtype).double())
    gx = sa.conv3d_backward_data(gy, w, x.shape, 1, 1, 1)
    assert torch.equal(gx.cpu().double(), orc.conv_reference(prob, ops, "bwd-data").to(dtype).double())
    half = cin // 2
    first, second = (t.contiguous(memory_format=CL) for t in (x[:, :half], x[:, half:]))
    if c3.is_supported_pair(first, second, w, None, 1, 1, 1):
        assert torch.equal(c3.conv3d_forward_pair(first, second, w, None, 1, 1, 1), sa.conv3d_forward(x, w, None, 1, 1, 1))
    if hasattr(y, "_sfh_gn_partials"):
        normed = sa.group_norm(y, 8, None, None, 1e-5, None, out_dtype=None)
        ref = torch.nn.functional.group_norm(y.double(), 8, None, None, 1e-5)
        # half a unit in the last place of a bf16 value is at most 2^-8 of it; the statistics are fp32
        assert orc.gn_rel_error(normed, ref) < 2.0 ** -8 + 1e-5
