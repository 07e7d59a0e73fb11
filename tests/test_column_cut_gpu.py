"""Convolutions that walk columns, at sizes where the cut leaves a workgroup one segment, several columns, or a last segment that is
shorter: integer-valued operands, so every result is the oracle's to the bit whatever the cut."""
import pytest
import torch

import scaffold_amd as sa
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

CASES = [
    # cin, cout, spatial, n
    (64, 128, (20, 20, 70), 1),   # weight gradient: 15 columns in two segments for 32 workgroups; forward on bricks
    (64, 128, (9, 60, 70), 1),    # 45 columns whole, two to a workgroup
    (32, 32, (11, 75, 97), 2),    # 40 columns a sample forward, 152 over the batch in the weight gradient
    (32, 64, (14, 100, 100), 1),  # 52 columns for 128 workgroups in two segments of four and three steps
    (32, 32, (5, 640, 40), 1),    # 160 columns of three steps forward, 320 in the weight gradient
]


@pytest.mark.parametrize("cin,cout,spatial,n", CASES)
def test_every_direction_is_the_oracles(device, cin, cout, spatial, n):
    prob = orc.ConvProblem(n=n, cin=cin, cout=cout, spatial=spatial, padding=(1, 1, 1), dtype=torch.bfloat16)
    ops = orc.make_inputs(prob, seed=cin + spatial[0], exact=True, density=0.02)
    x, w, gy = (ops[k].to(device) for k in ("input", "weight", "grad_output"))
    got = {"fwd": sa.conv3d_forward(x, w, None, 1, 1, 1), "bwd-data": sa.conv3d_backward_data(gy, w, x.shape, 1, 1, 1),
           "bwd-weight": sa.conv3d_backward_weight(x, w.shape, gy, 1, 1, 1)}
    for direction, y in got.items():
        want = orc.conv_reference(prob, ops, direction)
        assert torch.equal(y.cpu().double(), want.to(torch.bfloat16).double()), direction
