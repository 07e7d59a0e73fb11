"""Which weight gradients wait for the end of the backward pass: a pure function of the problem (no GPU needed)."""

import pytest
import torch

from scaffold_amd import modules as M


@pytest.mark.parametrize("spatial,cin,cout,family", [
    ((64, 128, 128), 64, 32, 1),      # 116 GFLOP: a place in the batch of large rows
    ((128, 128, 128), 64, 32, 1),     # 232 GFLOP: the last below the line
    ((128, 128, 128), 64, 64, 0),     # 464 GFLOP: computed in its own node
    ((8, 16, 16), 512, 256, 2),       # small volume
])
def test_large_problems_do_not_wait(spatial, cin, cout, family):
    weight = torch.nn.Parameter(torch.empty((cout, cin, 3, 3, 3), dtype=torch.bfloat16))
    for in_shape, padding in (((1, cin, *spatial), (1, 1, 1)), ((1, cin, spatial[0] + 2, *spatial[1:]), (0, 1, 1))):
        args = (torch.Size(in_shape), weight.shape, (1, 1, 1), padding, (1, 1, 1), torch.bfloat16)
        assert M._deferrable(weight, *args) == family
        assert M._deferrable(weight.detach(), *args) == 0    # not a parameter that takes a .grad
