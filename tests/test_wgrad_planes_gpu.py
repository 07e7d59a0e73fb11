"""Small-volume weight gradients whose blocks are shared by three workgroups (nine taps each), alone and in a list: ragged tiles
on every axis, paddings, batches, both tile shapes, one and several slices, results in the operands' type and in fp32."""
import pytest
import torch

import scaffold_amd as sa
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# (n, cin, cout, spatial, padding, dtype)
CASES = [
    (1, 32, 32, (1, 1, 1), 1, torch.bfloat16), (1, 64, 32, (5, 7, 9), 1, torch.bfloat16), (2, 32, 64, (3, 9, 16), 1, torch.float16),
    (1, 64, 64, (4, 8, 8), 1, torch.bfloat16), (1, 32, 32, (12, 10, 8), (0, 1, 2), torch.bfloat16), (2, 96, 64, (9, 17, 11), (2, 0, 1), torch.bfloat16),
    (1, 256, 256, (8, 16, 16), 1, torch.float16),  # 64 blocks: one slice, stored in place
    (1, 288, 256, (3, 5, 8), 1, torch.bfloat16),   # 72 blocks
    (1, 320, 288, (3, 5, 8), 1, torch.bfloat16),   # 90 blocks: more than the chip has room for three times
]


def _problem(n, cin, cout, spatial, padding, dtype, seed):
    prob = orc.ConvProblem(n=n, cin=cin, cout=cout, spatial=spatial, dtype=dtype,
                           padding=(padding,) * 3 if isinstance(padding, int) else padding)
    return prob, orc.make_inputs(prob, seed=seed)


@pytest.mark.parametrize("case", CASES)
def test_alone(case):
    prob, ops = _problem(*case, seed=3)
    x, gy = ops["input"].cuda(), ops["grad_output"].cuda()
    want = orc.conv_reference(prob, ops, "bwd-weight")
    got = sa.conv3d_backward_weight(x, prob.weight_shape, gy, 1, case[4])
    orc.assert_close(got, want, prob, "bwd-weight")
    wide = sa.conv3d_backward_weight(x, prob.weight_shape, gy, 1, case[4], grad_dtype=torch.float32)
    assert torch.equal(wide.to(got.dtype), got)


@pytest.mark.parametrize("grad_dtype", [None, torch.float32])
@pytest.mark.parametrize("extra", [0, 1, 2])
def test_in_a_list(grad_dtype, extra):
    # extra: a problem of 64 blocks more, with which three workgroups still share a block: the bits do not change. Or one of 272, with
    # which a workgroup takes whole blocks and sums a tile in one chain: another order of the same fp32 sums
    cases = [(1, 32, 32, (12, 10, 8), (0, 1, 2), torch.bfloat16), (1, 64, 64, (4, 8, 8), 1, torch.bfloat16), (1, 64, 32, (5, 7, 9), 1, torch.bfloat16),
             (1, 64, 64, (16, 16, 16), 1, torch.bfloat16)]
    more = [(1, 256, 256, (4, 8, 8), 1, torch.bfloat16)] if extra == 1 else [(1, 512, 544, (2, 4, 8), 1, torch.bfloat16)] if extra else []
    problems = [_problem(*c, seed=5 + i) for i, c in enumerate(cases + more)]
    items = [(o["input"].cuda(), p.weight_shape, o["grad_output"].cuda(), c) for (p, o), c in
             zip(problems, [(0, 1, 2), (1, 1, 1), (1, 1, 1), (1, 1, 1), (1, 1, 1)])]
    got = sa.conv3d_backward_weight_batch(items, grad_dtype=grad_dtype)
    for (prob, ops), g in zip(problems, got):
        orc.assert_close(g.to(torch.bfloat16), orc.conv_reference(prob, ops, "bwd-weight"), prob, "bwd-weight")
    if extra:
        short = sa.conv3d_backward_weight_batch(items[:4], grad_dtype=grad_dtype)
        assert all(torch.equal(a, b) for a, b in zip(short, got)) == (extra == 1)
        assert grad_dtype is None or all(_close_in_fp32(a, b) for a, b in zip(short, got))


def _close_in_fp32(a, b):
    # two orders of the same sums of up to 4096 products, each within 4e-7 of 64 bits (relative, in the norm; one chain measured at
    # 3.2e-7 over 200000)
    return bool((a - b).norm() <= 8e-7 * b.norm())


@pytest.mark.parametrize("grad_dtype", [None, torch.float32])
@pytest.mark.parametrize("n,cin,cout,spatial,padding", [
    (1, 32, 64, (18, 8, 16), 1),       # nine tiles: two parts, the last one short
    (2, 64, 64, (13, 13, 13), 1),      # 28 tiles in five parts, over two samples
    (1, 128, 64, (28, 9, 9), (0, 1, 2)),
    (3, 32, 32, (12, 9, 7), 1),        # rows of eight
    (1, 64, 128, (28, 13, 13), 1),     # too many output channels: whole
])
def test_blocks_cut_into_parts(n, cin, cout, spatial, padding, grad_dtype):
    """The slices of a list's problems lie beside those of its large rows; alone or in a list of few blocks, the bits of a problem are the
    same."""
    cases = [(n, cin, cout, spatial, padding, torch.bfloat16), (1, 32, 32, (4, 5, 33), 1, torch.bfloat16), (1, 32, 64, (11, 16, 16), 1, torch.bfloat16)]
    problems = [_problem(*c, seed=9 + i) for i, c in enumerate(cases)]
    items = [(o["input"].cuda(), p.weight_shape, o["grad_output"].cuda(), p.padding) for p, o in problems]
    got = sa.conv3d_backward_weight_batch(items, grad_dtype=grad_dtype)
    for (prob, ops), g in zip(problems, got):
        orc.assert_close(g.to(torch.bfloat16), orc.conv_reference(prob, ops, "bwd-weight"), prob, "bwd-weight")
    alone = sa.conv3d_backward_weight_batch(items[:1], grad_dtype=grad_dtype)
    assert torch.equal(alone[0], got[0])
    # beside 272 blocks of another problem a workgroup takes whole blocks: the parts' slices of all 27 taps
    wide, ops = _problem(1, 512, 544, (2, 4, 8), 1, torch.bfloat16, seed=12)
    beside = sa.conv3d_backward_weight_batch(items + [(ops["input"].cuda(), wide.weight_shape, ops["grad_output"].cuda(), wide.padding)],
                                             grad_dtype=grad_dtype)
    for (prob, o), g, b in zip(problems, got, beside):
        orc.assert_close(b.to(torch.bfloat16), orc.conv_reference(prob, o, "bwd-weight"), prob, "bwd-weight")
        assert grad_dtype is None or _close_in_fp32(b, g)
    orc.assert_close(beside[-1].to(torch.bfloat16), orc.conv_reference(wide, ops, "bwd-weight"), wide, "bwd-weight")


@pytest.mark.parametrize("case", [
    (1, 32, 32, (16, 16, 32), 1, torch.bfloat16),            # full rows of a small volume
    (1, 64, 32, (5, 7, 17), 1, torch.float16),               # rows a voxel past the small-volume kernel's
    (2, 32, 64, (9, 13, 37), (0, 1, 2), torch.bfloat16),     # cut rows over two samples
    (1, 96, 64, (3, 33, 20), 1, torch.bfloat16),
    (1, 288, 320, (2, 4, 18), 1, torch.bfloat16),            # 90 blocks: no room for three workgroups each
])
def test_wide_rows_in_tiles(case):
    """Problems with rows of more than 16 voxels that a launch of their own takes in tiles; a list still walks their columns."""
    test_alone(case)
    prob, ops = _problem(*case, seed=3)
    padding = (case[4],) * 3 if isinstance(case[4], int) else case[4]
    x, gy = ops["input"].cuda(), ops["grad_output"].cuda()
    alone = sa.conv3d_backward_weight(x, prob.weight_shape, gy, 1, padding, grad_dtype=torch.float32)
    (listed,) = sa.conv3d_backward_weight_batch([(x, prob.weight_shape, gy, padding)], grad_dtype=torch.float32)
    # two orders of the same fp32 sums: each within 2e-7 of 64 bits (relative, in the norm)
    assert (alone - listed).norm() <= 4e-7 * listed.norm()
