"""Which kernel a convolution's volume goes to, where two rules meet: the launch query is a pure function of the problem."""

import random

import pytest
import torch

from scaffold_amd import conv3d as c3


def _kernel(n, cin, cout, spatial, direction="fwd", padding=1):
    return c3.launch_geometry((n, cin, *spatial), (cout, cin, 3, 3, 3), 1, padding, 1, torch.bfloat16, direction)["kernel"]


@pytest.mark.parametrize("n,cin,spatial", [
    (32, 128, (32, 32, 32)),
    (16, 128, (64, 32, 32)),
    (8, 128, (128, 32, 32)),
    (10, 128, (64, 28, 28)),
    (16, 256, (48, 28, 20)),
])
def test_wide_kernel_steps_aside_for_bricks_only(n, cin, spatial):
    """Many small planes of a 64-channel output: the wide kernel's or, where its rule reckons the bricks cheaper, the brick kernel's.
    The small-volume kernel takes the same planes by its own rule and stages 3.75 voxels per output voxel."""
    assert _kernel(n, cin, 64, spatial) in ("wide", "brick")
    assert _kernel(n, 64, cin, spatial, "bwd-data") in ("wide", "brick")


@pytest.mark.parametrize("cin,cout,spatial,kernel", [
    (64, 64, (256, 16, 16), "brick"),    # 1024 pairs of blocks on whole bricks
    (128, 128, (128, 16, 16), "brick"),
    (256, 64, (256, 16, 16), "brick"),
    (64, 64, (192, 16, 16), "split"),    # 768: three rounds
    (128, 64, (200, 20, 20), "split"),   # 1500, but rows of 20 leave a third of the bricks empty
    (128, 128, (40, 32, 32), "split"),   # a plane that fills its share: whatever the depth
])
def test_deep_thin_volumes(cin, cout, spatial, kernel):
    """Deep volumes of small planes: past three rounds of the small-volume kernel's workgroups the brick kernel serves what it wastes
    little on -- and the same one whether the data gradient writes a shard's slab or the padded volume."""
    assert _kernel(1, cin, cout, spatial) == kernel
    padded = _kernel(1, cout, cin, spatial, "bwd-data")
    d, h, w = spatial
    assert padded == kernel and _kernel(1, cout, cin, (d + 2, h, w), "bwd-data", (0, 1, 1)) == padded


@pytest.mark.parametrize("cin,cout", [(64, 128), (64, 160), (64, 192), (64, 256), (64, 512), (64, 64), (128, 64), (128, 128), (256, 128), (512, 256)])
def test_slab_and_padded_volume_add_in_one_order(cin, cout):
    """Both forms of a depth shard's convolution, and of its data gradient, are one kernel's: bits must not depend on the form, and each
    kernel adds in an order of its own."""
    rng = random.Random(cin + cout)
    shapes = [(27, 61, 33), (47, 37, 36), (39, 45, 35), (9, 27, 50), (17, 36, 35), (33, 57, 50)]
    shapes += [tuple(round(4 * 16 ** rng.random()) for _ in range(3)) for _ in range(400)]
    for d, h, w in shapes:
        for direction in ("fwd", "bwd-data"):
            padded = _kernel(1, cin, cout, (d, h, w), direction)
            slab = _kernel(1, cin, cout, (d + 2, h, w), direction, (0, 1, 1))
            assert padded == slab, (direction, (d, h, w), padded, slab)


@pytest.mark.parametrize("cin,cout,spatial,forward,gradient", [
    (256, 256, (32, 32, 32), "split", "split"),
    (128, 128, (60, 30, 31), "split", "split"),
    (64, 64, (64, 32, 32), "split", "split"),
    (256, 256, (29, 28, 14), "split", "split"),
    (512, 512, (5, 8, 8), "brick", "brick"),     # eight slices of two chunks each
    (256, 256, (5, 8, 14), "split", "split"),    # eight of one: as many partial sums there
    (128, 128, (9, 12, 8), "split", "split"),    # four of one
    (256, 256, (11, 4, 9), "split", "split"),    # four of two
    (192, 256, (6, 15, 7), "split", "brick"),    # four of one and of two: the small-volume kernel cannot
    (64, 128, (14, 13, 6), "split", "brick"),
    (128, 64, (14, 13, 6), "brick", "split"),    # the gradient's two slices are one chunk each
    (512, 512, (9, 9, 6), "split", "split"),     # two of eight
    (128, 64, (20, 34, 42), "brick", "brick"),   # a plane past 32 x 32 that would gain a quarter
    (256, 512, (6, 7, 5), "brick", "brick"),     # eight of one, but 512 channels produced
    (64, 64, (9, 27, 50), "split", "brick"),     # a plane past 32 x 32
])
def test_launch_times_take_no_partial_sums_away(cin, cout, spatial, forward, gradient):
    """Four partial sums to a voxel are nearer the exact one than the bricks' single chain, eight slices nearer still: where the
    small-volume kernel served a volume, or the bricks in eight slices, no estimate of times moves it; nor a data gradient to another order."""
    assert _kernel(1, cin, cout, spatial) == forward
    assert _kernel(1, cin, cout, spatial, "bwd-data") == gradient


@pytest.mark.parametrize("cin,cout,spatial,records", [
    (32, 32, (54, 105, 99), 140),      # columns for every workgroup once; by their times 224
    (256, 256, (24, 20, 28), 240),     # bricks of 2 x 4 x 8; 210 of 4 x 4 x 4
    (512, 512, (12, 10, 14), 36),      # 30 of 2 x 2 x 16
    (64, 64, (55, 28, 41), 196),       # 336 of another brick
])
def test_groupnorm_records_do_not_go_by_times(cin, cout, spatial, records):
    """Records are sums of a launch's bricks: what a network computes behind them has the bits it had before launch times chose bricks."""
    assert c3._Problem((1, cin, *spatial), (cout, cin, 3, 3, 3), 1, 1, 1, torch.bfloat16).gn_records(8) == records


@pytest.mark.parametrize("n,cin,cout,spatial,slices", [
    (1, 128, 128, (43, 29, 34), 5),     # tiles; columns would be 16 slices
    (1, 64, 32, (54, 40, 76), 42),      # tiles; 120
    (1, 32, 32, (104, 52, 79), 83),     # tiles; 234
    (1, 32, 32, (96, 80, 112), 240),    # columns by both estimates
])
def test_weight_gradients_of_wide_rows_keep_the_tiles_shorter_sums(n, cin, cout, spatial, slices):
    """Columns sum longer chains than tiles: they are walked where both estimates find them quicker, not where one does."""
    assert c3.split_count((n, cin, *spatial), (cout, cin, 3, 3, 3), 1, 1, 1, torch.bfloat16) == slices


def test_fp32_weight_gradient_of_long_rows():
    """A row of 2 GiB and more: its offsets are 64-bit, the tiled kernel takes it (the untiled one makes no slices)."""
    assert c3.split_count((1, 32, 1, 1, 16_800_000), (32, 32, 3, 3, 3), 1, 1, 1, torch.float32) > 1
