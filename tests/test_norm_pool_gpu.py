"""The normalisation that pools its result in the same pass, against the two launches: the same bits, values and gradients."""

import ctypes

import pytest
import torch

import scaffold_amd as sa
from scaffold_amd import _lib
from scaffold_amd.modules import FastConv3d, FastGroupNorm, conv_then_norm
from scaffold_amd.pooling import FastMaxPool3d
from scaffold_amd.unet import UNet

pytestmark = pytest.mark.gpu
CL = torch.channels_last_3d


def _pair(c, device, dtype, relu=True):
    torch.manual_seed(1)
    conv = FastConv3d(c, c, 3, padding=1, bias=False).to(device, dtype).to(memory_format=CL)
    norm = FastGroupNorm(8, c, activation="relu" if relu else None).to(device, dtype)
    with torch.no_grad():
        norm.weight.add_(0.3 * torch.randn(c, device=device))
        norm.bias.add_(0.3 * torch.randn(c, device=device))
    conv.gn_groups = 8
    return conv, norm


@pytest.mark.parametrize("relu", [True, False])
@pytest.mark.parametrize("halo", [0, 1])
@pytest.mark.parametrize("n,c,spatial,dtype", [
    (1, 32, (8, 16, 33), torch.bfloat16),      # four threads to a cell; a column of cells that are not pooled
    (2, 64, (5, 7, 9), torch.bfloat16),        # odd on every axis, two samples
    (1, 64, (16, 32, 64), torch.float16),      # several passes a workgroup
    (1, 128, (2, 2, 2), torch.bfloat16),       # one cell
    (1, 256, (4, 9, 20), torch.bfloat16),
    (1, 512, (3, 8, 8), torch.bfloat16),       # 64 threads to a cell
])
def test_same_bits_as_two_launches(device, n, c, spatial, dtype, halo, relu):
    conv, norm = _pair(c, device, dtype, relu)
    norm.out_halo = halo
    pool = FastMaxPool3d(2)
    pool.out_halo = halo
    x0 = torch.randn(n, c, *spatial, device=device).to(dtype).contiguous(memory_format=CL)
    gp = torch.randn(n, c, *(s // 2 for s in spatial), device=device).to(dtype).contiguous(memory_format=CL)
    gs = torch.randn(n, c, *spatial, device=device).to(dtype).contiguous(memory_format=CL)
    results = []
    for fused in (False, True):
        norm.pool_next = halo if fused else None
        x = x0.clone().requires_grad_(True)
        torch.full((4 * x0.numel(),), float("nan"), device=device, dtype=dtype)
        y = conv_then_norm(conv, norm, x)
        # (a halo asks for one sample, and records come only from the kernels that offer them)
        assert hasattr(y, "_sfh_pooled") == (fused and not (halo and n > 1) and bool(y is not None and _records(conv, x0)))
        pooled, skip = pool.with_skip(y)
        assert not hasattr(y, "_sfh_pooled")
        slabs = [t._sfh_slab[0].clone() for t in (pooled, skip) if halo and n == 1]
        grads = torch.autograd.grad((pooled, skip), (x, conv.weight, norm.weight, norm.bias), (gp, gs))
        with torch.no_grad():
            again = pool(conv_then_norm(conv, norm, x0))
        assert torch.equal(again, pooled)
        results.append([pooled.detach(), skip.detach(), *slabs, *grads])
    assert all(torch.equal(a, b) for a, b in zip(*results))


def _records(conv, x):
    return getattr(conv(x), "_sfh_gn_partials", None) is not None


def test_what_is_not_reused(device):
    conv, norm = _pair(64, device, torch.bfloat16)
    pool, wide = FastMaxPool3d(2), FastMaxPool3d(2)
    wide.out_halo = 1
    x = torch.randn(1, 64, 8, 16, 16, device=device).to(torch.bfloat16).contiguous(memory_format=CL)
    norm.pool_next = 0
    with torch.no_grad():
        want = torch.nn.functional.max_pool3d(conv_then_norm(conv, norm, x).float(), 2)
        y = conv_then_norm(conv, norm, x)
        assert torch.equal(wide(y).float(), want) and hasattr(wide(y), "_sfh_slab")  # another halo
        y = conv_then_norm(conv, norm, x)
        a, b = pool(y), pool(y)                                                      # a second pooling has its own tensor
        assert a.data_ptr() != b.data_ptr() and torch.equal(a.float(), want) and torch.equal(b.float(), want)
        y = conv_then_norm(conv, norm, x).add_(1.0)                                  # written since
        assert torch.equal(pool(y), torch.nn.functional.max_pool3d(y.float(), 2).to(y.dtype))
    y = conv_then_norm(conv, norm, x.requires_grad_(True)).detach().requires_grad_(True)
    (g,) = torch.autograd.grad(pool(y).float().sum(), y)
    assert int((g != 0).sum()) == want.numel()
    with torch.no_grad():
        y = conv_then_norm(conv, norm, x)
    y.requires_grad_(True)  # pooled without indices, and a gradient wanted after all
    (h,) = torch.autograd.grad(pool(y).float().sum(), y)
    assert torch.equal(g, h)
    with torch.inference_mode():
        y = conv_then_norm(conv, norm, x.detach())
        assert not hasattr(y, "_sfh_pooled") and torch.equal(pool(y).float(), want)


def test_nan_and_infinity(device):
    conv, norm = _pair(32, device, torch.bfloat16)
    x = torch.randn(1, 32, 4, 8, 34, device=device).to(torch.bfloat16)
    x[0, 3, 1, 2, 3] = float("nan")
    x[0, 3, 1, 5, 20] = float("inf")
    x = x.contiguous(memory_format=CL)
    outs = []
    for pool_next in (None, 0):
        norm.pool_next = pool_next
        with torch.no_grad():
            y = conv_then_norm(conv, norm, x)
            outs.append((y.clone(), FastMaxPool3d(2)(y)))
    for a, b in zip(*outs):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())


@pytest.mark.parametrize("shard,size", [(False, (14, 25, 31)), (True, (16, 32, 64))])
def test_a_step_keeps_its_bits(device, shard, size):
    torch.manual_seed(5)
    net = UNet(3, 5, layers=2, base_width=32).to(device).to(memory_format=CL).set_shard_halo(shard)
    x = torch.randn(1, 3, *size, device=device).contiguous(memory_format=CL)
    target = torch.randint(0, 5, (1, *size), device=device)

    def step():
        net.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            logits = net(x)
            with torch.no_grad():
                quiet = net(x)
        loss = sa.ce_dice_loss(logits, target)
        loss.backward()
        assert torch.equal(logits, quiet)
        return [loss.detach(), logits.detach()] + [p.grad.clone() for p in net.parameters()]

    norms = [m for m in net.modules() if isinstance(m, FastGroupNorm) and m.pool_next is not None]
    assert len(norms) == 2 and all(m.pool_next == int(shard) for m in norms)
    got = step()
    for m in norms:
        m.pool_next = None
    assert all(torch.equal(a, b) for a, b in zip(step(), got))
    net.use_checkpointing()
    assert all(m.pool_next is None for m in net.modules() if isinstance(m, FastGroupNorm))


def _captured(fn):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side), torch.no_grad():
        fn()  # what a first call packs is not part of a capture
    torch.cuda.current_stream().wait_stream(side)
    with torch.cuda.graph(graph), torch.no_grad():
        out = fn()
    return graph, out


def _pooled(y):
    return torch.nn.functional.max_pool3d(y.float(), 2).to(y.dtype)


@pytest.mark.parametrize("halo", [0, 1])
@pytest.mark.parametrize("n,c,spatial", [(1, 32, (8, 16, 33)), (1, 64, (5, 7, 9)), (1, 128, (2, 2, 2)), (1, 512, (3, 8, 8))])
def test_handed_over_is_the_launched_one(device, n, c, spatial, halo):
    """What the normalisation pooled, taken by the pooling: values, slab and (through the gradients) indices of its own launch."""
    conv, norm = _pair(c, device, torch.bfloat16)
    norm.out_halo = norm.pool_next = halo
    pool = FastMaxPool3d(2)
    pool.out_halo = halo
    x0 = torch.randn(n, c, *spatial, device=device).to(torch.bfloat16).contiguous(memory_format=CL)
    gp, gs = (torch.randn(n, c, *s, device=device).to(torch.bfloat16).contiguous(memory_format=CL) for s in ([v // 2 for v in spatial], spatial))
    results = []
    for take in (True, False):
        x = x0.clone().requires_grad_(True)
        y = conv_then_norm(conv, norm, x)
        given = y.__dict__.pop("_sfh_pooled")
        pooled, skip = pool.with_skip(y, given if take else None)
        assert (pooled.data_ptr() == given[0].data_ptr()) == take
        slabs = [t._sfh_slab[0].clone() for t in (pooled, skip) if halo]
        results.append([pooled.detach(), skip.detach(), *slabs, *torch.autograd.grad((pooled, skip), (x, conv.weight, norm.weight, norm.bias), (gp, gs))])
    assert all(torch.equal(a, b) for a, b in zip(*results))


def test_handed_over_nan_infinity_and_another_halo(device):
    conv, norm = _pair(32, device, torch.bfloat16)
    norm.pool_next = 0
    pool, wide = FastMaxPool3d(2), FastMaxPool3d(2)
    wide.out_halo = 1
    x = torch.randn(1, 32, 4, 8, 34, device=device).to(torch.bfloat16)
    x[0, 3, 1, 2, 3] = float("nan")
    x[0, 3, 1, 5, 20] = float("inf")
    x = x.contiguous(memory_format=CL)
    with torch.no_grad():
        y = conv_then_norm(conv, norm, x)
        given = y.__dict__.pop("_sfh_pooled")
        want, taken, other = pool(y), pool.with_skip(y, given)[0], wide.with_skip(y, given)[0]
    assert taken.data_ptr() == given[0].data_ptr() and other.data_ptr() != given[0].data_ptr() and hasattr(other, "_sfh_slab")
    for got in (taken, other):
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())


@pytest.mark.parametrize("relu", [True, False])
@pytest.mark.parametrize("n,c,spatial,dtype", [
    (1, 32, (9, 35, 70), torch.float16),       # odd planes, several workgroups, two rows a thread at once
    (2, 64, (5, 7, 9), torch.bfloat16),        # two samples, less than one pass a workgroup
    (1, 64, (34, 64, 66), torch.bfloat16),     # several passes
    (1, 256, (2, 40, 3), torch.bfloat16),      # one cell deep and wide
    (1, 512, (3, 8, 8), torch.bfloat16),       # a group that one workgroup holds: summed before it
])
def test_gradients_meet_in_the_normalisation(device, n, c, spatial, dtype, relu):
    """The skip connection's gradient, the pooled tensor's, and both, through the launch that made the two and through a pooling of
    its own: the same bits."""
    conv, norm = _pair(c, device, dtype, relu)
    norm.pool_next = 0
    pool = FastMaxPool3d(2)
    x0 = torch.randn(n, c, *spatial, device=device).to(dtype).contiguous(memory_format=CL)
    gp, gs = (torch.randn(n, c, *s, device=device).to(dtype).contiguous(memory_format=CL) for s in ([v // 2 for v in spatial], spatial))
    for used in ("both", "skip", "pooled"):
        results = []
        for take in (True, False):
            x = x0.clone().requires_grad_(True)
            y = conv_then_norm(conv, norm, x)
            given = y.__dict__.pop("_sfh_pooled")
            outs, grads = zip(*[p for k, p in zip(("pooled", "skip"), zip(pool.with_skip(y, given if take else None), (gp, gs))) if used in ("both", k)])
            results.append(torch.autograd.grad(outs, (x, conv.weight, norm.weight, norm.bias), grads))
        assert all(torch.equal(a, b) for a, b in zip(*results)), used


@pytest.mark.parametrize("relu", [0, 1])
@pytest.mark.parametrize("n,c,spatial,dtype", [
    (2, 32, (1700, 5, 6), torch.bfloat16),    # a thread's next row is 64 voxels on: two planes, a row with a carry, and four voxels
    (2, 64, (1300, 3, 7), torch.float16),     # 32 on: a plane, a row and four voxels, a carry into either
    (2, 64, (33, 5, 6), torch.bfloat16),      # one pass
    (1, 32, (3400, 2, 17), torch.bfloat16),   # seven: the last one is not half of a pair
    (1, 64, (129, 128, 67), torch.bfloat16),  # 141.6 MB: operands read past the caches
    (2, 32, (65, 129, 130), torch.float16),   # 139.5 MB, two samples of odd planes
])
def test_pooled_gradient_in_both_passes(device, n, c, spatial, dtype, relu):
    """The two passes that take the pooling's gradient in, against the launch that sums and the two passes behind it: the same bits."""
    lib, code, groups = _lib.lib(), _lib.dtype_code(dtype), 8
    def volume(*extents):
        return torch.randn((n, *extents, c), device=device).to(dtype)
    torch.manual_seed(3)
    half = [v // 2 for v in spatial]
    x, gy, gp = volume(*spatial), volume(*spatial), volume(*half)
    gamma, beta, mean = (torch.randn(k, device=device) for k in (c, c, n * groups))
    rstd = torch.rand(n * groups, device=device) + 0.5
    pooled, idx = volume(*half), torch.empty((n, *half, c), dtype=torch.uint8, device=device)
    total = torch.empty_like(x)
    pd = _lib.PoolDesc(n, c, *spatial)
    gd = _lib.GroupNormDesc(n, c, groups, relu, spatial[0] * spatial[1] * spatial[2], 1e-5)
    stream = torch.cuda.current_stream().cuda_stream
    size = lib.sfh_groupnorm_bwd_workspace_bytes(ctypes.byref(gd), code)
    def run(call):
        out = torch.full_like(x, float("nan")), torch.empty(c, device=device), torch.empty(c, device=device)
        ws = torch.empty(size, dtype=torch.uint8, device=device)
        _lib.check(call(*(t.data_ptr() for t in out), ws.data_ptr(), size, stream), "groupnorm backward")
        return out
    _lib.check(lib.sfh_maxpool2_fwd(ctypes.byref(pd), code, volume(*spatial).data_ptr(), pooled.data_ptr(), idx.data_ptr(), stream), "pool")
    _lib.check(lib.sfh_maxpool2_bwd_add(ctypes.byref(pd), code, gp.data_ptr(), idx.data_ptr(), gy.data_ptr(), total.data_ptr(), stream), "pool")
    rest = [t.data_ptr() for t in (x, gamma, beta, mean, rstd)]
    extents, fp32 = (ctypes.c_int32 * 3)(*spatial), _lib.dtype_code(torch.float32)
    got = run(lambda *out: lib.sfh_groupnorm_bwd_pool(ctypes.byref(gd), extents, code, fp32, gy.data_ptr(), gp.data_ptr(), idx.data_ptr(), *rest, *out))
    want = run(lambda *out: lib.sfh_groupnorm_bwd(ctypes.byref(gd), code, code, fp32, total.data_ptr(), *rest, *out))
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_a_captured_pooling_reads_its_input(device):
    conv, norm = _pair(64, device, torch.bfloat16)
    norm.pool_next = 0
    pool = FastMaxPool3d(2)
    x = torch.randn(1, 64, 8, 16, 16, device=device).to(torch.bfloat16).contiguous(memory_format=CL)
    with torch.no_grad():
        y = conv_then_norm(conv, norm, x)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph), torch.no_grad():
        p = pool(y)
    for seed in range(3):
        torch.manual_seed(seed)
        with torch.no_grad():
            y.copy_(torch.randn_like(y))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(p, _pooled(y))


def test_what_was_pooled_from_a_static_output_is_kept(device):
    conv, norm = _pair(64, device, torch.bfloat16)
    norm.pool_next = 0
    x = torch.randn(1, 64, 8, 16, 16, device=device).to(torch.bfloat16).contiguous(memory_format=CL)
    graph, y = _captured(lambda: conv_then_norm(conv, norm, x))
    graph.replay()
    with torch.no_grad():
        p = FastMaxPool3d(2)(y)
    want = _pooled(y)
    for _ in range(2):
        x.copy_(torch.randn_like(x))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(p, want) and not torch.equal(_pooled(y), want)


def test_on_a_stream_of_its_own_and_after_a_write_nobody_counts(device):
    conv, norm = _pair(64, device, torch.bfloat16)
    norm.pool_next = 0
    pool = FastMaxPool3d(2)
    x = torch.randn(1, 64, 8, 16, 16, device=device).to(torch.bfloat16).contiguous(memory_format=CL)
    side = torch.cuda.Stream()
    with torch.no_grad():
        y = conv_then_norm(conv, norm, x)
        left = y._sfh_pooled[0]
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            y.record_stream(side)
            p = pool(y)
        torch.cuda.current_stream().wait_stream(side)
        assert p.data_ptr() != left.data_ptr() and torch.equal(p, left)  # memory of the stream it was asked for on
        y = conv_then_norm(conv, norm, x)
        y.data.neg_()
        assert torch.equal(pool(y), _pooled(y))


def test_a_network_takes_it_and_its_hooks_are_seen(device, monkeypatch):
    torch.manual_seed(5)
    net = UNet(3, 5, layers=2, base_width=32).to(device).to(memory_format=CL)
    x = torch.randn(1, 3, 16, 32, 32, device=device).contiguous(memory_format=CL)
    taken = []
    with_skip = FastMaxPool3d.with_skip
    monkeypatch.setattr(FastMaxPool3d, "with_skip", lambda self, y, given=None: taken.append(given is not None) or with_skip(self, y, given))

    def forward():
        taken.clear()
        with torch.autocast("cuda", dtype=torch.bfloat16), torch.no_grad():
            return net(x), list(taken)

    assert forward()[1] == [True, True]
    enc = net.down_list[0]

    def negate(module, args, out):
        out.data.neg_()

    handle = enc.register_forward_hook(negate)
    hooked, taken_then = forward()
    assert taken_then == [False, True]
    for m in net.modules():
        if isinstance(m, FastGroupNorm):
            m.pool_next = None
    assert torch.equal(hooked, forward()[0])
    handle.remove()
    assert not torch.equal(hooked, forward()[0])
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not hasattr(enc(x), "_sfh_pooled")  # a block by itself pools for nobody
