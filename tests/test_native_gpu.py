"""The C++ host path (``scaffold_amd/_native``): its autograd nodes where they differ from an ordinary forward and backward."""

import pytest
import torch

import scaffold_amd as sa

pytestmark = pytest.mark.gpu
CL = torch.channels_last_3d


def _x(device, c=32, n=1, dtype=torch.bfloat16):
    return torch.randn(n, c, 4, 4, 8, device=device).to(dtype).contiguous(memory_format=CL).requires_grad_()


def _ops(device):
    conv = sa.FastConv3d(32, 32, 3, padding=1, device=device, dtype=torch.bfloat16)
    up = sa.FastConvTranspose3d(32, 32, 2, stride=2, device=device, dtype=torch.bfloat16)
    norm = sa.FastGroupNorm(8, 32, activation="relu", device=device, dtype=torch.bfloat16)
    labels = torch.zeros(1, 4, 4, 8, dtype=torch.long, device=device)
    return {"conv": conv, "up": up, "norm": norm, "pool": sa.FastMaxPool3d(2), "skip": lambda x: sa.FastMaxPool3d(2).with_skip(x)[0],
            "loss": lambda x: sa.ce_dice_loss(x, labels)}


@pytest.mark.parametrize("name", ["conv", "up", "norm", "pool", "skip", "loss"])
def test_no_op_is_differentiated_twice_in_silence(device, name):
    """The gradient under create_graph is the ordinary one, and differentiating it raises instead of returning zeros."""
    op, x = _ops(device)[name], _x(device)
    (plain,) = torch.autograd.grad(op(x).float().square().sum(), x)
    (gx,) = torch.autograd.grad(op(x).float().square().sum(), x, create_graph=True)
    assert torch.equal(plain, gx) and gx.requires_grad
    with pytest.raises(RuntimeError, match="once_differentiable"):
        gx.float().sum().backward()


def test_gradients_only_where_they_are_wanted(device):
    conv, norm = _ops(device)["conv"], _ops(device)["norm"]
    x = _x(device)
    for op in (conv, norm):
        (gw,) = torch.autograd.grad(op(x.detach()).float().square().sum(), op.weight)
        gx, gw2, gb = torch.autograd.grad(op(x).float().square().sum(), (x, op.weight, op.bias))
        assert torch.equal(gw, gw2) and gx.shape == x.shape and gb.shape == op.bias.shape
        with torch.no_grad():
            assert not op(x).requires_grad


def test_empty_batch_through_the_up_convolution(device):
    up = _ops(device)["up"]
    x = torch.empty(0, 32, 4, 4, 8, device=device, dtype=torch.bfloat16).requires_grad_()
    y = up(x)
    assert y.shape == (0, 32, 8, 8, 16)
    gx, gw, gb = torch.autograd.grad(y.float().sum(), (x, up.weight, up.bias))
    assert gx.shape == x.shape and not gw.any() and not gb.any()


def test_a_tensor_changed_after_the_forward_is_noticed(device):
    conv, x = _ops(device)["conv"], _x(device)
    h = x * 1
    y = conv(h)
    with torch.no_grad():
        h.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.float().sum().backward()


def test_passes_that_overlap_keep_their_weight_gradients_apart(device):
    """Two threads run backward passes with deferred weight gradients at the same time, each on a stream of its own: every
    gradient is the one its pass alone would give."""
    import threading

    def make(seed):
        torch.manual_seed(seed)
        net = sa.UNet(1, 3, layers=2, base_width=32).to(device).to(torch.bfloat16).to(memory_format=CL).defer_weight_gradients()
        x = torch.randn(1, 1, 8, 16, 32, device=device).to(torch.bfloat16).contiguous(memory_format=CL)
        return net, x, torch.randint(0, 3, (1, 8, 16, 32), device=device)

    def grads(net, x, labels):
        net.zero_grad(set_to_none=True)
        sa.ce_dice_loss(net(x), labels).backward()
        return [p.grad.clone() for p in net.parameters()]

    jobs = [make(1), make(2)]
    want = [grads(*job) for job in jobs]
    got = [None, None]

    def run(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(3):
                got[i] = grads(*jobs[i])
            torch.cuda.current_stream().synchronize()

    torch.cuda.synchronize()
    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for w, g in zip(want, got):
        assert all(torch.equal(a, b) for a, b in zip(w, g))


def test_convolution_and_norm_in_one_call_are_the_two_modules(device):
    """``conv_then_norm`` gives the bits of ``norm(conv(x))`` in the forward and in every gradient, plain and into a slab, and
    leaves hooked or biased modules alone."""
    from scaffold_amd.modules import conv_then_norm

    def pair(bias=False):
        torch.manual_seed(3)
        conv = sa.FastConv3d(32, 64, 3, padding=1, bias=bias).to(device).to(memory_format=CL)
        norm = sa.FastGroupNorm(8, 64, activation="relu").to(device)
        conv.gn_groups = 8
        return conv, norm

    for halo in (0, 1):
        conv, norm = pair()
        norm.out_halo = halo
        x = _x(device).detach()
        runs = []
        for fused in (True, False):
            xi = x.clone().requires_grad_()
            with torch.autocast("cuda", dtype=torch.bfloat16):
                y = conv_then_norm(conv, norm, xi) if fused else norm(conv(xi))
            assert hasattr(y, "_sfh_slab") == bool(halo)
            grads = torch.autograd.grad(y, (xi, conv.weight, norm.weight, norm.bias), torch.ones_like(y) / 8)
            runs.append((y, *grads))
        assert all(torch.equal(a, b) for a, b in zip(*runs))
    conv, norm = pair()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        handle = conv.register_forward_hook(lambda *a: None)
        assert conv_then_norm(conv, norm, x) is None
        handle.remove()
        assert conv_then_norm(conv, norm, x) is not None
        assert conv_then_norm(pair(bias=True)[0], norm, x) is None


@pytest.mark.parametrize("attribute", ["forward", "_compiled_call_impl"])
def test_a_block_calls_what_an_instance_has_put_in_place_of_its_forward(device, attribute):
    """A wrapper set on one convolution or norm (an offloading hook, a probe, ``module.compile()``) runs inside a block too."""
    from scaffold_amd.unet import DoubleConv

    block = DoubleConv(32, 32, 8).to(device).to(memory_format=CL)
    x = _x(device).detach()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        want = block(x)
        for i in (0, 1, 3, 4):
            module, calls = block.double_conv[i], []
            setattr(module, attribute, lambda *a, _f=module.forward, **k: (calls.append(1), _f(*a, **k))[1])
            assert torch.equal(block(x), want) and len(calls) == 1
            if attribute == "forward":
                del module.forward
            else:
                module._compiled_call_impl = None


def test_geometry_in_a_subclass_of_int(device):
    """Sizes may be any ``int`` (a configuration's enum, say), through the modules and their gradients too."""
    import enum

    n = enum.IntEnum("n", {"one": 1, "two": 2})
    for dtype in (torch.bfloat16, torch.float32):
        for plain, other in ((sa.FastConv3d(32, 32, 3, padding=1), sa.FastConv3d(32, 32, 3, n.one, n.one, n.one)),
                             (sa.FastConvTranspose3d(32, 32, 2, 2), sa.FastConvTranspose3d(32, 32, n.two, n.two))):
            other.load_state_dict(plain.state_dict())
            runs = []
            for module in (plain, other):
                module.to(device, dtype).to(memory_format=CL)
                x = torch.linspace(-1, 1, 32 * 128, device=device).view(1, 32, 4, 4, 8).to(dtype).contiguous(memory_format=CL).requires_grad_()
                y = module(x)
                runs.append((y, *torch.autograd.grad(y, (x, *module.parameters()), torch.ones_like(y))))
            assert all(torch.equal(a, b) for a, b in zip(*runs))
    with pytest.raises(NotImplementedError):  # a bool is none
        sa.conv3d_forward(x.detach(), plain.weight.detach(), None, True, 1)


def test_the_skip_connection_is_not_written_in_place(device):
    """It is the pooled tensor's own memory: a write into it would change that tensor under its other uses, so autograd refuses
    it, as for any output of a function that returns views; out of place the gradients are those of x used three times."""
    pool = sa.FastMaxPool3d(2)
    x = _x(device)
    h = x * 1
    y, skip = pool.with_skip(h)
    assert skip.data_ptr() == h.data_ptr()
    with pytest.raises(RuntimeError, match="modified inplace"):
        skip.mul_(2)
    (got,) = torch.autograd.grad(y.float().sum() + (skip * 2).float().sum() + h.float().sum(), x)
    want = 3 + torch.autograd.grad(torch.nn.functional.max_pool3d(x.float(), 2).sum(), x)[0]
    assert torch.equal(got, want)
