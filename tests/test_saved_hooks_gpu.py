"""Gradients under saved-tensor hooks.  A hook may hand a saved tensor back in another layout: ``save_on_cpu`` returns it in
the default one, and the kernels read plain channels-last pointers.  The values are the ones that were saved, so every
gradient is the ordinary one, bit for bit; a hook that hands back something else is refused before anything is launched."""

import pytest
import torch

import scaffold_amd as sa
from scaffold_amd.modules import conv_then_norm

pytestmark = pytest.mark.gpu
CL = torch.channels_last_3d


def _x(device, c=32, dtype=torch.bfloat16):
    return torch.randn(2, c, 4, 6, 12, device=device).to(dtype).contiguous(memory_format=CL).requires_grad_()


def _to(module, device, dtype=torch.float32):
    return module.to(device=device, dtype=dtype).to(memory_format=CL)


def _cases(device):
    """name -> (function of its inputs, inputs, parameters)"""
    torch.manual_seed(11)
    conv = _to(sa.FastConv3d(32, 64, 3, padding=1), device)
    half = _to(sa.FastConv3d(32, 64, 3, padding=1, bias=False), device, torch.bfloat16)
    stem = _to(sa.FastConv3d(3, 32, 3, padding=1, bias=False), device)
    shard = _to(sa.FastConv3d(32, 32, 3, padding=1, bias=False), device)
    shard.shard_halo = True
    fp32 = _to(sa.FastConv3d(32, 32, 3, padding=1), device)
    head = _to(sa.FastConv3d(32, 6, 1), device)
    pair = _to(sa.FastConv3d(64, 32, 3, padding=1, bias=False), device)
    norm = _to(sa.FastGroupNorm(8, 64, activation="relu"), device)
    up = _to(sa.FastConvTranspose3d(32, 32, 2, stride=2), device)
    labels = torch.randint(0, 32, (2, 4, 6, 12), device=device)
    weight = torch.rand(32, device=device)
    block = sa.FastConv3d(32, 64, 3, padding=1, bias=False)
    block = _to(block, device)
    a, b = _x(device), _x(device)
    return {
        "conv": (conv, (a,), conv), "conv bf16 weights": (half, (a,), half), "stem": (stem, (_x(device, 3),), stem), "shard": (shard, (a,), shard),
        "conv fp32": (fp32, (_x(device, dtype=torch.float32),), fp32), "head": (head, (a,), head), "pair": (pair, (a, b), pair),
        "norm": (norm, (_x(device, 64),), norm), "up": (up, (a,), up), "conv and norm": (lambda x: conv_then_norm(block, norm, x), (a,), block),
        "pool": (sa.max_pool3d_2x, (a,), None), "loss": (lambda x: sa.ce_dice_loss(x, labels, weight), (a,), None),
    }


NAMES = ["conv", "conv bf16 weights", "stem", "shard", "conv fp32", "head", "pair", "norm", "up", "conv and norm", "pool", "loss"]


def _gradients(fn, inputs, module):
    wrt = [*inputs, *(module.parameters() if module is not None else ())]
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=inputs[0].dtype is torch.bfloat16):
        y = fn(*inputs)
    gy = torch.linspace(-1, 1, y.numel(), device=y.device).to(y.dtype).view(y.shape) if y.dim() else torch.ones_like(y)
    return torch.autograd.grad(y, wrt, gy)


@pytest.mark.parametrize("name", NAMES)
def test_another_layout_gives_the_same_gradients(device, name):
    fn, inputs, module = _cases(device)[name]
    want = _gradients(fn, inputs, module)
    with torch.autograd.graph.save_on_cpu(pin_memory=True):
        got = _gradients(fn, inputs, module)
    assert all(torch.equal(w, g) for w, g in zip(want, got))


@pytest.mark.parametrize("mode", [None, "end", "early"])
def test_a_networks_pass_with_waiting_weight_gradients(device, mode):
    torch.manual_seed(12)
    net = _to(sa.UNet(1, 3, layers=3, base_width=32), device).set_shard_halo(True)
    if mode:
        net.defer_weight_gradients(early=mode == "early")
    x = torch.randn(1, 1, 8, 32, 64, device=device).contiguous(memory_format=CL)
    labels = torch.randint(0, 3, (1, 8, 32, 64), device=device)

    def grads():
        net.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            logits = net(x)
        sa.ce_dice_loss(logits, labels).backward()
        return [p.grad.clone() for p in net.parameters()]

    want = grads()
    with torch.autograd.graph.save_on_cpu(pin_memory=True):
        got = grads()
    assert all(torch.equal(w, g) for w, g in zip(want, got))


@pytest.mark.parametrize("change", [lambda t: t.cpu(), lambda t: t.float().double(), lambda t: t.flatten()[:1]], ids=["host", "dtype", "shape"])
@pytest.mark.parametrize("name", ["conv", "up", "norm", "loss"])
def test_what_is_not_the_saved_tensor_is_refused(device, name, change):
    fn, inputs, module = _cases(device)[name]
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: change(t) if t.dim() == 5 else t):
        with pytest.raises(RuntimeError, match="a saved tensor came back as"):
            _gradients(fn, inputs, module)
