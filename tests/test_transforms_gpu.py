"""The host path under tracers and transforms: a traced module follows its inputs and parameters, and forward-mode
differentiation and functorch transforms are refused instead of dropping derivatives."""
import pytest
import torch

import scaffold_amd as sa

CL = torch.channels_last_3d
pytestmark = pytest.mark.gpu


def _modules():
    torch.manual_seed(5)
    conv = sa.FastConv3d(32, 32, 3, padding=1, bias=False)
    norm = sa.FastGroupNorm(8, 32, activation="relu")
    up = sa.FastConvTranspose3d(32, 16, 2, stride=2)
    stages = {"conv": conv, "norm": norm, "up": up, "pool": sa.FastMaxPool3d(2), "block": torch.nn.Sequential(conv, norm)}
    return {k: m.cuda().to(torch.bfloat16).to(memory_format=CL) for k, m in stages.items()}


def _x(seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn((1, 32, 6, 8, 12), generator=g, device="cuda").to(torch.bfloat16).contiguous(memory_format=CL)


@pytest.mark.parametrize("stage", ["conv", "norm", "up", "pool", "block"])
def test_traced_module_follows_its_input(stage):
    module = _modules()[stage]
    traced = torch.jit.trace(module, (_x(1),), check_trace=False)
    x = _x(2)
    a, b = x.clone().requires_grad_(), x.clone().requires_grad_()
    want, got = module(a), traced(b)
    assert torch.equal(want, got)
    gy = torch.randn_like(want)
    params = list(module.parameters())
    for w, t in zip(torch.autograd.grad(want, [a, *params], gy), torch.autograd.grad(got, [b, *params], gy)):
        assert torch.equal(w, t)


@pytest.mark.parametrize("stage", ["conv", "norm", "up", "pool"])
def test_forward_mode_and_functorch_are_refused(stage):
    module = _modules()[stage]
    x = _x(1)
    with torch.autograd.forward_ad.dual_level():
        with pytest.raises(NotImplementedError):
            module(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))
    with pytest.raises(RuntimeError):
        torch.func.vmap(module)(torch.stack((x, x)))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: module(t).float().sum())(x)


def test_loss_under_forward_mode_is_refused_and_traces():
    logits = torch.randn((1, 6, 4, 8, 8), device="cuda").contiguous(memory_format=CL)
    labels = torch.randint(0, 6, (1, 4, 8, 8), device="cuda")
    with torch.autograd.forward_ad.dual_level():
        with pytest.raises(NotImplementedError):
            sa.ce_dice_loss(torch.autograd.forward_ad.make_dual(logits, torch.ones_like(logits)), labels)
    traced = torch.jit.trace(sa.ce_dice_loss, (logits, labels), check_trace=False)
    assert torch.equal(traced(logits * 2, labels), sa.ce_dice_loss(logits * 2, labels))
