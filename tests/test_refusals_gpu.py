"""Calls that are not served are refused before anything is launched: the gate of the convolution modules comes before the
packing of their weights, and operands of two 16-bit types are not mixed because a packed weight is at hand."""

import pytest
import torch

import scaffold_amd as sa
from scaffold_amd import _lib
from scaffold_amd import conv3d as c3
from scaffold_amd import modules
from scaffold_amd.unet import DoubleConv

pytestmark = pytest.mark.gpu
CL = torch.channels_last_3d


def _x(device, c, dtype=torch.bfloat16):
    return torch.randn(1, c, 4, 8, 32, device=device).to(dtype).contiguous(memory_format=CL)


def _weights(module, device, kind):
    """The module with the weights a program may have: bf16 ones, fp32 masters, masters with an optimizer's bf16 copies."""
    module = module.to(device).to(memory_format=CL)
    if kind == "bf16":
        return module.to(torch.bfloat16)
    if kind == "shadows":
        for p in module.parameters():
            p._sfh_shadow, p._sfh_shadow_version = p.detach().to(torch.bfloat16), p._version
    return module


@pytest.mark.parametrize("kind", ["bf16", "masters", "shadows"])
@pytest.mark.parametrize("channels", [64, 16, 96])
def test_an_input_of_other_channels_packs_nothing(device, kind, channels, monkeypatch):
    packed = []
    for name in ("pack_weights", "PackedWeights"):
        real = getattr(c3, name)
        monkeypatch.setattr(c3, name, lambda *a, _real=real, **k: (packed.append(a), _real(*a, **k))[1])
    monkeypatch.setattr(modules, "_master_operands", lambda *a: packed.append(a))
    conv = _weights(sa.FastConv3d(32, 32, 3, padding=1, bias=False), device, kind)
    block = _weights(DoubleConv(32, 32, 8), device, kind)
    grouped = _weights(sa.FastConv3d(64, 64, 3, padding=1, groups=2, bias=False), device, kind)
    pair = _weights(sa.FastConv3d(64, 32, 3, padding=1, bias=False), device, kind)
    x = _x(device, channels)
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=kind != "bf16"):
        for call in (lambda: conv(x), lambda: block(x), lambda: grouped(_x(device, 64)), lambda: pair(_x(device, 32), x)):
            with pytest.raises(NotImplementedError):
                call()
    assert not packed


def test_packing_refuses_a_weight_of_another_input(device):
    w = torch.randn(32, 32, 3, 3, 3, device=device)
    assert _lib.native().pack_master(w, torch.bfloat16, (1, 64, 4, 8, 32), 1, 1, 1, True) == (None, None, False)
    with pytest.raises(ValueError, match="does not belong"):
        sa.pack_weights(w.to(torch.bfloat16), (1, 64, 4, 8, 32), 1, 1, 1)


@pytest.mark.parametrize("kind", ["bf16", "shadows"])
def test_two_16_bit_types_do_not_meet_over_a_packed_weight(device, kind):
    """Packed forms of a bf16 and of an fp16 weight have the same size: the weight's own dtype decides."""
    x = _x(device, 32, torch.float16)
    stages = [sa.FastConv3d(32, 32, 3, padding=1, bias=False), DoubleConv(32, 32, 8), sa.FastConvTranspose3d(32, 32, 2, stride=2, bias=False)]
    for module in stages:
        module = _weights(module, device, kind)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=kind != "bf16"):
            module(x.to(torch.bfloat16))            # the packed forms exist
            for grad in (True, False):
                with torch.set_grad_enabled(grad), pytest.raises(NotImplementedError):
                    module(x)


def test_an_operators_packed_weight_does_not_lift_the_dtype_rule(device):
    w = torch.randn(32, 32, 3, 3, 3, device=device).to(torch.bfloat16)
    x = _x(device, 32)
    pf, pd = sa.pack_weights(w, x.shape, 1, 1, 1)
    assert torch.equal(sa.conv3d_forward(x, w, None, 1, 1, packed_weight=pf), sa.conv3d_forward(x, w, None, 1, 1))
    for a, b in ((x.to(torch.float16), w), (x, w.to(torch.float16)), (x, w.float())):
        with pytest.raises(NotImplementedError):
            sa.conv3d_forward(a, b, None, 1, 1, packed_weight=pf)


@pytest.mark.parametrize("kind", ["bf16", "masters", "shadows"])
def test_a_weight_on_the_host_meets_no_kernel(device, kind, monkeypatch):
    """A module that was never moved to the GPU, given an input that was: refused before anything reads its weight."""
    packed = []
    for name in ("pack_weights", "PackedWeights"):
        monkeypatch.setattr(c3, name, lambda *a, **k: packed.append(a))
    host = torch.device("cpu")
    modules_ = [_weights(m, host, kind) for m in (sa.FastConv3d(32, 32, 3, padding=1, bias=False), DoubleConv(32, 32, 8),
                                                  sa.FastConvTranspose3d(32, 32, 2, stride=2, bias=False))]
    x = _x(device, 32)
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=kind != "bf16"):
        for module in modules_:
            with pytest.raises(NotImplementedError):
                module(x)
    assert not packed
