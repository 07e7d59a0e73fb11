"""Packed weight forms made straight from an fp32 master, and the module path that reads them under autocast."""

import pytest
import torch

import scaffold_amd as sa
from scaffold_amd import _lib

pytestmark = pytest.mark.gpu
CL = torch.channels_last_3d


@pytest.mark.parametrize("cin,cout,k,stride,spatial", [
    (32, 32, 3, 1, (4, 6, 18)), (64, 96, 3, 1, (3, 5, 9)), (256, 128, 3, 1, (4, 8, 8)), (64, 128, 2, 2, (4, 6, 8)),
])
@pytest.mark.parametrize("layout", ["channels_last", "contiguous", "offset"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rounded_on_the_way_is_cast_then_packed(device, cin, cout, k, stride, spatial, layout, dtype):
    g = torch.Generator().manual_seed(3)
    w = torch.randn((cout, cin, k, k, k), generator=g).to(device)
    if layout == "channels_last":
        w = w.contiguous(memory_format=CL)
    elif layout == "offset":  # off the 16-byte grid
        w = torch.empty(w.numel() + 1, device=device)[1:].view(w.shape).copy_(w)
    pad = 1 if k == 3 else 0
    in_shape = (1, cin, *spatial)
    want = sa.pack_weights(w.to(dtype), torch.Size(in_shape), stride, pad, 1)
    got = _lib.native().pack_master(w, dtype, in_shape, stride, pad, 1, True)
    assert got[2] and all(torch.equal(a, b) for a, b in zip(want, got))
    fwd_only = _lib.native().pack_master(w, dtype, in_shape, stride, pad, 1, False)
    assert fwd_only[1] is None and torch.equal(fwd_only[0], want[0])


def test_autocast_modules_without_an_optimizers_copies(device):
    """Same outputs and data gradients, bit for bit, as with the weights cast in front; the parameters' gradients arrive in
    fp32 unrounded (the cast path rounded them to 16 bits first)."""
    torch.manual_seed(5)
    x = torch.randn(1, 32, 6, 8, 20, device=device).to(torch.bfloat16).contiguous(memory_format=CL)
    for make in (lambda: sa.FastConv3d(32, 64, 3, padding=1, bias=True), lambda: sa.FastConv3d(32, 6, 1, bias=True),
                 lambda: sa.FastConvTranspose3d(32, 32, 2, stride=2)):
        m = make().to(device).to(memory_format=CL)
        half = make().to(device).to(memory_format=CL)
        half.load_state_dict(m.state_dict())
        half = half.to(torch.bfloat16)
        xa, xb = x.clone().requires_grad_(), x.clone().requires_grad_()
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = m(xa)
        ref = half(xb)
        assert torch.equal(y, ref)
        gy = torch.randn_like(y)
        y.backward(gy)
        ref.backward(gy)
        assert torch.equal(xa.grad, xb.grad)
        for p, q in zip(m.parameters(), half.parameters()):
            assert p.grad.dtype is torch.float32 and torch.equal(p.grad.to(torch.bfloat16), q.grad)
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
            assert torch.equal(m(x), y.detach())


def test_a_master_may_step_between_forward_and_backward(device):
    """As where autocast has cast the weight: the gradients are those of the weight the forward read."""
    from scaffold_amd.modules import conv_then_norm

    torch.manual_seed(6)
    norm = sa.FastGroupNorm(8, 32, activation="relu").to(device)
    conv = sa.FastConv3d(32, 32, 3, padding=1, bias=False)
    pair = sa.FastConv3d(64, 32, 3, padding=1, bias=False)
    x = torch.randn(1, 32, 4, 8, 32, device=device).to(torch.bfloat16).contiguous(memory_format=CL)
    for module, call in ((conv, conv), (conv, lambda t: conv_then_norm(conv, norm, t)), (pair, lambda t: pair(t, x)),
                         (sa.FastConv3d(32, 6, 1), None), (sa.FastConvTranspose3d(32, 32, 2, stride=2), None)):
        module.to(device).to(memory_format=CL)
        runs = []
        for step in (False, True):
            a = x.clone().requires_grad_()
            with torch.autocast("cuda", dtype=torch.bfloat16):
                y = (call or module)(a)
            if step:
                with torch.no_grad():
                    for p in module.parameters():
                        p.mul_(2)
            runs.append(torch.autograd.grad(y, (a, *module.parameters()), torch.ones_like(y)))
        assert all(torch.equal(p, q) for p, q in zip(*runs))
