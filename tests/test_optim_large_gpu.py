"""Clipped Adam on parameters of more chunks than its launch has workgroups, and past the sizes from which its arrays (16.8 M elements) and
the gradients of the norm (67.1 M) go past the caches."""

import pytest
import torch

import scaffold_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,offset,shadow", [
    ((2047 * 8192 + 1, 5), 0, None),                       # 2048 + 1 chunks, below the size
    ((2049 * 8192 + 3, 70001), 0, torch.bfloat16),         # a workgroup with two chunks; a cut chunk
    ((2 * 2048 * 8192 + 8191,), 0, torch.float16),         # every workgroup with two or three
    ((2050 * 8192 + 6,), 1, torch.bfloat16),               # off the 16-byte grid
    ((8200 * 8192 + 9, 33), 0, None),                      # the norm's loads too
])
def test_against_stock_adam(sizes, offset, shadow):
    def make(seed):
        g = torch.Generator(device="cuda").manual_seed(seed)
        return [torch.randn(n + offset, generator=g, device="cuda")[offset:] for n in sizes]

    ours, stock = ([t.requires_grad_(True) for t in make(0)] for _ in range(2))
    opt = sa.FusedClipAdam(ours, lr=1e-2, max_norm=1.0, shadow_dtype=shadow)
    ref = torch.optim.Adam(stock, lr=1e-2, foreach=False, fused=False)
    for step in range(2):
        for ps in (ours, stock):
            for p, gr in zip(ps, make(1 + step)):
                p.grad = gr
        opt.step()
        norm = torch.linalg.vector_norm(torch.cat([p.grad for p in stock]).double()).item()
        # a thread's sum of 32 squares, a tree, and the slots' in a tree: below 1e-5
        assert abs(opt.grad_norm.item() - norm) <= 1e-5 * norm
        scale = 1.0 / (norm + 1e-6)
        for p in stock:
            p.grad.mul_(scale)
        ref.step()
    for p, q in zip(ours, stock):
        a, b = opt.state[p], ref.state[q]
        assert torch.allclose(p, q, rtol=1e-5, atol=1e-6)
        # gradients are clipped to 1 / sqrt(elements) and less
        assert torch.allclose(a["exp_avg"], b["exp_avg"], rtol=2e-5, atol=1e-9) and torch.allclose(a["exp_avg_sq"], b["exp_avg_sq"], rtol=4e-5, atol=1e-14)
        if shadow is not None:
            assert torch.equal(p._sfh_shadow.reshape(-1), p.detach().to(shadow))
