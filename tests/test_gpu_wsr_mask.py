"""The keep mask of wsr_polysplat belongs to the call: what its owner writes into it between forward
and backward changes nothing."""
import pytest
import torch

from ttsplat import backward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bool, torch.uint8, torch.float32])
def test_mask_rewritten_before_the_backward(dtype):
    g = torch.Generator().manual_seed(4)
    G, P = 70, 300
    leaves = [t.cuda().requires_grad_(True) for t in
              (torch.randn(G, 6, generator=g) * 0.4, torch.rand(G, generator=g) + 0.05,
               torch.rand(G, 3, generator=g), torch.tensor(0.3))]
    phi = torch.randn(P, 6, generator=g).cuda()
    cb, R = torch.tensor([0.9, 0.5, 0.2]).cuda(), torch.randn(P, 3, generator=g).cuda()
    keep = torch.rand(G, generator=g) > 0.3

    def grads(rewrite):
        mask = keep.to("cuda", dtype)
        C = backward.wsr_polysplat(*leaves, phi, cb, mask)
        if rewrite:
            mask.copy_(~keep)
        return torch.autograd.grad((C * R).sum(), leaves)

    for a, b in zip(grads(True), grads(False)):
        assert torch.equal(a, b)
