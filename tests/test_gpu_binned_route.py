"""render_binned_device's own projection, bins and dispatch order against the general calls on the
same model: bins given by the caller, tiles in index order, a second projection."""
import pytest
import torch

from helpers import config_inputs
from ttsplat import binned, kernels
from ttsplat.camera import pinhole
from ttsplat.model import GaussianModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,K,G,H,W", [(16, 128, 1, 16, 32), (16, 96, 513, 48, 80),
                                       (16, 256, 2000, 128, 128), (32, 64, 700, 64, 96)])
def test_render_binned_matches_given_bins(S, K, G, H, W):
    _, P, _ = config_inputs("c1_ref", G=G)
    P = P.cuda()
    cam, tmap = pinhole(H, W, (0.3, 0.2, 3.0)), binned.TileMap(H, W, S)
    R = torch.randn(H, W, 3, generator=torch.Generator().manual_seed(2)).cuda()
    out = []
    for given in (False, True):
        model = GaussianModel(P.clone())
        model.params.requires_grad_(True)
        model.w_b_raw.requires_grad_(True)
        bins = None
        if given:
            with torch.no_grad():
                bins = binned.render_binned_device(model, cam, tmap, K=K, return_bins=True)[1]
        img = binned.render_binned_device(model, cam, tmap, K=K, cached_bins=bins)
        g = torch.autograd.grad((img * R).sum(), [model.params, model.w_b_raw])
        with torch.no_grad():
            assert torch.equal(binned.render_binned_device(model, cam, tmap, K=K), img)
        out.append((img.detach(), *g))
    assert torch.equal(out[0][0], out[1][0])
    for a, b in zip(out[0][1:], out[1][1:]):
        # given bins scatter their slots with atomics: up to 9 terms in another order
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-5 * float(b.abs().max()))


@pytest.mark.parametrize("S,K,G", [(16, 64, 900), (16, 200, 3000), (32, 128, 5), (16, 32, 0)])
def test_int64_ids_are_the_int32_ones(S, K, G):
    H, W = 64, 96
    g = torch.Generator().manual_seed(G)
    mu = (torch.rand(G, 2, generator=g) * torch.tensor([W * 1.2, H * 1.2]) - 5).cuda()
    keep = (torch.rand(G, generator=g) > 0.2).cuda()
    span = binned.TileMap(H, W, S).span
    a = kernels.assign_bins(mu, keep, H, W, S, K, span)
    b = kernels.assign_bins(mu, keep, H, W, S, K, span, idx_dtype=torch.int64)
    assert b[0].dtype == torch.int64 and torch.equal(a[0].long(), b[0])
    assert all(torch.equal(x, y) for x, y in zip(a[1:], b[1:]))
    for k in (keep, keep.float(), keep.to(torch.uint8)):
        idx, valid = binned.assign_bins(mu, k, binned.TileMap(H, W, S), 1, K)
        assert torch.equal(idx, b[0]) and valid.dtype == torch.bool
        assert torch.equal(valid, b[1].bool())


@pytest.mark.parametrize("dense", [False, True])
def test_background_inputs_between_forward_and_backward(dense):
    """c_b, and a w_b_raw that needs no gradient, may change in place before the backward; w_b_raw's
    gradient can be differentiated again (through softplus: the renders themselves cannot)."""
    from ttsplat.render import render
    _, P, _ = config_inputs("c1_ref", G=200)
    cam, tmap = pinhole(32, 48, (0.3, 0.2, 3.0)), binned.TileMap(32, 48)

    def image(model):
        return render(model, cam, "A") if dense else binned.render_binned_device(model, cam, tmap)

    model = GaussianModel(P.cuda())
    model.params.requires_grad_(True)
    img = image(model)
    model.c_b.mul_(0.5)
    model.w_b_raw.add_(1.0)
    img.square().sum().backward()
    assert bool(torch.isfinite(model.params.grad).all())

    model = GaussianModel(P.cuda())
    w = model.w_b_raw.requires_grad_(True)
    c = model.c_b.requires_grad_(True)
    loss = image(model).square().sum()
    gw, gc = torch.autograd.grad(loss, [w, c], retain_graph=True)
    assert gw.shape == w.shape and torch.equal(gc, torch.zeros(3, device="cuda"))
    (g2,) = torch.autograd.grad(loss, w, create_graph=True)
    assert torch.allclose(gw, g2, rtol=1e-5)
    (gg,) = torch.autograd.grad(g2, w)
    s = torch.sigmoid(w.detach())
    assert torch.allclose(gg, g2.detach() * (1 - s), rtol=1e-5)
