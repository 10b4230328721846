"""The splat backward's 512-thread blocks (up to 512 tiles) and the 256-thread ones past them, on the
projection and on the slot records, against the kernel on gathered operands: every slot's gradients
(its theta's taken on to conic and mean by the formula), slots with holes, few and many per tile."""
import pytest
import torch

from helpers import config_inputs
from oracle import splat as osplat
from ttsplat import binned, kernels
from ttsplat.camera import pinhole

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,G,K,holes", [(16, 16, 3, 1, False), (16, 16, 90, 33, True),
                                           (128, 128, 2000, 128, True), (128, 64, 3000, 300, False),
                                           (256, 512, 4000, 64, False), (272, 512, 4000, 64, True)])
def test_backward_matches_gathered_operands(H, W, G, K, holes):
    print(f"[wide] {H}x{W} {G} {K}", flush=True)
    _, P, _ = config_inputs("c1_ref", G=G)
    T = (H // 16) * (W // 16)
    camb = pinhole(H, W, (0.2, 0.3, 3.0)).device_block("cuda")
    order = torch.empty(T, device="cuda", dtype=torch.int32)
    rec = torch.empty(T, K, 12, device="cuda")
    pos = torch.empty(T, device="cuda", dtype=torch.int32)
    proj, _, idx, valid, _, _ = kernels.geom_fwd_assign_bins(P.cuda(), camb, H, W, 16, K, 2048,
                                                             order=order, slot_rec=rec,
                                                             pos_count=pos)
    bg = torch.tensor([0.05, 1.0, 0.9, 0.8], device="cuda")
    origins = binned.TileMap(H, W, 16, device="cuda").origins.double()
    g = torch.Generator().manual_seed(K)
    gi = torch.randn(H, W, 3, generator=g).cuda()

    def check(gslot, gwb, valid):
        th, col, oc = kernels.theta_gather(proj, idx, valid, H, W, 16, 4.0)
        gw2 = torch.empty(T, device="cuda")
        gth, gcol, goc = kernels.splat_bwd_theta(th, col, oc, bg, H, W, 16, img, den, gi, gw2)
        v = valid.bool()
        want = torch.cat([gcol, goc[..., None]], -1)[v]
        # 256 pixel terms in another order, against the tile's largest gradient
        tol = 256 * 2.0 ** -22 * float(want.abs().max())
        assert float((gslot[..., 5:9][v] - want).abs().max()) <= tol
        assert float((gwb - gw2).abs().max()) <= 256 * 2.0 ** -22 * float(gw2.abs().max())
        p = proj[idx.long()].double()
        conic, mu = p[..., 2:5].requires_grad_(True), p[..., 0:2].detach().requires_grad_(True)
        th2 = osplat.theta_u_gathered(conic, mu, origins, 4.0)
        want = torch.cat(torch.autograd.grad(th2, [conic, mu], gth.double()), -1)[v]
        got = gslot[..., 0:5].double()[v]
        # the contract of the slot gradients: 1e-3 relative L2 (a row of 16 left out is 1/16 or so)
        for c in range(5):
            e = float((got[:, c] - want[:, c]).norm() / want[:, c].norm())
            print(f"  column {c}: {e:.2e}", flush=True)
            assert e <= 1e-3, (c, e)

    img, den = kernels.splat_fwd(proj, idx, valid, bg, H, W, 16, 4.0)
    gwb = torch.empty(T, device="cuda")
    check(kernels.splat_bwd_rec(rec, pos, order, bg, H, W, 16, 4.0, img, den, gi, gwb=gwb), gwb,
          valid)
    if holes:
        valid = valid * (torch.rand(T, K, generator=g) > 0.4).to(torch.uint8).cuda()
        img, den = kernels.splat_fwd(proj, idx, valid, bg, H, W, 16, 4.0)
    gwb = torch.empty(T, device="cuda")
    check(kernels.splat_bwd(proj, idx, valid, bg, H, W, 16, 4.0, img, den, gi, gwb=gwb), gwb, valid)
