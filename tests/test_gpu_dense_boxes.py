"""The dense backward's ways through the gaussians of a block: two large boxes walked jointly, one
large box among small ones, by one block and in shares; against autograd of the formula in 64 bits,
and twice with the same result."""
import pytest
import torch

from ttsplat import _lib, kernels

from test_gpu_dense_cull import grads, oracle, oracle_detached_z, records, render

pytestmark = pytest.mark.gpu


# four waves per gaussian (G <= 4096, or 2^17 pixels and more), sixteen and one; cells of 8 x 8
# pixels cut at the image's edge; `big` every how many gaussians (1: all); thin ones (no box:
# condition past the bound) among them
@pytest.mark.parametrize("G,H,W,big,cond", [
    (1, 300, 301, 1, 10.0), (3, 9, 700, 1, 10.0), (4, 64, 64, 1, 10.0), (5, 131, 77, 1, 10.0),
    (9, 1, 1201, 1, 10.0), (40, 203, 199, 1, 30.0), (41, 333, 400, 3, 10.0),
    (260, 150, 160, 97, 10.0), (257, 150, 103, 1, 10.0), (300, 510, 515, 40, 10.0),
    (18, 120, 130, 2, 1e5), (4101, 97, 60, 1, 10.0), (4103, 91, 95, 600, 10.0),
    (4102, 64, 33, 3, 10.0)])
@pytest.mark.parametrize("arm", ["A", "SZ", "RV"])
def test_backward_follows_autograd(G, H, W, big, cond, arm):
    print(f"[boxes] {G} {H}x{W} {big} {arm}", flush=True)
    proj = records(G, H, W, seed=G, cond=10.0, size=2.0)
    wide = records(G, H, W, seed=G + 1, cond=cond, size=1.5 * max(H, W))
    proj[::big] = wide[::big]
    proj[:, 6:10] *= 0.2          # revealage: many opaque layers would leave nothing to see
    gi = torch.randn(H, W, 3, generator=torch.Generator().manual_seed(3))
    got, gwb = grads(proj.cuda(), H, W, arm, gi.cuda())
    again, gwb2 = grads(proj.cuda(), H, W, arm, gi.cuda())
    assert torch.equal(got, again) and torch.equal(gwb, gwb2)
    P = proj.double().requires_grad_(True)
    beta = torch.tensor(3.0, dtype=torch.float64, requires_grad=True)
    (oracle_detached_z(P, H, W, arm, beta) * gi.double()).sum().backward()
    ref = torch.cat([P.grad[:, 2:5], P.grad[:, 0:2], P.grad[:, 6:10]], 1)
    # the contract of the dense gradients: 1e-3 relative L2 (u carries 12 eps cond)
    for sl in (slice(0, 3), slice(3, 5), slice(5, 8), slice(8, 9)):
        e = float((got[:, sl].cpu().double() - ref[:, sl]).norm() / ref[:, sl].norm())
        print(f"  {sl.start}: {e:.2e}")
        assert e <= 1e-3, (sl, e)
    if arm == "SZ":
        d = abs(float(got[:, 9].double().sum()) - float(beta.grad))
        assert d <= 1e-3 * abs(float(beta.grad)) + 1e-5


# every pair visited (up to 2, 8, 16 and 32 gaussians by arm and size); tiles of 16 with 256, 512
# and 1024 threads, of 32 and of 8; lists of whole-image boxes with a small or thin one in between
@pytest.mark.parametrize("G,H,W", [(2, 31, 9), (8, 40, 33), (16, 257, 3), (17, 60, 70),
                                   (32, 263, 259), (33, 263, 259), (129, 257, 264), (130, 401, 330),
                                   (300, 262, 258), (257, 529, 512), (70, 513, 520),
                                   (1100, 70, 90)])
@pytest.mark.parametrize("arm", ["A", "SZ", "RV"])
def test_forward_of_large_boxes_follows_the_formula(G, H, W, arm):
    print(f"[boxes-fwd] {G} {H}x{W} {arm}", flush=True)
    proj = records(G, H, W, seed=G, cond=10.0, size=1.5 * max(H, W))
    proj[::37] = records(G, H, W, seed=G + 1, cond=1e5, size=30.0)[::37]
    proj[:, 6:10] *= 0.1
    # u carries 12 eps (a dx^2 + c dy^2) / k
    ref = oracle(proj, H, W, arm)
    assert float((render(proj.cuda(), H, W, arm).cpu() - ref).abs().max()) <= 1e-4


@pytest.mark.parametrize("arm", ["A", "SZ", "RV"])
def test_wide_images_give_up_the_boxes(arm):
    """A side over 65536: every pair is visited, in both passes."""
    H, W, G = 1, 65537, 40
    proj = records(G, H, W, seed=1, cond=10.0, size=3.0)
    proj[0, 0], proj[1, 0] = 65530.0, 2.0
    gi = torch.randn(H, W, 3, generator=torch.Generator().manual_seed(3))
    P = proj.double().requires_grad_(True)
    beta = torch.tensor(3.0, dtype=torch.float64)
    ref = oracle_detached_z(P, H, W, arm, beta)
    (ref * gi.double()).sum().backward()
    assert float((render(proj.cuda(), H, W, arm).cpu() - ref.detach()).abs().max()) <= 1e-4
    got = grads(proj.cuda(), H, W, arm, gi.cuda())[0].cpu().double()[:, :9]
    want = torch.cat([P.grad[:, 2:5], P.grad[:, 0:2], P.grad[:, 6:10]], 1)
    for sl in (slice(0, 3), slice(3, 5), slice(5, 8), slice(8, 9)):
        assert float((got[:, sl] - want[:, sl]).norm()) <= 1e-3 * float(want[:, sl].norm())


def test_backward_of_more_blocks_than_a_grid_row():
    """Over 2^21 blocks: the last gaussians' gradients (2^23 and more of them, four to a block) are
    those of the same gaussians alone."""
    H, W, n = 6, 5, 12
    tail = records(n, H, W, seed=2).cuda()
    proj = torch.zeros((1 << 23) + n, 12, device="cuda")
    proj[:, 0], proj[:, 2], proj[:, 4] = -100.0, 1.0, 1.0
    proj[-n:] = tail
    bg = torch.tensor([0.05, 0.9, 1.0, 0.8], device="cuda")
    img, den = kernels.render_dense(tail, H, W, 4.0, bg)
    gi = torch.randn(H, W, 3, generator=torch.Generator().manual_seed(1)).cuda()
    got, gwb = kernels.render_dense_bwd(proj, H, W, 4.0, bg, img, den, gi)
    few, gwb2 = kernels.render_dense_bwd(torch.cat([tail] * 400), H, W, 4.0, bg, img, den, gi)
    assert torch.equal(got[-n:], few[-n:]) and torch.equal(gwb, gwb2)
    assert not bool(got[:-n].any())


@pytest.mark.parametrize("arm", ["A", "SZ", "RV"])
@pytest.mark.parametrize("G", [40, 300])
def test_backward_of_images_past_one_run(G, arm):
    """2^25 pixels are one run of the backward: an image of rows past it against the same gaussians
    on a crop around the cut, and the workspace."""
    W, H, cut = 8192, 4096 + 40, 4096
    crop = records(G, 80, 120, seed=4, size=4.0)
    crop[:, 1] = (crop[:, 1] * 64).round() / 64        # the same place 4056 rows further down
    crop[:, 0] = crop[:, 0].clamp(10, 110)
    full = crop.clone()
    full[:, 1] += cut - 40
    g = torch.Generator().manual_seed(3)
    gi = torch.zeros(H, W, 3, device="cuda")
    gc = torch.randn(80, 120, 3, generator=g).cuda()
    gi[cut - 40:, :120] = gc
    assert _lib.load().tts_dense_workspace_bytes(G, H * W) < 1 << 30
    a, wa = grads(full.cuda(), H, W, arm, gi)
    b, wb = grads(crop.cuda(), 80, 120, arm, gc)
    # the same terms in another order
    for sl in (slice(0, 3), slice(3, 5), slice(5, 8), slice(8, 9)):
        assert float((a[:, sl] - b[:, sl]).norm()) <= 1e-3 * float(b[:, sl].norm())
    assert abs(float(wa) - float(wb)) <= 1e-3 * abs(float(wb)) + 1e-4


def test_backward_of_rows_past_one_run():
    """One row of more than 2^25 pixels: the second run has no gradient to add."""
    W = (1 << 25) + 70
    proj = records(9, 1, 200, seed=4, size=4.0).cuda()
    gi = torch.zeros(1, W, 3, device="cuda")
    gi[0, :200] = torch.randn(200, 3, generator=torch.Generator().manual_seed(3)).cuda()
    a, wa = grads(proj, 1, W, "A", gi)
    b, wb = grads(proj, 1, 200, "A", gi[:, :200].contiguous())
    assert float((a - b).norm()) <= 1e-4 * float(b.norm())
    assert abs(float(wa) - float(wb)) <= 1e-4 * abs(float(wb)) + 1e-4
