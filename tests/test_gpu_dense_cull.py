"""The dense kernels visit only the gaussians whose support may reach a pixel: the same results as
visiting all of them, at tile edges, list overflows, thin and huge gaussians and non-finite values.

A gaussian whose depth is 1e19 is taken everywhere (the support box is given up for values whose
product with a zero weight need not be zero), and arm A does not read the depth: that is the
general path through the same kernels."""
import pytest
import torch

from ttsplat import kernels

pytestmark = pytest.mark.gpu

BG = [0.05, 0.9, 1.0, 0.8]


def records(G, H, W, seed, cond=100.0, size=3.0):
    """proj [G,12]: conics of condition up to `cond`, means in and around the image."""
    g = torch.Generator().manual_seed(seed)
    u = lambda *s: torch.rand(*s, generator=g, dtype=torch.float64)
    big = size ** 2 * (0.2 + 3.0 * u(G))                     # larger variance, pixels^2
    small = big / torch.exp(torch.log(torch.tensor(cond)) * u(G))
    t = 3.14159 * u(G)
    cs, sn = torch.cos(t), torch.sin(t)
    a = cs * cs / big + sn * sn / small
    c = sn * sn / big + cs * cs / small
    b = cs * sn * (1 / big - 1 / small)
    mu = torch.stack([(1.4 * u(G) - 0.2) * W, (1.4 * u(G) - 0.2) * H], 1)
    o = 0.05 + 0.9 * u(G)
    P = torch.zeros(G, 12, dtype=torch.float64)
    P[:, 0:2], P[:, 2], P[:, 3], P[:, 4] = mu, a, b, c
    P[:, 5] = 2.0 + 2.0 * u(G)
    P[:, 6:9], P[:, 9], P[:, 10] = u(G, 3) * o[:, None], o, o
    return P.float()


def everywhere(proj):
    p = proj.clone()
    p[:, 5] = 1e19
    return p


def oracle(proj, H, W, arm, beta=3.0, k=4.0):
    P = proj.double()
    y, x = torch.meshgrid(torch.arange(H).double() + 0.5, torch.arange(W).double() + 0.5,
                          indexing="ij")
    dx, dy = x.reshape(-1, 1) - P[:, 0], y.reshape(-1, 1) - P[:, 1]
    w = (1 - (P[:, 2] * dx * dx + 2 * P[:, 3] * dx * dy + P[:, 4] * dy * dy) / k).clamp(min=0) ** 2
    if arm == "SZ":
        W0 = w * P[:, 9]
        zs = (W0 * P[:, 5]).sum(1, keepdim=True) / (W0.sum(1, keepdim=True) + 1e-6)
        w = w * torch.sigmoid(-beta * (P[:, 5] - zs))
    num, den = w @ P[:, 6:9], (w * P[:, 9]).sum(1, keepdim=True)
    bg = torch.tensor(BG).double()
    if arm == "RV":
        R = torch.exp(torch.log1p(-(w * P[:, 9]).clamp(max=1 - 1e-4)).sum(1, keepdim=True))
        img = num / (den + 1e-6) * (1 - R) + bg[1:] * R
    else:
        img = (num + bg[0] * bg[1:]) / (den + bg[0])
    return img.reshape(H, W, 3)


def render(proj, H, W, arm="A"):
    bg = torch.tensor(BG, device="cuda")
    if arm == "A":
        return kernels.render_dense(proj, H, W, 4.0, bg)[0]
    sz = torch.tensor([3.0], device="cuda") if arm == "SZ" else None
    return kernels.render_dense_arm(proj, H, W, 4.0, bg, arm, sz)[0]


# tile sides 8, 16 and 32 with ragged edges; one gaussian, one round of tests, several; lists that
# overflow between rounds (size 40: every gaussian reaches every tile)
SIZES = [(1, 7, 9, 3.0), (513, 33, 41, 3.0), (1025, 257, 263, 3.0), (2600, 90, 70, 40.0),
         (1300, 260, 270, 60.0), (1100, 561, 545, 30.0)]


@pytest.mark.parametrize("G,H,W,size", SIZES)
@pytest.mark.parametrize("arm", ["A", "SZ", "RV"])
def test_forward_follows_the_formula(G, H, W, size, arm):
    print(f"[cull] {G} {H}x{W} {arm}", flush=True)
    proj = records(G, H, W, seed=G, size=size)
    ref = oracle(proj, H, W, arm)
    # u carries 12 eps cond (a dx^2 + c dy^2) / k, cond 100: ~1e-4 at worst, averaged over gaussians
    assert float((render(proj.cuda(), H, W, arm).cpu() - ref).abs().max()) <= 1e-4


def test_forward_single_gaussians_are_bit_identical_to_the_general_path():
    """Thin ones included (condition up to 1e7, past the bound's limit)."""
    H, W = 40, 37
    for i, cond in enumerate([1.0, 30.0, 1e3, 1e5, 1e7] * 30):
        p = records(1, H, W, seed=100 + i, cond=cond, size=[0.5, 4.0, 30.0][i % 3]).cuda()
        assert torch.equal(render(p, H, W), render(everywhere(p), H, W)), (i, cond)


@pytest.mark.parametrize("G,H,W,size", SIZES[1:])
def test_forward_sums_match_the_general_path(G, H, W, size):
    p = records(G, H, W, seed=7, cond=1e4, size=size).cuda()
    # two sums of at most G non-negative terms in another order, each within G 2^-24 relative
    assert torch.allclose(render(p, H, W), render(everywhere(p), H, W), rtol=4 * G * 2.0 ** -24,
                          atol=0)


@pytest.mark.parametrize("col,value", [(6, float("nan")), (9, float("inf")), (2, float("nan")),
                                       (0, float("nan"))])
def test_forward_non_finite_record_reaches_every_pixel(col, value):
    """0 * inf and NaN weights give NaN at every pixel, as visiting every pair does."""
    H, W = 50, 66
    p = records(70, H, W, seed=3)
    p[11, 0:2] = -500.0
    p[11, col] = value
    assert bool(torch.isnan(render(p.cuda(), H, W)).any(-1).all())


def grads(proj, H, W, arm, gi):
    """Backward of `render`: (grad [G,9 or 10], gwb)."""
    bg = torch.tensor(BG, device="cuda")
    if arm == "A":
        img, den = kernels.render_dense(proj, H, W, 4.0, bg)
        return kernels.render_dense_bwd(proj, H, W, 4.0, bg, img, den, gi)
    sz = torch.tensor([3.0], device="cuda") if arm == "SZ" else None
    img, den, aux = kernels.render_dense_arm(proj, H, W, 4.0, bg, arm, sz)
    return kernels.render_dense_arm_bwd(proj, H, W, 4.0, bg, arm, img, den, aux, gi, sz)


# row shares 16, 4 and 1; one wave per gaussian (G > 4096, small image) and four (large image);
# a box of one pixel row, boxes larger than the image
@pytest.mark.parametrize("G,H,W,size", [(1, 5, 70, 3.0), (63, 40, 23, 3.0), (65, 33, 31, 50.0),
                                        (255, 1, 90, 3.0), (300, 64, 48, 6.0),
                                        (4101, 41, 27, 2.0), (4097, 400, 340, 0.7)])
@pytest.mark.parametrize("arm", ["A", "SZ", "RV"])
def test_backward_follows_autograd(G, H, W, size, arm):
    print(f"[cull-bwd] {G} {H}x{W} {arm}", flush=True)
    proj = records(G, H, W, seed=G, cond=10.0, size=size)
    if H * W * G > 2e7:       # the 64-bit reference visits every pair: a corner of the image
        proj[:, 0:2] = proj[:, 0:2] % 40
    h, w = (H, W) if H * W * G <= 2e7 else (56, 56)
    g = torch.Generator().manual_seed(3)
    gi = torch.zeros(H, W, 3)
    gi[:h, :w] = torch.randn(h, w, 3, generator=g)
    got, gwb = grads(proj.cuda(), H, W, arm, gi.cuda())
    P = proj.double().requires_grad_(True)
    beta = torch.tensor(3.0, dtype=torch.float64, requires_grad=True)
    img = oracle_detached_z(P, h, w, arm, beta)
    (img * gi[:h, :w].double()).sum().backward()
    ref = torch.cat([P.grad[:, 2:5], P.grad[:, 0:2], P.grad[:, 6:10]], 1)
    # the contract of the dense gradients: 1e-3 relative L2 (u carries 12 eps cond, cond 10)
    for sl in (slice(0, 3), slice(3, 5), slice(5, 8), slice(8, 9)):
        e = float((got[:, sl].cpu().double() - ref[:, sl]).norm() / ref[:, sl].norm())
        assert e <= 1e-3, (sl, e)
    if arm == "SZ":
        assert abs(float(got[:, 9].double().sum()) - float(beta.grad)) <= 1e-3 * abs(float(beta.grad)) + 1e-5


def oracle_detached_z(P, H, W, arm, beta):
    Pz = torch.cat([P[:, :5], P[:, 5:6].detach(), P[:, 6:]], 1)
    return oracle(Pz, H, W, arm, beta)


@pytest.mark.parametrize("arm", ["A", "SZ", "RV"])
def test_backward_non_finite_image_gradient_reaches_every_gaussian(arm):
    H, W = 40, 40
    proj = records(300, H, W, seed=5).cuda()
    gi = torch.ones(H, W, 3, device="cuda")
    gi[3, 4, 1] = float("nan")
    got, _ = grads(proj, H, W, arm, gi)
    assert bool(torch.isnan(got[:, 8]).all()) and bool(torch.isnan(got[:, 0:5]).all())


@pytest.mark.parametrize("G,H,W,size", [(300, 50, 41, 4.0), (4200, 30, 50, 2.0)])
def test_backward_matches_the_general_path(G, H, W, size):
    """Boxes against the whole image (depth 1e19), thin gaussians included: the pairs outside the
    box add exact zeros, so only the order of the sums differs."""
    p = records(G, H, W, seed=9, cond=1e5, size=size).cuda()
    gi = torch.randn(H, W, 3, generator=torch.Generator().manual_seed(1)).cuda()
    bg = torch.tensor(BG, device="cuda")
    img, den = kernels.render_dense(p, H, W, 4.0, bg)
    a, _ = kernels.render_dense_bwd(p, H, W, 4.0, bg, img, den, gi)
    b, _ = kernels.render_dense_bwd(everywhere(p), H, W, 4.0, bg, img, den, gi)
    # H W terms in another order; they cancel in part, so against each column's largest gradient
    assert float(((a - b).abs() / b.abs().amax(0)).max()) <= H * W * 2.0 ** -24


def test_backward_softz_product_past_the_float_range():
    """o_col (Z/den0) (z - z*) has three factors: where it overflows, zero weights give NaN, as
    visiting every pair does, also for a gaussian whose support misses the image."""
    H, W = 24, 31
    proj = records(40, H, W, seed=2)
    proj[7, 0:2] = -400.0
    proj[7, 9] = 1e17
    beta = torch.tensor([1e-17], device="cuda")
    img, den, aux = kernels.render_dense_arm(proj.cuda(), H, W, 4.0,
                                             torch.tensor(BG, device="cuda"), "SZ", beta)
    aux[..., 0], aux[..., 1] = 1e17, 1e-30     # z*, den0: Z/den0 is about 1e13
    gi = torch.randn(H, W, 3, generator=torch.Generator().manual_seed(1)).cuda()
    got, _ = kernels.render_dense_arm_bwd(proj.cuda(), H, W, 4.0, torch.tensor(BG, device="cuda"),
                                          "SZ", img, den, aux, gi, beta)
    assert bool(torch.isnan(got[7, 0:5]).all())
