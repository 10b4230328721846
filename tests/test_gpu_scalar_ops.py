"""The loss value, the background block and the target statistics against their formulas."""
import pytest
import torch
import torch.nn.functional as F

from ttsplat import kernels
from ttsplat.binned import _raw_background
from ttsplat.loss import loss_fn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W", [(11, 11), (27, 75), (400, 640), (2000, 1100)])
@pytest.mark.parametrize("lam", [0.2, 0.0, 1.0])
def test_loss_value(H, W, lam):
    n, ns = kernels.loss_partials_count(H, W)
    p = torch.rand(n, generator=torch.Generator().manual_seed(H)) * 2560
    s, l1 = p[:ns].double().sum(), p[ns:].double().sum()
    ref = (1 - lam) * l1 / (3.0 * H * W) + lam * (1 - s / (3.0 * (H - 10) * (W - 10)))
    got = kernels.loss_from_partials(p.cuda(), H, W, lam)
    assert got.shape == () and got.dtype == torch.float32
    # 64-bit sums rounded once
    assert abs(float(got) - float(ref)) <= 2.0 ** -23 * abs(float(ref)) + 1e-12
    assert abs(float(kernels.loss_from_partials(p, H, W, lam)) - float(ref)) <= 1e-6 * abs(float(ref)) + 1e-12


@pytest.mark.parametrize("raw", [-90.0, -3.0, 0.0, 15.0, 20.0, 20.5, 300.0, float("nan")])
@pytest.mark.parametrize("n", [1, 63, 257, 8040])
def test_background_block_and_gradient(raw, n):
    w = torch.tensor(raw, requires_grad=True)
    ref = F.softplus(w)
    c = torch.tensor([0.1, 0.7, 1.0])
    bg = kernels.background(w.detach().cuda(), c.cuda())
    assert torch.equal(bg[1:].cpu(), c)
    # one exp and one log1p, a few ulp each
    assert torch.allclose(bg[0].cpu(), ref.detach(), rtol=1e-6, atol=1e-44, equal_nan=True)
    gwb = torch.randn(n, generator=torch.Generator().manual_seed(n))
    (gr,) = torch.autograd.grad(ref, w, gwb.double().sum().float())
    g = kernels.background_grad(gwb.cuda(), w.detach().cuda())
    assert g.shape == w.shape
    assert torch.allclose(g.cpu(), gr, rtol=1e-6, atol=1e-44, equal_nan=True)


def test_background_of_other_model_forms():
    """Numbers, CPU tensors, other types and shapes convert, and gradients flow back through."""
    class M:
        pass
    for w, c in ((-3.0, (1.0, 1.0, 1.0)), (torch.tensor([-2.0], dtype=torch.float64), torch.ones(3, 1)),
                 (torch.tensor([[0.5]]).cuda(), torch.ones(1, 3, dtype=torch.float64))):
        m = M()
        m.w_b_raw, m.c_b = w, c
        a, b = _raw_background(m, torch.device("cuda"))
        bg = kernels.background(a, b.contiguous())
        assert torch.allclose(bg[0].cpu(), F.softplus(torch.as_tensor(w).float()).reshape(()).cpu(), rtol=1e-6)


@pytest.mark.parametrize("H,W", [(11, 11), (12, 84), (26, 74), (27, 75), (43, 139), (131, 173)])
def test_target_statistics_and_planar_copy(H, W):
    """Tiles of 64 x 16 map pixels: one tile, exact multiples, one pixel over, ragged."""
    g = torch.Generator().manual_seed(W)
    y = torch.rand(H, W, 3, generator=g) * 1.4 - 0.2          # the clamp is in use
    st = kernels.loss_stats(y.cuda()).cpu()
    n = (H - 10) * (W - 10)
    planar = st[6 * n:].view(3, H, W)
    assert torch.equal(planar, y.permute(2, 0, 1))
    c = torch.arange(11).double() - 5
    t = torch.exp(-c * c / 4.5)
    k = torch.outer(t, t)[None, None] / t.sum() ** 2
    yy = y.double().clamp(0, 1).permute(2, 0, 1)[:, None]
    mu, e2 = F.conv2d(yy, k)[:, 0], F.conv2d(yy * yy, k)[:, 0]
    got = st[:6 * n].view(2, 3, W - 10, H - 10).transpose(2, 3).double()
    # 22 fp32 products and sums of values in [0, 1]
    assert float((got[0] - mu).abs().max()) <= 3e-6
    assert float((got[1] - (e2 - mu * mu)).abs().max()) <= 3e-6


def test_loss_fn_value_and_gradient_scale():
    g = torch.Generator().manual_seed(1)
    x = torch.rand(40, 50, 3, generator=g).cuda().requires_grad_(True)
    y = torch.rand(40, 50, 3, generator=g).cuda()
    loss = loss_fn(x, y)
    (g1,) = torch.autograd.grad(loss, x, retain_graph=True)
    (g2,) = torch.autograd.grad(loss * 3.0, x)
    assert torch.allclose(3.0 * g1, g2, rtol=1e-6)


@pytest.mark.parametrize("G", [0, 1, 255, 256, 257, 1000])
def test_geometry_launches_carry_the_background(G):
    """geom_fwd writes the block background() makes; geom_bwd writes background_grad's result, takes
    rows of 10 and slot gradients through the inverse table."""
    from helpers import config_inputs
    _, P, cam = config_inputs("c1_ref", G=max(G, 1))
    P, camb = P[:G].cuda(), cam.device_block("cuda")
    w, c = torch.tensor(-1.5).cuda(), torch.tensor([0.2, 0.4, 0.9]).cuda()
    bg = torch.full((4,), -1.0, device="cuda")
    proj, keep = kernels.geom_fwd(P, camb, background=(w, c, bg))
    assert torch.equal(bg, kernels.background(w, c))
    if G == 0:
        return
    assert torch.equal(proj, kernels.geom_fwd(P, camb)[0])
    g = torch.Generator().manual_seed(G)
    gwb = torch.randn(77, generator=g).cuda()
    g10 = torch.randn(G, 10, generator=g).cuda()
    want = kernels.geom_bwd(P, camb, g10[:, :9].contiguous())
    gw = torch.empty_like(w)
    assert torch.equal(kernels.geom_bwd(P, camb, g10, background=(gwb, w, gw)), want)
    assert torch.equal(gw, kernels.background_grad(gwb, w))
    gslot = torch.randn(8, 16, 9, generator=g).cuda()
    inv = torch.randint(-1, 128, (G, 9), generator=g, dtype=torch.int32).cuda()
    ref = kernels.geom_bwd(P, camb, kernels.slot_reduce(gslot, inv))
    got = kernels.geom_bwd(P, camb, gslot, inv=inv)
    # the same sum and formulas, contracted by the compiler per kernel
    assert torch.allclose(got, ref, rtol=1e-4, atol=1e-5 * float(ref.abs().max()))


def test_loss_value_of_a_tensor_weight_and_of_tracked_partials():
    H, W = 40, 50
    p = torch.rand(kernels.loss_partials_count(H, W)[0], device="cuda", requires_grad=True)
    lam = torch.tensor([0.0, 0.2, 1.0], device="cuda", requires_grad=True)
    v = kernels.loss_from_partials(p, H, W, lam)
    one = [kernels.loss_from_partials(p.detach(), H, W, float(x)) for x in lam.detach()]
    assert torch.allclose(v.detach(), torch.stack(one), rtol=1e-6)   # the weight in 32 bits
    gp, gl = torch.autograd.grad(v.sum(), [p, lam])
    assert bool((gp != 0).any()) and gl.shape == (3,)
