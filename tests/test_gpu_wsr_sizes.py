"""wsr_dense and its backward at the edges of their blocks: 64 and 256 pixels, 1024 staged
gaussians or pixels, 16 waves with nothing to do, bands, keep flags of each type."""
import pytest
import torch

from ttsplat import backward, kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G,P,keep", [(1, 1, None), (1, 65, "bool"), (15, 64, "float"),
                                      (63, 1023, "u8"), (64, 1025, None), (65, 129, "bool"),
                                      (1023, 63, "bool"), (1025, 300, None), (2100, 257, "u8"),
                                      (5, 32769, "bool"), (130, 33000, None), (3000, 2049, None),
                                      (32, 32767, "u8"), (33, 255, "bool"), (100, 32771, "bool"),
                                      (101, 32833, None), (300, 33023, "u8"), (301, 32769, None),
                                      (257, 1, "bool")])
def test_wsr_follows_the_formula(G, P, keep):
    print(f"[wsr] {G} {P} {keep}", flush=True)
    g = torch.Generator().manual_seed(G * 7 + P)
    th = torch.randn(G, 6, generator=g) * 0.4
    phi = torch.randn(P, 6, generator=g)
    o, col = torch.rand(G, generator=g) + 0.05, torch.rand(G, 3, generator=g)
    kp = torch.rand(G, generator=g) > 0.3
    k = {None: None, "bool": kp, "float": kp.float(), "u8": kp.to(torch.uint8)}[keep]
    R = torch.randn(P, 3, generator=g)
    wb, cb = 0.3, torch.tensor([0.9, 0.5, 0.2])

    dev = [t.cuda().requires_grad_(True) for t in (th, o, col, torch.tensor(wb))]
    C = backward.wsr_polysplat(*dev, phi.cuda(), cb.cuda(), None if k is None else k.cuda())
    got = torch.autograd.grad((C * R.cuda()).sum(), dev)

    ref = [t.double().requires_grad_(True) for t in (th, o, col, torch.tensor(wb))]
    Cr = backward_formula(ref, phi.double(), cb.double(), None if k is None else kp.double())
    want = torch.autograd.grad((Cr * R.double()).sum(), ref)
    # u: 6 products; the image a ratio of sums of non-negative terms
    assert float((C.detach().cpu() - Cr.detach()).abs().max()) <= 1e-4
    for a, b in zip(got, want):
        assert float((a.cpu().double() - b).norm()) <= 1e-3 * float(b.norm()) + 1e-5


def backward_formula(leaves, phi, cb, keep):
    th, o, col, wb = leaves
    w = (phi @ th.T).clamp(min=0) ** 2 * o
    if keep is not None:
        w = w * keep
    return (w @ col + wb * cb) / (w.sum(1, keepdim=True) + wb)


def test_wsr_is_deterministic_and_gradients_sum_over_bands():
    g = torch.Generator().manual_seed(3)
    th, phi = torch.randn(70, 6, generator=g).cuda(), torch.randn(5000, 6, generator=g).cuda()
    o, col = torch.rand(70, generator=g).cuda(), torch.rand(70, 3, generator=g).cuda()
    bg = torch.tensor([0.3, 1.0, 1.0, 1.0], device="cuda")
    gC = torch.randn(5000, 3, generator=g).cuda()
    C, den = kernels.wsr_dense(th, o, col, None, phi, bg)
    a = kernels.wsr_dense_bwd(th, o, col, None, phi, bg, C, den, gC)
    b = kernels.wsr_dense_bwd(th, o, col, None, phi, bg, C, den, gC)
    assert all(torch.equal(x, y) for x, y in zip(a, b))


def test_wsr_bands_of_many_gaussians():
    """Bands past one round of blocks (G 20000: 313 blocks a band, 8 bands of uneven length)."""
    g = torch.Generator().manual_seed(5)
    G, P = 20000, 9001
    leaves = [t.cuda() for t in (torch.randn(G, 6, generator=g) * 0.2, torch.rand(G, generator=g),
                                 torch.rand(G, 3, generator=g), torch.tensor(0.3))]
    phi, cb = torch.randn(P, 6, generator=g).cuda(), torch.tensor([0.9, 0.5, 0.2]).cuda()
    R = torch.randn(P, 3, generator=g).cuda()
    dev = [t.requires_grad_(True) for t in leaves]
    got = torch.autograd.grad((backward.wsr_polysplat(*dev, phi, cb) * R).sum(), dev)
    ref = [t.detach().double().requires_grad_(True) for t in leaves]
    C = backward_formula(ref, phi.double(), cb.double(), None)
    for a, b in zip(got, torch.autograd.grad((C * R.double()).sum(), ref)):
        assert float((a.double() - b).norm()) <= 1e-3 * float(b.norm()) + 1e-5
