"""The loss kernel's tile heights (8, 16, 24 and 40 rows, by the image's size) against the 64-bit
loss: one tile, ragged edges, and sizes that take each height."""
import pytest
import torch

from oracle import loss as oloss
from ttsplat import kernels

pytestmark = pytest.mark.gpu

# blocks of 40 / 24 / 16 / 8 rows per CU decide: the last four sizes take 16, 24, 40 and 24 rows
@pytest.mark.parametrize("H,W", [(11, 11), (12, 74), (18, 75), (19, 139), (97, 65), (160, 320),
                                 (305, 470), (250, 390), (401, 385), (590, 770)])
def test_loss_and_gradient(H, W):
    print(f"[loss] {H}x{W}", flush=True)
    g = torch.Generator().manual_seed(H)
    x = torch.rand(H, W, 3, generator=g) * 1.2 - 0.1          # the clamp's gate is in use
    y = torch.rand(H, W, 3, generator=g)
    part = torch.empty(kernels.loss_partials_count(H, W)[0], device="cuda")
    got = kernels.loss_grad(x.cuda(), y.cuda(), 0.2, partials=part).cpu().double()
    xr = x.double().requires_grad_(True)
    ref = oloss.loss_fn(xr, y.double())
    ref.backward()
    # the contract of the loss: value 1e-5, gradient 1e-4 relative L2
    assert abs(float(kernels.loss_from_partials(part, H, W, 0.2)) - float(ref.detach())) <= 1e-5
    assert float((got - xr.grad).norm()) <= 1e-4 * float(xr.grad.norm())
    # every pixel, not only their sum: largest difference against the largest gradient
    assert float((got - xr.grad).abs().max()) <= 1e-3 * float(xr.grad.abs().max())


def test_heights_taken():
    """The rows a size takes, from its block count (3 channels, 64-column tiles)."""
    def rows(H, W):
        n = kernels.loss_partials_count(H, W)[1] // (3 * ((W + 63) // 64))
        return [r for r in (8, 16, 24, 40) if (H + r - 1) // r == n]
    for (H, W), r in (((128, 128), 8), ((320, 480), 16), ((250, 390), 24), ((401, 385), 40),
                      ((600, 800), 24), ((832, 1264), 40)):
        assert r in rows(H, W), (H, W, rows(H, W))
