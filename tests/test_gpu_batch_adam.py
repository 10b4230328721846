"""geom_bwd_adam_acc (a batch's last view and its Adam update in one launch) against
geom_bwd_accum + adam + zero_, at the edges of its 64-row blocks."""
import pytest
import torch

from helpers import config_inputs
from ttsplat import kernels
from ttsplat.step import lr_vector

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G", [1, 63, 64, 65, 1000])
def test_last_view_with_adam(G):
    _, P, cam = config_inputs("c1_ref", G=G)
    camb = cam.device_block("cuda")
    g = torch.Generator().manual_seed(G)
    T, K = 64, 32
    gslot = torch.randn(T, K, 9, generator=g).cuda()
    inv = torch.randint(-1, T * K, (G, 9), generator=g, dtype=torch.int32).cuda()
    out = []
    for fused in (False, True):
        p = P.cuda()
        gen = torch.Generator().manual_seed(5)
        m, v = (torch.rand(G, 14, generator=gen).cuda() * s for s in (1e-2, 1e-4))
        gacc = torch.randn(G, 14, generator=gen).cuda()
        step = kernels.adam_state("cuda")
        kernels.adam_advance(step)
        lr = lr_vector(device="cuda")
        if fused:
            kernels.geom_bwd_adam_acc(p, camb, gslot, inv, gacc, 0.25, m, v, lr, step)
        else:
            kernels.geom_bwd_accum(p, camb, gslot, inv, gacc, 0.25)
            kernels.adam(p, m, v, gacc, lr, step)
            kernels.zero_(gacc)
        assert float(gacc.abs().max()) == 0.0
        out.append((p, m, v))
    for a, b in zip(*out):
        # the same formulas, contracted by the compiler per kernel: one or two ulp of a sum
        assert torch.allclose(a, b, rtol=2e-5, atol=1e-7)
