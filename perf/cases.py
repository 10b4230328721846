"""What this framework is used for, as timed cases.

Six kinds of work, each through an entry point that a program calls:

  train    ttsplat.step.TrainStep, captured once: one pass is `steps` training steps
  render   ttsplat.binned.render_binned_device without gradients: one frame
  binned   render_binned_device -> loss_fn -> gradients: one step of a torch training loop
  dense    ttsplat.render.render (arms A, B, SZ, RV), with or without loss and gradients
  wsr      ttsplat.backward.wsr_polysplat with its manual backward
  bins     ttsplat.binned.assign_bins

Scenes are seeded draws of the distributions of the repository's benchmark configurations
(uniform or clustered means, log-uniform scales, orbit cameras at distance 3, fov 50 degrees);
targets are smooth seeded images in [0, 1].
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "tt-splat_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

SH_C0 = 0.28209479177387814
K_POLY, NEAR, BLUR = 4.0, 0.2, 0.3
W_B_RAW = -3.0
LR, MEANS_LR = 1e-3, 1.6e-4
MCMC = dict(lambda_o=0.01, lambda_s=0.01, noise_lr=5e5, relocate_every=0, seed=0)


def listed():
    return [
        # The smallest training step in use: 2000 gaussians, 128x128, bf16 render, one step per
        # call.  Latency and launches.
        dict(name="train_2k_128_bf16", kind="train", G=2000, H=128, W=128, K=128, cams=2, steps=1,
             dtype="bf16", clustered=False),
        # An object-sized scene trained as the reference's trainer runs by default: bins rebuilt
        # every 5th step, runs of 8 steps.
        dict(name="train_10k_800", kind="train", G=10000, H=800, W=800, K=128, cams=4, steps=8,
             dtype="fp32", clustered=False, bin_every=5),
        # The benchmark's headline: 100k clustered gaussians at 1264x832, rebinned every step.
        dict(name="train_100k_1264x832", kind="train", G=100000, H=832, W=1264, K=128, cams=4,
             steps=8, dtype="fp32", clustered=True),
        # The same scene with view-dependent colour and MCMC regulariser and noise.
        dict(name="train_100k_sh3_mcmc", kind="train", G=100000, H=832, W=1264, K=128, cams=2,
             steps=1, dtype="fp32", clustered=True, sh_degree=3, mcmc=True),
        # The largest: a million gaussians at 1920x1072, K = 256, one update per 4 views.
        dict(name="train_1m_1920x1072_bf16", kind="train", G=1000000, H=1072, W=1920, K=256,
             cams=4, steps=1, dtype="bf16", clustered=True, batch=4),
        # One frame of a viewer.
        dict(name="render_100k_1264x832", kind="render", G=100000, H=832, W=1264, K=128,
             clustered=True),
        # A torch training loop's step on the binned render, odd counts.
        dict(name="binned_30k_640x480", kind="binned", G=30011, H=480, W=640, K=128,
             clustered=False),
        # The dense overfit loop's step (one view) at its own size.
        dict(name="dense_grad_2k_128", kind="dense", G=2000, H=128, W=128, arm="A", grad=True,
             sh_degree=0),
        # An occlusion arm on a ragged image, with view-dependent colour.
        dict(name="dense_grad_sz_3k_173x131", kind="dense", G=3001, H=131, W=173, arm="SZ",
             grad=True, sh_degree=2),
        # Dense evaluation of an object-sized scene.
        dict(name="dense_eval_10k_800", kind="dense", G=10000, H=800, W=800, arm="A", grad=False,
             sh_degree=0),
        # The explicit-basis op, forward and backward.
        dict(name="wsr_2k_128", kind="wsr", G=2000, H=128, W=128, keep=True),
        # Binning alone of a million means.
        dict(name="bins_1m_1920x1072", kind="bins", G=1000000, H=1072, W=1920, K=256,
             clustered=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above."""
    kind = rng.choice(["train", "train", "render", "binned", "dense", "dense", "wsr", "bins"])
    if kind == "wsr":
        return dict(kind="wsr", G=_log(rng, 100, 6000), H=_log(rng, 17, 200),
                    W=_log(rng, 17, 200), keep=rng.random() < 0.5)
    if kind == "dense":
        grad = rng.random() < 0.7
        return dict(kind="dense", G=_log(rng, 200, 10000), H=_log(rng, 24, 300 if grad else 800),
                    W=_log(rng, 24, 300 if grad else 800), arm=rng.choice(["A", "A", "B", "SZ", "RV"]),
                    grad=grad, sh_degree=rng.choice([0, 0, 1, 3]))
    case = dict(kind=kind, H=16 * _log(rng, 5, 60), W=16 * _log(rng, 5, 100),
                K=rng.choice([64, 128, 128, 256]), clustered=rng.random() < 0.5)
    if kind == "bins":
        return dict(case, G=_log(rng, 1000, 1000000))
    if kind == "render":
        return dict(case, G=_log(rng, 1000, 300000))
    if kind == "binned":
        return dict(case, G=_log(rng, 1000, 100000))
    case.update(G=_log(rng, 1000, 200000), cams=rng.choice([2, 3]), steps=rng.choice([1, 8]),
                dtype=rng.choice(["fp32", "fp32", "bf16"]))
    extra = rng.choice(["plain", "plain", "bin_every", "batch", "sh", "mcmc"])
    if extra == "bin_every":
        case["bin_every"] = rng.choice([2, 5])
    elif extra == "batch":
        case.update(batch=case["cams"], steps=1)
    elif extra == "sh":
        case["sh_degree"] = rng.choice([1, 2, 3])
    elif extra == "mcmc":
        case["mcmc"] = True
    return case


# ------------------------------------------------------------------------------ inputs --
def _params(case, seed):
    """[G,14] parameters on the CPU: means, quaternions, log-scales, SH-DC colour, opacity."""
    G, g = case["G"], torch.Generator("cpu").manual_seed(int(seed))
    if case.get("clustered"):
        centres = torch.rand(20, 3, generator=g) * 4.0 - 2.0
        means = centres[torch.randint(0, 20, (G,), generator=g)]
        means = means + 0.2 * torch.randn(G, 3, generator=g)
    else:
        means = torch.rand(G, 3, generator=g) * 2.0 - 1.0
    lo, hi = (0.002, 0.05) if G > 300000 else (0.01, 0.1)
    scales = math.log(lo) + torch.rand(G, 3, generator=g) * (math.log(hi) - math.log(lo))
    q = torch.randn(G, 4, generator=g)
    q = q / q.norm(dim=1, keepdim=True)
    o = 0.05 + 0.9 * torch.rand(G, 1, generator=g)
    dc = (torch.rand(G, 3, generator=g) - 0.5) / SH_C0
    return torch.cat([means, q, scales, dc, torch.log(o / (1.0 - o))], 1).contiguous()


def _rest(case, seed):
    g = torch.Generator("cpu").manual_seed(int(seed) + 7919)
    return 0.1 * torch.randn(case["G"], 15, 3, generator=g)


def _eyes(n, seed):
    g, eyes = torch.Generator("cpu").manual_seed(int(seed) + 104729), []
    while len(eyes) < n:
        v = torch.randn(3, generator=g)
        v = v / v.norm()
        if abs(float(v[1])) <= 0.95:
            eyes.append((3.0 * v).tolist())
    return eyes


def _target(case, seed):
    """A smooth image with a little texture, [H,W,3] in [0,1]."""
    H, W = case["H"], case["W"]
    g = torch.Generator("cpu").manual_seed(int(seed) + 15485863)
    low = torch.rand(1, 3, max(2, H // 32), max(2, W // 32), generator=g)
    img = F.interpolate(low, size=(H, W), mode="bilinear", align_corners=True)[0]
    img = (img.permute(1, 2, 0) + 0.03 * torch.randn(H, W, 3, generator=g)).clamp(0.0, 1.0)
    return img.contiguous().cuda()


def _cameras(case, seed):
    from ttsplat.camera import pinhole
    return [pinhole(case["H"], case["W"], e) for e in _eyes(case.get("cams", 1), seed)]


def _phi_theta(case, seed):
    """The explicit-basis op's operands: pixel monomials in image-centred coordinates, and the
    theta of projected gaussians over them (computed in 64 bits, kept in 32)."""
    H, W = case["H"], case["W"]
    P = _params(case, seed).double()
    pr = _project(P, _camera64(case, seed, 0, "cpu"))
    mx, my = pr["mu"][:, 0] - W / 2.0, pr["mu"][:, 1] - H / 2.0
    a, b, c = pr["conic"].unbind(1)
    ik = 1.0 / K_POLY
    theta = torch.stack([-a * ik, -c * ik, -2 * b * ik, 2 * (a * mx + b * my) * ik,
                         2 * (b * mx + c * my) * ik,
                         1 - (a * mx * mx + 2 * b * mx * my + c * my * my) * ik], 1)
    px = (torch.arange(W).double() + 0.5 - W / 2.0).repeat(H)
    py = (torch.arange(H).double() + 0.5 - H / 2.0).repeat_interleave(W)
    phi = torch.stack([px * px, py * py, px * py, px, py, torch.ones_like(px)], 1)
    g = torch.Generator("cpu").manual_seed(int(seed) + 32452843)
    keep = (torch.rand(case["G"], generator=g) > 0.1) if case["keep"] else None
    return dict(theta=theta.float(), phi=phi.float(), o=torch.sigmoid(P[:, 13]).float(),
                color=torch.rand(case["G"], 3, generator=g), keep=keep,
                gC=torch.randn(H * W, 3, generator=g) / (3.0 * H * W))


def _model(case, seed):
    from ttsplat.model import GaussianModel
    rest = _rest(case, seed).cuda() if case.get("sh_degree") else None
    model = GaussianModel(_params(case, seed).cuda(), w_b_raw=W_B_RAW, color_rest=rest)
    return model


def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        from ttsplat.step import TrainStep
        targets = [_target(case, seed + 31 * i) for i in range(case["cams"])]
        deg = case.get("sh_degree", 0)
        ts = TrainStep(_params(case, seed).cuda(), _cameras(case, seed), targets, K=case["K"],
                       w_b_raw=W_B_RAW, batch=case.get("batch", 1), dtype=case["dtype"],
                       sh_degree=deg, sh_rest=_rest(case, seed) if deg else None,
                       mcmc=dict(MCMC) if case.get("mcmc") else None,
                       bin_every=case.get("bin_every", 1))
        ts.capture()
        return dict(kind=kind, ts=ts, at=0, n=case["steps"])
    if kind == "wsr":
        s = {k: None if v is None else v.cuda() for k, v in _phi_theta(case, seed).items()}
        s.update(kind=kind, c_b=torch.ones(3, device="cuda"),
                 w_b=torch.tensor(0.05, device="cuda", requires_grad=True))
        for n in ("theta", "o", "color"):
            s[n].requires_grad_(True)
        return s
    from ttsplat import binned
    if kind == "bins":
        pr = _project(_params(case, seed).cuda().double(), _camera64(case, seed, 0, "cuda"))
        return dict(kind=kind, mu=pr["mu"].float().contiguous(), keep=pr["keep"], K=case["K"],
                    tmap=binned.TileMap(case["H"], case["W"]))
    model = _model(case, seed)
    s = dict(kind=kind, model=model, cam=_cameras(case, seed)[0])
    s["cam"].device_block("cuda")
    if kind in ("render", "binned"):
        s.update(tmap=binned.TileMap(case["H"], case["W"]), K=case["K"])
    if kind == "dense":
        s.update(arm=case["arm"], sh_degree=case["sh_degree"], grad=case["grad"])
    if kind == "binned" or case.get("grad"):
        s["target"] = _target(case, seed)
        leaves = [model.params]
        if case.get("arm") != "RV":        # revealage has no background weight
            leaves += [model.w_b_raw]
        if case.get("arm") == "B":
            leaves += [model.depth_beta, model.depth_tau]
        if case.get("arm") == "SZ":
            leaves += [model.softz_beta]
        if case.get("sh_degree"):
            leaves += [model.color_rest]
        s["leaves"] = [t.requires_grad_(True) for t in leaves]
    return s


def run(state):
    kind = state["kind"]
    if kind == "train":
        ts = state["ts"]
        if state["n"] == 1:
            ts.step(state["at"])
        else:
            ts.run(state["at"], state["n"])
        state["at"] = (state["at"] + state["n"]) % ts.n_steps
        out = dict(params=ts.P, m=ts.m, v=ts.v, image=ts.image)
        if ts.sh is not None:
            out["sh"] = ts.sh
        return out
    if kind == "wsr":
        from ttsplat.backward import wsr_polysplat
        leaves = [state["theta"], state["o"], state["color"], state["w_b"]]
        C = wsr_polysplat(*leaves, state["phi"], state["c_b"], state["keep"])
        return [C.detach(), *torch.autograd.grad(C, leaves, state["gC"])]
    from ttsplat import binned
    if kind == "bins":
        return list(binned.assign_bins(state["mu"], state["keep"], state["tmap"], 1, state["K"]))
    if kind == "render":
        with torch.no_grad():
            return binned.render_binned_device(state["model"], state["cam"], state["tmap"],
                                               K=state["K"])
    if kind == "binned":
        img = binned.render_binned_device(state["model"], state["cam"], state["tmap"],
                                          K=state["K"])
    else:
        from ttsplat.render import render
        if not state["grad"]:
            with torch.no_grad():
                return render(state["model"], state["cam"], state["arm"],
                              sh_degree=state["sh_degree"])
        img = render(state["model"], state["cam"], state["arm"], sh_degree=state["sh_degree"])
    from ttsplat.loss import loss_fn
    loss = loss_fn(img, state["target"], 0.2)
    return [img.detach(), loss.detach(), *torch.autograd.grad(loss, state["leaves"])]


# -------------------------------------------------------------------- what it cannot do without --
def _pairs(case):
    """(pixel, gaussian) pairs that carry weight, roughly: the support of a gaussian of the
    scene's mean scale at distance 3 is an ellipse of radius sqrt(k) sigma."""
    f = 0.5 * case["W"] / math.tan(math.radians(25.0))
    lo, hi = (0.002, 0.05) if case["G"] > 300000 else (0.01, 0.1)
    s2 = (hi * hi - lo * lo) / (2.0 * math.log(hi / lo))      # mean square of a log-uniform scale
    area = math.pi * K_POLY * (s2 * f * f / 9.0 + BLUR)
    return case["G"] * min(area, case["H"] * case["W"])


def work(case):
    G, P, kind = case["G"], case["H"] * case["W"], case["kind"]
    if kind == "wsr":   # every pixel and every gaussian of an arbitrary basis: 22 and 44 flop
        return dict(bytes=4 * (G * 20 + P * (6 + 3 + 3)), flops=(22 + 44) * G * P)
    if kind == "bins":
        T = P // 256
        return dict(bytes=9 * G + T * case["K"] * 9, flops=0)
    if kind == "dense":
        pairs = _pairs(case)
        sh = 180 * G if case["sh_degree"] else 0
        if not case["grad"]:
            return dict(bytes=56 * G + sh + 12 * P, flops=22 * pairs)
        return dict(bytes=112 * G + 2 * sh + (12 + 12) * P, flops=66 * pairs + 1056 * P)
    T = P // 256
    pairs = min(_pairs(case), 256.0 * T * case["K"])
    if kind == "render":
        return dict(bytes=56 * G + 12 * P, flops=22 * pairs)
    if kind == "binned":
        return dict(bytes=112 * G + 24 * P, flops=66 * pairs + 1056 * P)
    views = case["steps"] * case.get("batch", 1)
    state = (56 * 6 if not case.get("sh_degree") else (56 + 180) * 6) * G
    return dict(bytes=views * 12 * P + case["steps"] * state,
                flops=views * (66 * pairs + 1056 * P))


def tolerance(case):
    """Four times the largest distance from exact() over some sixty drawn cases."""
    kind = case["kind"]
    if kind == "bins":
        return "exact"
    if kind == "wsr":
        return {"rel": 1e-3}    # 2.4e-4 seen: theta's terms cancel in u
    if kind == "train":
        # 2.5e-2 seen with bf16 weights and colours in the render; 2.1e-4 in 32 bits, where one
        # mean on the edge of a quantised distance takes another slot
        return {"rel": 1e-1 if case["dtype"] == "bf16" else 1e-3}
    return {"rel": 8e-5}        # 2.1e-5 seen, in the gradients


# --------------------------------------------------------------------- plain torch, 64 bits --
def _camera64(case, seed, i, dev):
    """Camera i as (R, t, f, cx, cy) in 64 bits (its rotation rounded to 32 bits, as stored)."""
    eye = torch.tensor(_eyes(case.get("cams", 1), seed)[i])
    fwd = -eye / eye.norm()
    right = torch.linalg.cross(torch.tensor([0.0, 1.0, 0.0]), fwd)
    right = right / right.norm()
    R = torch.stack([right, torch.linalg.cross(fwd, right), fwd])
    t = -(R @ eye)
    f = 0.5 * case["W"] / math.tan(math.radians(50.0) / 2.0)
    return dict(R=R.double().to(dev), t=t.double().to(dev), f=float(torch.tensor(f)),
                cx=case["W"] / 2.0, cy=case["H"] / 2.0)


def _project(P, cam):
    q = P[:, 3:7] / P[:, 3:7].norm(dim=1, keepdim=True).clamp(min=1e-12)
    w, x, y, z = q.unbind(1)
    Rq = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                      2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                      2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)],
                     1).reshape(-1, 3, 3)
    M = cam["R"] @ (Rq * torch.exp(P[:, 7:10])[:, None, :])
    pc = P[:, 0:3] @ cam["R"].T + cam["t"]
    zc = pc[:, 2]
    zz = zc.clamp(min=NEAR)
    f, zero = cam["f"], torch.zeros_like(zz)
    mu = torch.stack([f * pc[:, 0] / zz + cam["cx"], f * pc[:, 1] / zz + cam["cy"]], 1)
    J = torch.stack([f / zz, zero, -f * pc[:, 0] / zz ** 2, zero, f / zz, -f * pc[:, 1] / zz ** 2],
                    1).reshape(-1, 2, 3)
    A = J @ M
    S = A @ A.transpose(1, 2)
    s00, s11, s01 = S[:, 0, 0] + BLUR, S[:, 1, 1] + BLUR, S[:, 0, 1]
    det = (s00 * s11 - s01 * s01).clamp(min=1e-12)
    return dict(mu=mu, conic=torch.stack([s11 / det, -s01 / det, s00 / det], 1), z=zc,
                keep=zc > NEAR)


def _colour(P, cam, rest, deg, through_direction):
    if not deg:
        return (0.5 + SH_C0 * P[:, 10:13]).clamp(min=0.0)
    d = P[:, 0:3] + cam["R"].T @ cam["t"]
    d = d if through_direction else d.detach()
    x, y, z = (d / d.norm(dim=1, keepdim=True)).unbind(1)
    b = [-0.4886025119029199 * y, 0.4886025119029199 * z, -0.4886025119029199 * x]
    if deg > 1:
        b += [1.0925484305920792 * x * y, -1.0925484305920792 * y * z,
              0.31539156525252005 * (2 * z * z - x * x - y * y), -1.0925484305920792 * x * z,
              0.5462742152960396 * (x * x - y * y)]
    if deg > 2:
        b += [-0.5900435899266435 * y * (3 * x * x - y * y), 2.890611442640554 * x * y * z,
              -0.4570457994644658 * y * (4 * z * z - x * x - y * y),
              0.3731763325901154 * z * (2 * z * z - 3 * x * x - 3 * y * y),
              -0.4570457994644658 * x * (4 * z * z - x * x - y * y),
              1.445305721320277 * z * (x * x - y * y),
              -0.5900435899266435 * x * (x * x - 3 * y * y)]
    b = torch.stack(b, 1)
    return (0.5 + SH_C0 * P[:, 10:13] + (b[:, :, None] * rest[:, :b.shape[1]]).sum(1)).clamp(min=0.0)


def _bins(mu, keep, H, W, K, span=2048):
    """idx[T,K], valid[T,K] by the binning rule: per 16x16 tile, the K smallest
    (clamped integer distance^2, stencil index, id) among the means of the 3x3 cells around it."""
    mu = mu.detach().float()
    nx, ny = W // 16, H // 16
    T, dev, G = nx * ny, mu.device, mu.shape[0]
    gx = (mu[:, 0] / 16.0).floor().long().clamp(0, nx - 1)
    gy = (mu[:, 1] / 16.0).floor().long().clamp(0, ny - 1)
    tiles, ids, q = [], [], []
    for dy in (-1, 0, 1):
        for dx in (-1, 0, 1):
            tx, ty = gx + dx, gy + dy
            g = (keep & (tx >= 0) & (tx < nx) & (ty >= 0) & (ty < ny)).nonzero()[:, 0]
            tx, ty = tx[g], ty[g]
            ex = mu[g, 0] - (tx.float() + 0.5) * 16.0
            ey = mu[g, 1] - (ty.float() + 0.5) * 16.0
            xx, yy = ex * ex, ey * ey
            tiles.append(ty * nx + tx)
            ids.append(g)
            q.append((xx + yy).double().clamp(0, span - 1).long())
    tiles, ids, q = torch.cat(tiles), torch.cat(ids), torch.cat(q)
    order = torch.sort(tiles * span + q, stable=True).indices
    tiles, ids = tiles[order], ids[order]
    starts = torch.searchsorted(tiles, torch.arange(T, device=dev))
    rank = torch.arange(tiles.numel(), device=dev) - starts[tiles]
    kept = rank < K
    idx = torch.zeros(T * K, dtype=torch.long, device=dev)
    valid = torch.zeros(T * K, dtype=torch.bool, device=dev)
    at = tiles[kept] * K + rank[kept]
    idx[at] = ids[kept]
    valid[at] = True
    return idx.view(T, K), valid.view(T, K)


def _ssim_loss(x, y, lam=0.2):
    g = torch.arange(11, dtype=torch.float64, device=x.device) - 5
    g = torch.exp(-g * g / (2 * 1.5 * 1.5))
    g = g / g.sum()

    def filt(a):
        n, m = a.shape[0] - 10, a.shape[1] - 10
        a = sum(g[i] * a[i:i + n] for i in range(11))
        return sum(g[i] * a[:, i:i + m] for i in range(11))

    l1 = (x - y).abs().mean()
    x, y = x.clamp(0, 1), y.clamp(0, 1)
    fx, fy = filt(x), filt(y)
    sx, sy, sxy = filt(x * x) - fx * fx, filt(y * y) - fy * fy, filt(x * y) - fx * fy
    s = ((2 * fx * fy + 1e-4) * (2 * sxy + 9e-4)) / ((fx * fx + fy * fy + 1e-4) * (sx + sy + 9e-4))
    return (1 - lam) * l1 + lam * (1 - s.mean())


def _blend(case, pr, colour, o, w_b, extra, px, py, at):
    """Colours of the pixels px, py [n, p] blended over the gaussians at [n, K]; o carries each
    listed gaussian's weight (0 where a slot is empty)."""
    mu, con, z = pr["mu"][at], pr["conic"][at], pr["z"].detach()[at][:, None]
    dx, dy = px[:, :, None] - mu[:, None, :, 0], py[:, :, None] - mu[:, None, :, 1]
    Q = con[:, None, :, 0] * dx * dx + 2 * con[:, None, :, 1] * dx * dy + con[:, None, :, 2] * dy * dy
    w = o[:, None] * (1.0 - Q / K_POLY).clamp(min=0.0) ** 2
    arm = case.get("arm", "A")
    if arm == "SZ":
        zs = (w * z).sum(2, keepdim=True) / (w.sum(2, keepdim=True) + 1e-6)
        w = w * torch.sigmoid(-extra["softz_beta"] * (z - zs))
    num = torch.matmul(w, colour)
    den = w.sum(2, keepdim=True)
    if arm == "RV":
        R = torch.exp(torch.log1p(-w.clamp(0.0, 1.0 - 1e-4)).sum(2, keepdim=True))
        return num / (den + 1e-6) * (1.0 - R) + R
    return (num + w_b) / (den + w_b)


def _image64(case, leaves, cam, want):
    """The image in 64 bits; with `want`, a function of the image whose gradients with respect
    to the leaves come back too: (image, value, gradients)."""
    H, W, dev = case["H"], case["W"], leaves["P"].device

    def operands():
        P = leaves["P"]
        pr = _project(P, cam)
        dense = case["kind"] == "dense"
        col = _colour(P, cam, leaves.get("rest"), case.get("sh_degree", 0), dense)
        o = pr["keep"].double() * torch.sigmoid(P[:, 13])
        if case.get("arm") == "B":
            o = o * torch.sigmoid(leaves["depth_beta"] * (leaves["depth_tau"] - pr["z"]))
        return pr, col, o, F.softplus(leaves["w_b_raw"])

    with torch.no_grad():
        pr = operands()[0]
        if case["kind"] == "dense":
            S, T = 1, H * W
            idx = torch.arange(case["G"], device=dev)[None]
            valid, nx = torch.ones_like(idx, dtype=torch.bool), W
        else:
            S, nx, T = 16, W // 16, (H // 16) * (W // 16)
            idx, valid = leaves.get("bins") or _bins(pr["mu"], pr["keep"], H, W, case["K"])
    sub = torch.arange(S * S, device=dev)
    step = max(1, int(1.5e8) // (idx.shape[1] * S * S))
    chunks = [torch.arange(i, min(i + step, T), device=dev) for i in range(0, T, step)]

    def pixels(t):
        px = (t % nx * S)[:, None] + (sub % S)[None]
        py = (t // nx * S)[:, None] + (sub // S)[None]
        return py * W + px, px.double() + 0.5, py.double() + 0.5

    def part(ops, t):
        pr, col, o, w_b = ops
        at, px, py = pixels(t)
        if S == 1:   # dense: all pixels of the chunk over all gaussians
            return at, _blend(case, pr, col, o[None], w_b, leaves, px.T, py.T, idx).reshape(-1, 3)
        oo = o[idx[t]] * valid[t].double()
        return at, _blend(case, pr, col[idx[t]], oo, w_b, leaves, px, py, idx[t]).reshape(-1, 3)

    with torch.no_grad():
        ops, img = operands(), torch.zeros(H * W, 3, dtype=torch.float64, device=dev)
        for t in chunks:
            at, c = part(ops, t)
            img[at.reshape(-1)] = c
    img = img.view(H, W, 3)
    if want is None:
        return img
    x = img.clone().requires_grad_(True)
    value = want(x)
    gimg = torch.autograd.grad(value, x)[0].reshape(-1, 3)
    ops = operands()
    cut = [{k: v.detach().requires_grad_(v.requires_grad) for k, v in ops[0].items()},
           *[v.detach().requires_grad_(True) for v in ops[1:]]]
    beta = [leaves["softz_beta"]] if case.get("arm") == "SZ" else []
    inner = [cut[0]["mu"], cut[0]["conic"], *cut[1:], *beta]
    total = [torch.zeros_like(v) for v in inner]
    for t in chunks:
        at, c = part(cut, t)
        for s, g in zip(total, torch.autograd.grad(c, inner, gimg[at.reshape(-1)],
                                                   allow_unused=True)):
            if g is not None:
                s += g
    outer = [ops[0]["mu"], ops[0]["conic"], *ops[1:]]
    names = [n for n in ("P", "w_b_raw", "depth_beta", "depth_tau", "rest") if n in leaves]
    got = dict(zip(names, torch.autograd.grad(outer, [leaves[n] for n in names], total[:5],
                                              allow_unused=True)))
    if beta:
        got["softz_beta"] = total[5]
    return img, value.detach(), got


def _leaves64(case, seed):
    d = dict(P=_params(case, seed), w_b_raw=torch.tensor(W_B_RAW))
    if case.get("arm") == "B":
        d.update(depth_beta=torch.tensor(1.0), depth_tau=torch.tensor(3.0))
    if case.get("arm") == "SZ":
        d["softz_beta"] = torch.tensor(4.0)
    if case.get("sh_degree"):
        d["rest"] = _rest(case, seed)
    return {k: v.double().cuda().requires_grad_(True) for k, v in d.items()}


def exact(case, seed):
    kind, H, W = case["kind"], case["H"], case["W"]
    if kind == "bins":
        pr = _project(_params(case, seed).cuda().double(), _camera64(case, seed, 0, "cuda"))
        return list(_bins(pr["mu"].float(), pr["keep"], H, W, case["K"]))
    if kind == "wsr":
        s = {k: None if v is None else v.cuda().double() for k, v in _phi_theta(case, seed).items()}
        leaves = [s["theta"], s["o"], s["color"], torch.tensor(0.05, dtype=torch.float64).cuda()]
        leaves = [t.requires_grad_(True) for t in leaves]
        th, o, col, w_b = leaves
        w = o[None] * (s["phi"] @ th.T).clamp(min=0.0) ** 2
        if s["keep"] is not None:
            w = w * s["keep"][None]
        C = (w @ col + w_b) / (w.sum(1, keepdim=True) + w_b)
        return [C.detach(), *torch.autograd.grad(C, leaves, s["gC"])]
    if kind == "train":
        if case.get("mcmc") or case["G"] * case["steps"] * case.get("batch", 1) > 1000000:
            return None    # random noise, or too long
        return _train64(case, seed)
    leaves, cam = _leaves64(case, seed), _camera64(case, seed, 0, "cuda")
    if kind == "render" or not case.get("grad", True):
        return _image64(case, leaves, cam, None)
    y = _target(case, seed).double()
    img, loss, g = _image64(case, leaves, cam, lambda x: _ssim_loss(x, y))
    names = [n for n in ("P", "w_b_raw", "depth_beta", "depth_tau", "softz_beta", "rest")
             if n in leaves and not (n == "w_b_raw" and case.get("arm") == "RV")]
    return [img, loss, *[g[n] for n in names]]


def _train64(case, seed):
    leaves, B = _leaves64(case, seed), case.get("batch", 1)
    n_steps, every = case["cams"] // B, case.get("bin_every", 1)
    lr = torch.full((14,), LR, dtype=torch.float64, device="cuda")
    lr[0:3] = MEANS_LR
    names = ["P"] + (["rest"] if "rest" in leaves else [])
    rate = dict(P=lr, rest=LR / 20.0)
    m = {n: torch.zeros_like(leaves[n]) for n in names}
    v = {n: torch.zeros_like(leaves[n]) for n in names}
    ys = [_target(case, seed + 31 * i).double() for i in range(case["cams"])]
    for it in range(case["steps"]):
        g = {n: 0.0 for n in names}
        for b in range(B):
            ci = (it % n_steps) * B + b
            cam = _camera64(case, seed, ci, "cuda")
            if it % every == 0:
                leaves.pop("bins", None)
                with torch.no_grad():
                    pr = _project(leaves["P"], cam)
                bins = _bins(pr["mu"], pr["keep"], case["H"], case["W"], case["K"])
            img, _, got = _image64(case, dict(leaves, bins=bins), cam,
                                   lambda x: _ssim_loss(x, ys[ci]))
            g = {n: g[n] + got[n] / B for n in names}
        t = it + 1
        for n in names:
            m[n] = 0.9 * m[n] + 0.1 * g[n]
            v[n] = 0.999 * v[n] + 0.001 * g[n] ** 2
            up = rate[n] * (m[n] / (1 - 0.9 ** t)) / ((v[n] / (1 - 0.999 ** t)).sqrt() + 1e-8)
            leaves[n] = (leaves[n].detach() - up).requires_grad_(True)
    out = dict(params=leaves["P"].detach(), m=m["P"], v=v["P"], image=img)
    if "rest" in leaves:
        out["sh"] = leaves["rest"].detach().permute(1, 2, 0).contiguous()
    return out
