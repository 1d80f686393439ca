"""What the trainer is used for, as cases that can be timed: training steps over
the range of scenes and options, and the calls a program makes between them.

A training case is one turn of a session's loop: a few steps enqueued
(`stepOnce`, or `stepViews` for batches of views), then the loss read, which
waits for them. The updated Gaussians stay on the GPU, as in a training loop;
they are read back when somebody looks at them (`_Answer`). The other cases
are the calls that hand something to the host: a rendered view, the PSNR of
held-out views, the Gaussians for a checkpoint.

Scenes: means uniform in a box, log-scales normal, random rotations, opacity
logits N(0, 1), cameras on a ring that look at the centre, the focal length
1100/1600 of the width. Targets are smooth images with noise and an invalid
border, as undistorted photographs have.

`exact` is the same step in float64 by plain torch: projection, compositing
by tiles, the loss, its gradient by autograd and Adam.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "splat.js_amd", "py"))

import gsabi  # noqa: E402
import scenes  # noqa: E402

PRECISIONS = {"f32": gsabi.GS_PREC_F32, "mixed": gsabi.GS_PREC_MIXED, "bf16": gsabi.GS_PREC_BF16,
              "fp16": gsabi.GS_PREC_FP16}
BASE = {"kind": "train", "n": 20000, "w": 320, "h": 240, "cams": 1, "uneven": False, "deg": 2, "prec": "f32",
        "ssim": False, "camopt": False, "accum_f32": False, "views": 1, "steps": 8, "ls_mu": -4.0, "ls_sd": 0.5,
        "box": 5.0, "ring": 8.0, "keys": 0}
ITER = 5000       # past the ramp of one SH band per 1000 iterations: all bands train
POS_LR = 1.6e-4


def _case(name=None, **kw):
    c = dict(BASE, **kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the gradient-check rig's size: what a step costs when there is next to nothing to compute
        _case("rig_160", n=160, w=64, h=64, deg=0, steps=4, box=1.2, ring=3.0, ls_mu=-2.6),
        # a first preview: 20k Gaussians, 320x240, under the L1 + D-SSIM loss
        _case("preview_20k_ssim", n=20000, w=320, h=240, ssim=True, steps=8, box=1.0, ring=3.0),
        # a phone capture while its poses and exposures are refined: ragged sizes, SH degree 3, 16-bit storage
        _case("phone_123k_camopt", n=123457, w=737, h=411, cams=8, deg=3, prec="mixed", camopt=True, steps=8),
        # the default capacity, a ragged view, the L1 + D-SSIM loss
        _case("photo_600k_ssim", n=600000, w=1237, h=933, cams=4, prec="bf16", ssim=True, steps=4),
        # the plain FP32 step at the benchmark's size
        _case("train_1m_f32", n=1000000, w=1600, h=900, cams=8, steps=8),
        # the batched step at the benchmark's size: 8 views, 16-bit storage
        _case("train_1m_bf16_8views", n=1000000, w=1600, h=900, cams=16, prec="bf16", views=8, steps=2),
        # a batch over photographs of different sizes
        _case("uneven_400k_fp16_5views", n=400003, w=1920, h=1080, cams=5, uneven=True, prec="fp16", views=5, steps=2),
        # large splats: every tile holds thousands of keys (early training, close views)
        _case("stress_1m_2views", n=1000000, w=1920, h=1080, cams=4, deg=3, views=2, steps=2, ls_mu=-3.0, ls_sd=1.0,
              keys=120000000),
        # a viewer's frame
        _case("view_1m_1080p", kind="render", n=1000000, w=1920, h=1080, prec="bf16"),
        # held-out views scored between training stretches
        _case("eval_250k", kind="eval", n=250000, w=979, h=546, cams=4),
        # large splats scored as they start, before training shrinks them: some 90M keys a view
        _case("eval_stress_1m", kind="eval", n=1000000, w=1920, h=1080, cams=2, deg=3, ls_mu=-3.0, ls_sd=1.0,
              keys=120000000),
        # a checkpoint
        _case("checkpoint_300k", kind="checkpoint", n=300000, deg=3),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["train"] * 6 + ["render", "eval", "checkpoint"])
    w = log(64, 1920)
    c = {"kind": kind, "n": log(160, 1100000), "w": w, "h": max(48, min(1080, int(w * rng.uniform(0.5, 0.8)))),
         "cams": rng.randint(1, 6), "deg": rng.choice([0, 1, 2, 2, 3]),
         "prec": rng.choice(["f32", "f32", "mixed", "bf16", "fp16"])}
    if c["n"] < 5000:
        c.update(box=1.2, ring=3.0, ls_mu=-2.8)
    if kind == "train":
        c["steps"] = rng.randint(1, 6)
        form = rng.choice(["single", "single", "ssim", "camopt", "views", "views", "large"])
        if form == "ssim":
            c["ssim"] = True
        elif form == "camopt":
            c["camopt"] = True
        elif form == "views":
            c.update(views=rng.randint(2, 8), cams=8, uneven=rng.random() < 0.5, steps=rng.randint(1, 2))
        elif form == "large":
            c.update(n=log(20000, 400000), ls_mu=-3.0, ls_sd=1.0, box=5.0, ring=8.0, keys=60000000, steps=2)
    return _case(**c)


# ---- inputs ----

def _sizes(c):
    """Width and height of each camera's image; uneven: from half the size up to it."""
    out = []
    for k in range(c["cams"]):
        s = 0.5 + 0.5 * k / max(1, c["cams"] - 1) if c["uneven"] else 1.0
        out.append((max(16, int(c["w"] * s)), max(16, int(c["h"] * s))))
    return out


def _cameras(c):
    cams = scenes.ring_cameras(c["cams"], c["ring"], c["w"], c["h"], 0.0)
    for k, (cam, (w, h)) in enumerate(zip(cams, _sizes(c))):
        cam.update(imgIdx=k, f=1100.0 / 1600.0 * w, cx=w / 2, cy=h / 2, w=w, h=h)
    return cams


def _inputs(c, seed):
    """(params n x 16, sh n x 3K or None, cameras, one h x w x 3 target per camera), tensors on the GPU."""
    g = torch.Generator("cuda").manual_seed(seed)
    n, K = c["n"], scenes.sh_k(c["deg"])

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    def uniform(*shape):
        return torch.rand(*shape, generator=g, device="cuda")

    p = torch.zeros(n, 16, device="cuda")
    p[:, 0:3] = (2 * uniform(n, 3) - 1) * c["box"]
    p[:, 3:6] = c["ls_mu"] + c["ls_sd"] * normal(n, 3)
    q = normal(n, 4)
    p[:, 6:10] = q / q.norm(dim=1, keepdim=True).clamp_min(1e-6)
    p[:, 10:13] = torch.logit(uniform(n, 3), eps=1e-3)
    p[:, 13] = normal(n)
    sh = 0.05 * normal(n, 3 * K) if K else None
    images = []
    for w, h in _sizes(c):
        y, x = torch.meshgrid(torch.arange(h, device="cuda") / h, torch.arange(w, device="cuda") / w, indexing="ij")
        a = uniform(3, 4) * 6.0 + 1.0
        im = torch.stack([0.5 + 0.3 * torch.sin(a[k, 0] * x + a[k, 1] * y) * torch.cos(a[k, 2] * y - a[k, 3] * x)
                          for k in range(3)], dim=2)
        im = (im + 0.1 * normal(h, w, 3)).clamp(0.0, 1.0)
        im[: max(1, h // 64)] = -1.0   # no photograph there
        images.append(im)
    return p, sh, _cameras(c), images


def _options(c):
    o = {"shDeg": c["deg"], "precision": PRECISIONS[c["prec"]], "maxSplats": c["n"], "posLr": POS_LR, "seed": 7,
         "viewsPerStep": max(1, c["views"]), "camOpt": int(c["camopt"]), "expComp": int(c["camopt"]),
         "gradAccum": gsabi.GS_ACCUM_F32 if c["accum_f32"] else gsabi.GS_ACCUM_FIXED,
         "loss": gsabi.GS_LOSS_L1_DSSIM if c["ssim"] else gsabi.GS_LOSS_CHARBONNIER}
    if c["keys"]:
        o["entriesCap"] = c["keys"]
    return o


def prepare(case, seed):
    c = case
    p, sh, cams, images = _inputs(c, seed)
    t = gsabi.createTrainer(**_options(c))
    t.setup({"data": p.cpu().numpy(), "n": c["n"], "sh": None if sh is None else sh.cpu().numpy()}, cams,
            [{"tw": im.shape[1], "th": im.shape[0], "rgb": im.reshape(-1).cpu().numpy()} for im in images],
            max(k["w"] for k in cams), max(k["h"] for k in cams), c["ring"])
    t.iter = ITER
    return {"case": c, "trainer": t, "cams": cams}


class _Answer(dict):
    """A training pass's results: the loss, and the Gaussians in the trainer's
    own buffers, which readGaussians gives when they are looked at."""

    def __init__(self, loss, trainer):
        super().__init__(loss=loss, params=None)
        self._trainer = trainer
        if trainer.shK:
            self["sh"] = None

    def __getitem__(self, key):
        if key == "loss":
            return super().__getitem__(key)
        g = self._trainer.readGaussians()
        return g["data"] if key == "params" else g["sh"]


def _views_of(c, step):
    """The cameras of a pass's step: in turn around the ring."""
    return [(step * c["views"] + k) % c["cams"] for k in range(c["views"])]


def run(state):
    c, t = state["case"], state["trainer"]
    if c["kind"] == "render":
        return t.renderView(state["cams"][0])
    if c["kind"] == "eval":
        return [t.evalCamPsnr(k) for k in range(c["cams"])]
    if c["kind"] == "checkpoint":
        g = t.readGaussians()
        return {"params": g["data"], "sh": g["sh"]}
    for s in range(c["steps"]):
        if c["views"] > 1:
            t.stepViews(_views_of(c, s))
        else:
            t.stepOnce(_views_of(c, s)[0])
    return _Answer(t.readLoss(), t)


# ---- what a pass cannot do without ----

def _pairs(c, w, h):
    """About how many (pixel, Gaussian) pairs one view blends: the visible
    Gaussians' footprints, at most some 100 a pixel before it is opaque."""
    f, z = 1100.0 / 1600.0 * w, c["ring"]
    area = math.pi * 9.0 * (0.3 + math.exp(2 * c["ls_mu"] + c["ls_sd"] ** 2) * (f / z) ** 2)
    return min(0.5 * c["n"] * area, 100.0 * w * h)


def work(case):
    """Parameters, coefficients and moments read and written once per Adam
    step, targets read once per view; per Gaussian and view about 400 floating
    operations (900 with the chain), per blended pair 30 (100 with the
    backward)."""
    c = case
    n, C = c["n"], 3 * scenes.sh_k(c["deg"])
    sb, mb = (4 if c["prec"] == "f32" else 2), (2 if c["prec"] == "mixed" else 4)
    scene = n * (56.0 + sb * C)
    sizes = _sizes(c)
    if c["kind"] == "checkpoint":
        return {"bytes": scene + n * (64.0 + 4 * C), "flops": 0.0}
    if c["kind"] == "render":
        w, h = sizes[0]
        return {"bytes": scene + 16.0 * w * h, "flops": 400.0 * n + 30 * _pairs(c, w, h)}
    if c["kind"] == "eval":
        return {"bytes": sum(scene + 4.0 * w * h for w, h in sizes),
                "flops": sum(400.0 * n + 30 * _pairs(c, w, h) for w, h in sizes)}
    total = {"bytes": 0.0, "flops": 0.0}
    for s in range(c["steps"]):
        total["bytes"] += 2 * scene + 4.0 * mb * n * (14 + C)
        for v in _views_of(c, s):
            w, h = sizes[v]
            total["bytes"] += 4.0 * w * h
            total["flops"] += 900.0 * n + 100 * _pairs(c, w, h)
    return total


# ---- the same in float64 ----

E_CUT, A_MIN, TILE = 4.5, 0.0039, 16
SH_C = [0.4886025119029199, 1.0925484305920792, 0.31539156525252005, 0.5462742152960396, 0.5900435899266435,
        2.890611442640554, 0.4570457994644658, 0.3731763325901154, 1.445305721320277]


def _basis(v, deg):
    x, y, z = v.unbind(1)
    xx, yy, zz = x * x, y * y, z * z
    c = SH_C
    Y = [-c[0] * y, c[0] * z, -c[0] * x]
    if deg > 1:
        Y += [c[1] * x * y, -c[1] * y * z, c[2] * (2 * zz - xx - yy), -c[1] * x * z, c[3] * (xx - yy)]
    if deg > 2:   # the last one is the reference's x (xx - yy)
        Y += [-c[4] * y * (3 * xx - yy), c[5] * x * y * z, -c[6] * y * (4 * zz - xx - yy),
              c[7] * z * (2 * zz - 3 * xx - 3 * yy), -c[6] * x * (4 * zz - xx - yy), c[8] * z * (xx - yy),
              -c[4] * x * (xx - yy)]
    return torch.stack(Y, dim=1)


def _project(p, sh, cam, deg):
    """Screen-space mean, conic, opacity and colour (9 columns), depth, tile
    rectangle and the Gaussians that are seen."""
    R = torch.tensor(cam["R"], dtype=torch.float64, device=p.device).float().double().reshape(3, 3)
    t = torch.tensor(cam["t"], dtype=torch.float64, device=p.device).float().double()
    f, W, H = cam["f"], cam["w"], cam["h"]
    pc = p[:, 0:3] @ R.T + t
    near = pc[:, 2] >= 0.05
    z = torch.where(near, pc[:, 2], torch.ones_like(pc[:, 2]))
    q = p[:, 6:10] / p[:, 6:10].norm(dim=1, keepdim=True)
    w, x, y, k = q.unbind(1)
    rot = torch.stack([1 - 2 * (y * y + k * k), 2 * (x * y - w * k), 2 * (x * k + w * y),
                       2 * (x * y + w * k), 1 - 2 * (x * x + k * k), 2 * (y * k - w * x),
                       2 * (x * k - w * y), 2 * (y * k + w * x), 1 - 2 * (x * x + y * y)], dim=1).reshape(-1, 3, 3)
    M = rot * p[:, None, 3:6].clamp(-12.0, 6.0).exp()
    T0 = (f / z)[:, None] * R[0] - (f * pc[:, 0] / z ** 2)[:, None] * R[2]
    T1 = (f / z)[:, None] * R[1] - (f * pc[:, 1] / z ** 2)[:, None] * R[2]
    a, b = (M * T0[:, :, None]).sum(1), (M * T1[:, :, None]).sum(1)
    va, vb, vc = (a * a).sum(1), (a * b).sum(1), (b * b).sum(1)
    ad, cd = va + 0.3, vc + 0.3
    det = ad * cd - vb * vb
    comp = ((va * vc - vb * vb).clamp_min(1e-30) / det).sqrt()
    opa = torch.sigmoid(p[:, 13].clamp(-9.0, 9.0))
    mx, my = f * pc[:, 0] / z + cam["cx"], f * pc[:, 1] / z + cam["cy"]
    col = torch.sigmoid(p[:, 10:13].clamp(-9.0, 9.0))
    if deg:
        u = p[:, 0:3] + R.T @ t
        Y = _basis(u / u.norm(dim=1, keepdim=True).clamp_min(1e-9), deg)
        col = (col + (sh.reshape(len(p), 3, -1) * Y[:, None, :]).sum(2)).clamp_min(0.0)
    rec = torch.cat([torch.stack([mx, my, cd / det, -vb / det, ad / det, opa * comp], dim=1), col], dim=1)
    with torch.no_grad():
        mid = 0.5 * (ad + cd)
        lmax = mid + (mid * mid - det).clamp_min(0.0).sqrt()
        emax = torch.log((opa * comp / A_MIN).clamp_min(1.0001)).clamp_max(E_CUT)
        rad = ((2 * emax).sqrt() * lmax.sqrt()).clamp_max(W)
        ok = near & (opa * comp >= A_MIN) & (mx + rad >= 0) & (my + rad >= 0) & (mx - rad <= W) & (my - rad <= H)
        tx, ty = (W + TILE - 1) // TILE, (H + TILE - 1) // TILE
        rect = torch.stack([((mx - rad) / TILE).floor().clamp(0, tx - 1), ((mx + rad) / TILE).floor().clamp(0, tx - 1),
                            ((my - rad) / TILE).floor().clamp(0, ty - 1), ((my + rad) / TILE).floor().clamp(0, ty - 1)],
                           dim=1).long()
    return rec, pc[:, 2].detach(), rect, ok


def _tiles(depth, rect, ok, W, H):
    """Groups of tiles with like numbers of Gaussians: (tile ids, their Gaussians in depth order, -1 padded)."""
    tx, ty = (W + TILE - 1) // TILE, (H + TILE - 1) // TILE
    seen = ok.nonzero()[:, 0]
    seen = seen[torch.argsort(depth[seen].float(), stable=True)]
    r = rect[seen]
    wide, tall = r[:, 1] - r[:, 0] + 1, r[:, 3] - r[:, 2] + 1
    cnt = wide * tall
    who = torch.repeat_interleave(torch.arange(len(seen), device=r.device), cnt)
    at = torch.arange(len(who), device=r.device) - (cnt.cumsum(0) - cnt)[who]
    tile = (r[who, 2] + at // wide[who]) * tx + r[who, 0] + at % wide[who]
    order = torch.argsort(tile, stable=True)
    who, counts = seen[who[order]], torch.bincount(tile, minlength=tx * ty)
    start = counts.cumsum(0) - counts
    by = torch.argsort(counts, descending=True)
    sizes = counts[by].tolist()
    k = 0
    while k < len(by):
        K = max(1, sizes[k])
        m = min(len(by) - k, max(1, 160000 // K))
        ids = by[k:k + m]
        j = torch.arange(K, device=by.device)
        idx = torch.where(j < counts[ids][:, None], start[ids][:, None] + j, -1)
        yield ids, torch.where(idx >= 0, who[idx.clamp_min(0)], -1) if len(who) else idx
        k += m


def _blend(rec, ids, idx, W):
    """Colour and final transmittance of the tiles' pixels: (m, 256, 3), (m, 256)."""
    tx = (W + TILE - 1) // TILE
    pix = torch.arange(TILE * TILE, device=ids.device)
    px = ((ids % tx) * TILE)[:, None] + pix % TILE + 0.5
    py = ((ids // tx) * TILE)[:, None] + pix // TILE + 0.5
    r = rec[idx.clamp_min(0)]
    dx, dy = px[:, None, :] - r[:, :, 0:1], py[:, None, :] - r[:, :, 1:2]
    e = (0.5 * (r[:, :, 2:3] * dx * dx + r[:, :, 4:5] * dy * dy) + r[:, :, 3:4] * dx * dy).clamp_min(0.0)
    alpha = (r[:, :, 5:6] * torch.exp(-e)).clamp_max(0.99)
    take = (e.detach() <= E_CUT) & (alpha.detach() >= A_MIN) & (idx >= 0)[:, :, None]
    step = torch.log1p(-torch.where(take, alpha, torch.zeros_like(alpha)))
    before = step.cumsum(1) - step
    take = take & (before.detach() >= math.log(1e-4))
    step = torch.where(take, step, torch.zeros_like(step))
    wgt = torch.where(take, alpha * torch.exp(before), torch.zeros_like(alpha))
    return torch.einsum("mkp,mkc->mpc", wgt, r[:, :, 6:9]), torch.exp(step.sum(1))


def _image(rec, depth, rect, ok, W, H, grad=None):
    """The image h x w x 4 (colour, 1 - T); with grad (h x w x 3): the gradient of rec instead."""
    tx, ty = (W + TILE - 1) // TILE, (H + TILE - 1) // TILE

    def tiled(im):
        return im.reshape(ty, TILE, tx, TILE, -1).permute(0, 2, 1, 3, 4).reshape(tx * ty, TILE * TILE, -1)

    if grad is None:
        out = torch.zeros(tx * ty, TILE * TILE, 4, dtype=torch.float64, device=rec.device)
        with torch.no_grad():
            for ids, idx in _tiles(depth, rect, ok, W, H):
                C, T = _blend(rec, ids, idx, W)
                out[ids, :, :3], out[ids, :, 3] = C, 1 - T
        return out.reshape(ty, tx, TILE, TILE, 4).permute(0, 2, 1, 3, 4).reshape(ty * TILE, tx * TILE, 4)[:H, :W]
    full = torch.zeros(ty * TILE, tx * TILE, 3, dtype=torch.float64, device=rec.device)
    full[:H, :W] = grad
    full = tiled(full)
    leaf = rec.detach().requires_grad_()
    for ids, idx in _tiles(depth, rect, ok, W, H):
        C, _ = _blend(leaf, ids, idx, W)
        C.backward(full[ids])
    return leaf.grad


def _loss(img, tgt, ssim):
    """(sum of squared errors, valid pixels, the loss) of an image against its 8-bit target."""
    valid = tgt[:, :, 0] >= 0
    y = torch.where(valid[:, :, None], torch.floor(tgt.double() * 255.0 + 0.5).clamp(0, 255) / 255.0, 0.0)
    x = torch.where(valid[:, :, None], img, torch.zeros_like(img))
    err = x - y
    sq, count = float((err.detach() ** 2).sum()), int(valid.sum())
    if not ssim:
        return sq, count, ((err * err + 0.0009).sqrt() - 0.03)[valid].sum()
    g = torch.exp(-(torch.arange(11, dtype=torch.float64, device=img.device) - 5) ** 2 / (2 * 1.5 ** 2))
    g = g / g.sum()

    def blur(v):
        v = v.permute(2, 0, 1)[:, None]
        v = torch.nn.functional.pad(v, (5, 5, 5, 5))
        v = sum(g[k] * v[:, :, :, k:k + v.shape[3] - 10] for k in range(11))
        v = sum(g[k] * v[:, :, k:k + v.shape[2] - 10] for k in range(11))
        return v[:, 0].permute(1, 2, 0)

    ux, uy = blur(x), blur(y)
    vx, vy, cxy = blur(x * x) - ux * ux, blur(y * y) - uy * uy, blur(x * y) - ux * uy
    s = ((2 * ux * uy + 1e-4) * (2 * cxy + 9e-4)) / ((ux * ux + uy * uy + 1e-4) * (vx + vy + 9e-4))
    return sq, count, (0.8 * err.abs() + 0.2 * (1 - s))[valid].sum()


def _adam(v, grad, m, s, lr, t):
    g = torch.where(grad.abs() < 1e18, grad, torch.zeros_like(grad))
    m.mul_(0.9).add_(g, alpha=0.1)
    s.mul_(0.999).addcmul_(g, g, value=0.001)
    return v - lr * (m / (1 - 0.9 ** t)) / ((s / (1 - 0.999 ** t)).sqrt() + 1e-15)


def _train64(c, p, sh, cams, images):
    n, deg, radius = c["n"], c["deg"], c["ring"]
    p = p.double()[:, :14].contiguous()
    sh = None if sh is None else sh.double()
    m, s = torch.zeros_like(p), torch.zeros_like(p)
    mh, ss = (None, None) if sh is None else (torch.zeros_like(sh), torch.zeros_like(sh))
    it, t, sq, count = ITER, ITER, 0.0, 0
    lr = torch.tensor([0.0] * 3 + [5e-3] * 3 + [1e-3] * 4 + [1.5e-2] * 3 + [2.5e-2], dtype=torch.float64, device=p.device)
    for k in range(c["steps"]):
        g, gs = torch.zeros_like(p), None if sh is None else torch.zeros_like(sh)
        for v in _views_of(c, k):
            pl = p.clone().requires_grad_()
            sl = None if sh is None else sh.clone().requires_grad_()
            cam = cams[v]
            rec, depth, rect, ok = _project(pl, sl, cam, deg)
            img = _image(rec.detach(), depth, rect, ok, cam["w"], cam["h"])[:, :, :3].clone().requires_grad_()
            a, b, loss = _loss(img, images[v], c["ssim"])
            sq, count = sq + a, count + b
            loss.backward()
            grec = _image(rec, depth, rect, ok, cam["w"], cam["h"], grad=img.grad)
            if grec is None or not bool(ok.any()):
                continue
            ls = pl[:, 3:6].clamp(-12.0, 6.0)
            spread = 0.5 * ((ls - ls.mean(1, keepdim=True)) ** 2).sum(1)   # the anisotropy regulariser
            ((rec * torch.where(ok[:, None], grec, 0.0)).sum() + 0.005 * spread[ok].sum()).backward()
            g += torch.where(ok[:, None], pl.grad, 0.0)
            if sl is not None:
                gs += torch.where(ok[:, None], sl.grad, 0.0)
        it, t = it + c["views"], t + 1
        lr[0:3] = POS_LR * 0.01 ** min(1.0, it / (0.75 * 60000))
        o = torch.sigmoid(p[:, 13].clamp(-9.0, 9.0))
        g[:, 13] += 0.01 * o * (1 - o)
        p = _adam(p, g, m, s, lr, t)
        p[:, 3:6] = p[:, 3:6].clamp(math.log(radius * 1e-4), math.log(radius * 0.05))
        p[:, 10:14] = p[:, 10:14].clamp(-8.0, 8.0)
        if sh is not None:
            sh = _adam(sh, gs, mh, ss, 1.25e-4, t)
    full = torch.zeros(n, 16, dtype=torch.float64, device=p.device)
    full[:, :14] = p
    out = {"loss": sq / (3.0 * max(1, count)), "params": full.cpu().numpy()}
    if sh is not None:
        out["sh"] = sh.cpu().numpy()
    return out


def exact(case, seed):
    c = case
    if c["ls_sd"] > 0.9 and c["n"] > 50000:
        return None   # tens of millions of keys a view
    p, sh, cams, images = _inputs(c, seed)
    if c["kind"] == "checkpoint":
        return {"params": p.double().cpu().numpy(), "sh": None if sh is None else sh.double().cpu().numpy()}
    if c["kind"] == "train":
        return _train64(c, p, sh, cams, images)
    out = []
    for cam, tgt in zip(cams, images):
        rec, depth, rect, ok = _project(p.double(), None if sh is None else sh.double(), cam, c["deg"])
        img = _image(rec, depth, rect, ok, cam["w"], cam["h"])
        if c["kind"] == "render":
            return img.cpu().numpy()
        sq, count, _ = _loss(img[:, :, :3], tgt, False)
        out.append(-10.0 * math.log10(sq / (3.0 * max(1, count))))
    return out
