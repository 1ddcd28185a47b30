"""Performance cases of gsplat_amd: the calls a user's program makes through
the package's public entry points, with the sizes they are made at.

``listed()`` holds the named cases and ``draw()`` more of the same ranges;
``prepare()`` makes a case's inputs on the GPU, ``run()`` is one pass,
``work()`` its unavoidable bytes and arithmetic, ``tolerance()`` how far two
correct float32 implementations may be apart, and ``exact()`` the same outputs
in float64 from plain torch operations.

Kinds of case:
  train   rasterization() and its backward, from the gradient a loss hands to
          the render, to every Gaussian parameter;
  render  rasterization() without gradients;
  step    a whole optimizer step: activations of the raw parameters,
          rasterization() with absgrad, backward with the fused densification
          statistics, SelectiveAdam over six parameter groups;
  ops     the gsplat.cuda wrappers called one by one (dense projection,
          spherical harmonics, tile intersection, offsets, rasterizer), and
          the backward through them;
  adam    SelectiveAdam.step alone, under a visibility mask.
"""

from __future__ import annotations

import math

import torch

import gsplat_amd as gs
from gsplat_amd.strategy.stats import fuse_grad2d_stats

DEV = "cuda:0"
TILE = 16

_DEFAULTS = {
    "scene": "cloud", "batch": 1, "cameras": 1, "sh": -1, "channels": 3, "mode": "RGB",
    "packed": True, "antialiased": False, "background": False, "alpha_grad": False,
    "radius_clip": 0.0, "scale": -4.0,
}


def _case(kind, n, width, height, **kw):
    return {"kind": kind, "n": n, "width": width, "height": height, **_DEFAULTS, **kw}


def listed():
    return [
        # A first look at the library: ten thousand coloured Gaussians in
        # front of one small camera.  Launches and host time decide it.
        dict(_case("train", 10_000, 256, 256, scene="slab", sh=0, scale=-3.0),
             name="train_toy"),
        # One view of a trained scene's parameters, the ordinary training
        # step of a 3D Gaussian splatting trainer: a million Gaussians, SH 3.
        dict(_case("train", 1_000_000, 1280, 720, sh=3), name="train_1m_sh3"),
        # A batch of views a step, colours and expected depth under loss.
        dict(_case("train", 500_000, 960, 540, sh=1, cameras=8, mode="RGB+ED"),
             name="train_8views_rgb_ed"),
        # The dense (unpacked) layout with antialiasing, a background and a
        # loss on the alphas too; an image that no tile size divides.
        dict(_case("train", 300_000, 1237, 821, sh=2, packed=False, antialiased=True,
                   background=True, alpha_grad=True, scale=-3.6),
             name="train_unpacked_aa"),
        # Feature fields: 32 channels per Gaussian instead of a colour.
        dict(_case("train", 111_785, 1920, 1080, channels=32, scale=-3.3),
             name="train_32_channels"),
        # Many small scenes in one call (batch dimensions).
        dict(_case("train", 10_000, 320, 180, batch=16, scene="slab", packed=False,
                   scale=-3.0),
             name="train_batch16"),
        # A viewer's frame of a small scene: latency of one forward pass.
        dict(_case("render", 60_000, 640, 360, sh=3, scale=-3.2), name="render_small"),
        # A frame of a large captured scene around the camera.
        dict(_case("render", 6_000_000, 1920, 1080, scene="box", sh=3),
             name="render_6m_1080p"),
        # The trainer's whole step at two million Gaussians.
        dict(_case("step", 2_000_000, 1600, 1040, sh=3), name="step_2m_adam"),
        # A program written against the wrappers instead of rasterization().
        dict(_case("ops", 200_000, 801, 603, sh=3, packed=False, scale=-3.5),
             name="ops_dense_chain"),
        # The masked optimizer update of a million Gaussians, of which this
        # step's view saw about two thirds.
        dict(_case("adam", 1_000_000, 1, 1, sh=3), name="selective_adam_1m"),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def image(lo, hi):
        h = size(lo, hi)
        return int(h * rng.uniform(1.0, 1.9)), h

    def fitted(n):
        # Gaussians of a scene get smaller as there are more of them
        return round(-4.0 + math.log(1e6 / n) / 3.0 * 0.9, 2)

    kind = rng.choice(["train", "train", "train", "render", "render", "step", "ops", "adam"])
    if kind == "train":
        form = rng.choice(["view", "view", "views", "dense", "features", "batch", "small"])
        if form == "small":
            n = size(5_000, 50_000)
            w, h = image(160, 400)
            return _case("train", n, w, h, scene="slab", sh=rng.choice([-1, 0, 3]), scale=-3.0,
                         packed=rng.random() < 0.7)
        if form == "batch":
            n = size(5_000, 20_000)
            w, h = image(120, 220)
            return _case("train", n, w, h, scene="slab", batch=rng.randint(2, 16), scale=-3.0,
                         sh=rng.choice([-1, 1]), packed=rng.random() < 0.3)
        if form == "features":
            n = size(30_000, 120_000)
            w, h = image(300, 1000)
            return _case("train", n, w, h, channels=rng.choice([8, 16, 24, 32]),
                         scale=fitted(n), packed=rng.random() < 0.6)
        if form == "views":
            n = size(50_000, 400_000)
            w, h = image(240, 500)
            return _case("train", n, w, h, cameras=rng.randint(2, 8), scale=fitted(n),
                         sh=rng.choice([0, 1, 2, 3]), packed=rng.random() < 0.7,
                         mode=rng.choice(["RGB", "RGB+D", "RGB+ED"]))
        n = size(50_000, 1_200_000)
        w, h = image(360, 900)
        dense = form == "dense"
        return _case("train", n, w, h, scale=fitted(n), sh=rng.choice([1, 2, 3, 3]),
                     packed=not dense, antialiased=rng.random() < 0.4,
                     background=rng.random() < 0.5, alpha_grad=rng.random() < 0.4,
                     radius_clip=rng.choice([0.0, 0.0, 3.0]),
                     mode=rng.choice(["RGB", "RGB", "RGB+ED", "ED"]))
    if kind == "render":
        n = size(30_000, 5_000_000)
        w, h = image(300, 1080)
        if n > 1_000_000 or rng.random() < 0.3:
            return _case("render", n, w, h, scene="box", sh=rng.choice([0, 3, 3]),
                         packed=rng.random() < 0.8)
        return _case("render", n, w, h, scale=fitted(n), sh=rng.choice([-1, 1, 3]),
                     mode=rng.choice(["RGB", "RGB", "RGB+ED"]), packed=rng.random() < 0.8,
                     antialiased=rng.random() < 0.3)
    if kind == "step":
        n = size(200_000, 1_500_000)
        w, h = image(500, 900)
        return _case("step", n, w, h, sh=rng.choice([1, 2, 3, 3]), scale=fitted(n))
    if kind == "ops":
        n = size(20_000, 400_000)
        w, h = image(200, 800)
        return _case("ops", n, w, h, sh=rng.choice([0, 1, 2, 3, 4]), packed=False,
                     scale=fitted(n))
    return _case("adam", size(50_000, 2_000_000), 1, 1, sh=rng.choice([0, 1, 2, 3, 3]))


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------
def _look_at(px, py, pz):
    """World-to-camera matrix of a camera at (px, py, pz) looking at the
    origin (x right, y down, z forward)."""
    p = torch.tensor([px, py, pz], dtype=torch.float64)
    z = -p / p.norm()
    x = torch.linalg.cross(z, torch.tensor([0.0, -1.0, 0.0], dtype=torch.float64))
    x = x / x.norm()
    y = torch.linalg.cross(z, x)
    m = torch.eye(4, dtype=torch.float64)
    m[:3, :3] = torch.stack([x, y, z])
    m[:3, 3] = -m[:3, :3] @ p
    return m.float()


def _cameras(c):
    """viewmats [C, 4, 4] and Ks [C, 3, 3] of one scene of the case."""
    C, W, H = c["cameras"], c["width"], c["height"]
    focal = {"slab": 1.0, "cloud": 0.78125, "box": 0.625}[c["scene"]] * W
    if c["scene"] != "cloud":
        views = torch.eye(4).repeat(C, 1, 1)
    elif C == 1:
        views = torch.eye(4)[None].clone()
        views[0, 2, 3] = 6.0
    else:
        focal = W / 1.2
        views = torch.stack([_look_at(5 * math.cos(2 * math.pi * k / C), -1.0,
                                      5 * math.sin(2 * math.pi * k / C)) for k in range(C)])
    K = torch.tensor([[focal, 0.0, W / 2.0], [0.0, focal, H / 2.0], [0.0, 0.0, 1.0]])
    return views, K[None].repeat(C, 1, 1)


def _gaussians(c, seed):
    """Raw parameters (before the activations) on the GPU."""
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    B, n = c["batch"], c["n"]
    lead = (B, n) if B > 1 else (n,)

    def normal(*tail, s=1.0):
        return torch.randn(*lead, *tail, generator=g, device=DEV) * s

    def uniform(*tail):
        return torch.rand(*lead, *tail, generator=g, device=DEV)

    if c["scene"] == "slab":
        means = uniform(3) * 2 - 1
        means[..., 2] += 3.0
        spread, logit = 0.5, 1.0
    elif c["scene"] == "box":
        means = (uniform(3) - 0.5) * torch.tensor([40.0, 10.0, 40.0], device=DEV)
        spread, logit = 1.0, 2.0
    else:
        means = normal(3, s=2.0)
        spread, logit = 0.7, 1.5
    quats = normal(4)
    raw = {
        "means": means,
        "quats": quats / quats.norm(dim=-1, keepdim=True),
        "log_scales": normal(3, s=spread) + c["scale"],
        "logits": normal(s=logit),
    }
    if c["sh"] >= 0:
        k = (c["sh"] + 1) ** 2
        raw["colors"] = torch.cat([normal(1, 3, s=0.5), normal(k - 1, 3, s=0.05)], dim=-2)
    else:
        raw["colors"] = uniform(c["channels"])
    return raw, g


def _channels(c):
    d = 3 if c["sh"] >= 0 else c["channels"]
    return {"RGB": d, "D": 1, "ED": 1}.get(c["mode"], d + 1)


def _loss_grads(c, g):
    """What an L1 loss hands back: +-1/n for every value of the render (and
    of the alphas), as a mean over n values gives it."""
    lead = ((c["batch"],) if c["batch"] > 1 else ()) + (c["cameras"], c["height"], c["width"])

    def signs(d):
        shape = lead + (d,)
        up = torch.rand(shape, generator=g, device=DEV) < 0.5
        return torch.where(up, 1.0, -1.0) / math.prod(shape)

    return signs(_channels(c)), signs(1) if c["alpha_grad"] else None


_LRS = {  # a trainer's rates, late in the schedule (a hundredth of the first ones)
    "means": 1.6e-6, "log_scales": 5e-5, "quats": 1e-5, "logits": 5e-4, "sh0": 2.5e-5,
    "shN": 1.25e-6,
}
_BETAS, _EPS = (0.9, 0.999), 1e-15


def _optimizer_state(c, seed):
    """Six parameter groups with moments as in the middle of a training."""
    raw, g = _gaussians(c, seed)
    colors = raw.pop("colors")
    raw["sh0"] = colors[:, :1].contiguous()
    raw["shN"] = colors[:, 1:].contiguous()
    if raw["shN"].numel() == 0:
        del raw["shN"]
    moments = {}
    for k, p in raw.items():
        m = torch.randn(p.shape, generator=g, device=DEV) * 1e-7
        v = (torch.rand(p.shape, generator=g, device=DEV) + 0.1) * 1e-12
        moments[k] = (m, v)
    return raw, moments, g


def _selective_adam(raw, moments):
    params = {k: torch.nn.Parameter(v) for k, v in raw.items()}
    opt = gs.SelectiveAdam([{"params": [p], "lr": _LRS[k], "name": k}
                            for k, p in params.items()], eps=_EPS, betas=_BETAS)
    for k, p in params.items():
        opt.state[p] = {"step": torch.tensor(0.0), "exp_avg": moments[k][0],
                        "exp_avg_sq": moments[k][1]}
    return params, opt


def _adam_inputs(c, seed):
    raw, moments, g = _optimizer_state(c, seed)
    grads = {k: torch.randn(p.shape, generator=g, device=DEV) * 1e-6 for k, p in raw.items()}
    visible = torch.rand(c["n"], generator=g, device=DEV) < 0.66
    return raw, moments, grads, visible


def _rasterization_kwargs(c):
    return {
        "sh_degree": c["sh"] if c["sh"] >= 0 else None, "packed": c["packed"],
        "render_mode": c["mode"], "radius_clip": c["radius_clip"],
        "rasterize_mode": "antialiased" if c["antialiased"] else "classic",
    }


def _backgrounds(c, g):
    if not c["background"]:
        return None
    lead = ((c["batch"],) if c["batch"] > 1 else ()) + (c["cameras"],)
    d = 3 if c["sh"] >= 0 else c["channels"]
    return torch.rand(*lead, d, generator=g, device=DEV)


def _inputs(c, seed):
    """Activated parameters, cameras, backgrounds and the loss's gradients."""
    raw, g = _gaussians(c, seed)
    params = {"means": raw["means"], "quats": raw["quats"], "scales": raw["log_scales"].exp(),
              "opacities": torch.sigmoid(raw["logits"]), "colors": raw["colors"]}
    views, Ks = _cameras(c)
    if c["batch"] > 1:
        views = views.repeat(c["batch"], 1, 1, 1)
        Ks = Ks.repeat(c["batch"], 1, 1, 1)
    return params, views.to(DEV), Ks.to(DEV), _backgrounds(c, g), g


def prepare(case, seed):
    c = case
    if c["kind"] == "adam":
        raw, moments, grads, visible = _adam_inputs(c, seed)
        params, opt = _selective_adam(raw, moments)
        for k, p in params.items():
            p.grad = grads[k]
        return {"case": c, "params": params, "opt": opt, "visible": visible}
    if c["kind"] == "step":
        raw, moments, g = _optimizer_state(c, seed)
        params, opt = _selective_adam(raw, moments)
        views, Ks = _cameras(c)
        v_rc, _ = _loss_grads(c, g)
        return {"case": c, "params": params, "opt": opt, "views": views.to(DEV),
                "Ks": Ks.to(DEV), "v_rc": v_rc, "grad2d": torch.zeros(c["n"], device=DEV),
                "count": torch.zeros(c["n"], device=DEV)}
    params, views, Ks, bg, g = _inputs(c, seed)
    s = {"case": c, "views": views, "Ks": Ks, "bg": bg}
    if c["kind"] == "render":
        s["params"] = params
    else:
        s["params"] = {k: v.requires_grad_() for k, v in params.items()}
        s["v_rc"], s["v_ra"] = _loss_grads(c, g)
    return s


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------
def run(state):
    return {"train": _run_train, "render": _run_render, "step": _run_step, "ops": _run_ops,
            "adam": _run_adam}[state["case"]["kind"]](state)


def _rasterize(s, p):
    c = s["case"]
    colors = p["colors"] if c["mode"] not in ("D", "ED") else None
    kw = _rasterization_kwargs(c)
    if colors is None:
        kw["sh_degree"] = None
    return gs.rasterization(p["means"], p["quats"], p["scales"], p["opacities"], colors,
                            s["views"], s["Ks"], c["width"], c["height"],
                            backgrounds=s["bg"], **kw)


def _run_render(s):
    with torch.no_grad():
        rc, ra, _ = _rasterize(s, s["params"])
    return {"colors": rc, "alphas": ra}


def _pull_back(s, rc, ra):
    """Gradients of every parameter the render depends on."""
    p = s["params"]
    if s["case"]["mode"] in ("D", "ED"):
        p = {k: v for k, v in p.items() if k != "colors"}
    outs, ups = [rc], [s["v_rc"]]
    if s["v_ra"] is not None:
        outs, ups = outs + [ra], ups + [s["v_ra"]]
    return dict(zip(p, torch.autograd.grad(outs, list(p.values()), ups)))


def _run_train(s):
    rc, ra, _ = _rasterize(s, s["params"])
    return {"colors": rc.detach(), "alphas": ra.detach(), "grads": _pull_back(s, rc, ra)}


def _run_ops(s):
    c, p = s["case"], s["params"]
    W, H, C = c["width"], c["height"], c["cameras"]
    tw, th = math.ceil(W / TILE), math.ceil(H / TILE)
    radii, means2d, depths, conics, _ = gs.fully_fused_projection(
        p["means"], None, p["quats"], p["scales"], s["views"], s["Ks"], W, H,
        opacities=p["opacities"])
    R, t = s["views"][:, :3, :3], s["views"][:, :3, 3]
    centers = -(R * t[:, :, None]).sum(dim=1)
    dirs = p["means"][None] - centers[:, None]
    coeffs = p["colors"][None].expand(C, *p["colors"].shape)
    colors = gs.spherical_harmonics(c["sh"], dirs, coeffs, masks=(radii > 0).all(dim=-1))
    colors = torch.clamp_min(colors + 0.5, 0.0)
    opac = p["opacities"][None].expand(C, c["n"])
    _, isect_ids, flatten_ids = gs.isect_tiles(means2d, radii, depths, TILE, tw, th,
                                               conics=conics, opacities=opac)
    offsets = gs.isect_offset_encode(isect_ids, C, tw, th)
    rc, ra = gs.rasterize_to_pixels(means2d, conics, colors, opac, W, H, TILE, offsets,
                                    flatten_ids)
    return {"colors": rc.detach(), "alphas": ra.detach(), "grads": _pull_back(s, rc, ra)}


def _optimizer_outputs(s):
    state = s["opt"].state
    return {k: {"param": p.detach(), "exp_avg": state[p]["exp_avg"],
                "exp_avg_sq": state[p]["exp_avg_sq"]} for k, p in s["params"].items()}


def _run_adam(s):
    s["opt"].step(s["visible"])
    return _optimizer_outputs(s)


def _run_step(s):
    c, p = s["case"], s["params"]
    colors = torch.cat([p["sh0"], p["shN"]], dim=1)
    rc, ra, meta = gs.rasterization(
        p["means"], p["quats"], p["log_scales"].exp(), torch.sigmoid(p["logits"]), colors,
        s["views"], s["Ks"], c["width"], c["height"], absgrad=True, **_rasterization_kwargs(c))
    s["grad2d"], s["count"], fused = fuse_grad2d_stats(meta, s["grad2d"], s["count"], c["n"])
    torch.autograd.backward([rc], [s["v_rc"]])
    if not fused:
        s["grad2d"], s["count"] = gs.accumulate_grad2d_stats(
            meta, s["grad2d"], s["count"], c["n"], packed=c["packed"], absgrad=True)
    s["opt"].step(None)
    s["opt"].zero_grad(set_to_none=True)
    return {"colors": rc.detach(), "alphas": ra.detach(), "grad2d": s["grad2d"],
            "count": s["count"], "groups": _optimizer_outputs(s)}


# --------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------
def work(case):
    """Bytes: every input read once, every output written once (float32).
    Arithmetic: the compositing of about 60 Gaussians per pixel (what these
    scenes reach before a pixel is opaque), 30 operations each forward and 70
    backward, more with more channels, and some 500 per Gaussian and camera."""
    c = case
    n, k = c["n"] * c["batch"], (c["sh"] + 1) ** 2 * 3 if c["sh"] >= 0 else c["channels"]
    per = 3 + 4 + 3 + 1 + k
    if c["kind"] == "adam":
        seen = 0.66
        return {"bytes": 4.0 * 7 * n * per * seen + n, "flops": 12.0 * n * per * seen}
    pixels = c["batch"] * c["cameras"] * c["width"] * c["height"]
    d = _channels(c)
    forward = 4.0 * (n * per + pixels * (d + 1))
    flops_f = pixels * 60.0 * (24 + 2 * d) + 500.0 * n * c["cameras"]
    if c["kind"] == "render":
        return {"bytes": forward, "flops": flops_f}
    backward = 4.0 * (n * per + pixels * (d + (1 if c["alpha_grad"] else 0)))
    flops_b = pixels * 60.0 * (60 + 4 * d) + 1000.0 * n * c["cameras"]
    if c["kind"] != "step":
        return {"bytes": forward + backward, "flops": flops_f + flops_b}
    # the update reads parameters, gradients and both moments and writes all
    # but the gradients; the statistics are two accumulators
    return {"bytes": forward + backward + 4.0 * 6 * n * per + 16.0 * n,
            "flops": flops_f + flops_b + 12.0 * n * per}


def tolerance(case):
    """About four times the largest error seen against ``exact()`` over the
    listed cases and two dozen drawn ones.  Renders: 2e-5 (a pixel whose alpha
    or transmittance lies at a threshold may take or leave one Gaussian, up to
    7e-3 of the render).  Gradients: 6e-4, single ones 0.24, since their terms
    cancel by three to five orders of magnitude.  A step's moments hold a
    tenth of the gradient: 4e-5 and 1.3e-2.  Adam: 2e-7 and 1e-6."""
    if case["kind"] == "adam":
        return {"rel": 6e-7, "max": 4e-6}
    if case["kind"] == "render":
        return {"rel": 1e-4, "max": 0.03}
    if case["kind"] == "step":
        return {"rel": 2e-4, "max": 0.05}
    return {"rel": 2.5e-3, "max": 0.9}


# --------------------------------------------------------------------------
# The same in float64, from plain torch operations
# --------------------------------------------------------------------------
def _sh_basis(degree, d):
    """Real spherical harmonics Y_lm of unit directions d [n, 3] for l up to
    ``degree``, m = -l .. l, as sqrt((2l+1)/4pi) times the polynomials of the
    Cartesian form with the sign (-1)^m of the Condon-Shortley phase."""
    x, y, z = d.unbind(-1)
    pi = math.pi
    one = torch.ones_like(x)
    out = [one * math.sqrt(1 / (4 * pi))]
    if degree >= 1:
        a = math.sqrt(3 / (4 * pi))
        out += [-a * y, a * z, -a * x]
    if degree >= 2:
        a, b = math.sqrt(15 / (4 * pi)), math.sqrt(5 / (16 * pi))
        out += [a * x * y, -a * y * z, b * (3 * z * z - 1), -a * x * z,
                a / 2 * (x * x - y * y)]
    if degree >= 3:
        a, b = math.sqrt(35 / (32 * pi)), math.sqrt(105 / (4 * pi))
        e, f = math.sqrt(21 / (32 * pi)), math.sqrt(7 / (16 * pi))
        out += [-a * y * (3 * x * x - y * y), b * x * y * z, -e * y * (5 * z * z - 1),
                f * z * (5 * z * z - 3), -e * x * (5 * z * z - 1),
                b / 2 * z * (x * x - y * y), -a * x * (x * x - 3 * y * y)]
    if degree >= 4:
        a, b = 3 * math.sqrt(35 / (16 * pi)), 3 * math.sqrt(35 / (32 * pi))
        e, f = 3 * math.sqrt(5 / (16 * pi)), 3 * math.sqrt(5 / (32 * pi))
        out += [a * x * y * (x * x - y * y), -b * y * z * (3 * x * x - y * y),
                e * x * y * (7 * z * z - 1), -f * y * z * (7 * z * z - 3),
                3 / 16 / math.sqrt(pi) * (35 * z ** 4 - 30 * z * z + 3),
                -f * x * z * (7 * z * z - 3), e / 2 * (x * x - y * y) * (7 * z * z - 1),
                -b * x * z * (x * x - 3 * y * y),
                a / 4 * (x ** 4 - 6 * x * x * y * y + y ** 4)]
    return torch.stack(out, dim=-1)


def _mat_mul(A, B):
    """[..., i, k] x [..., k, j] by products and a sum."""
    return (A[..., :, :, None] * B[..., None, :, :]).sum(dim=-2)


def _project64(c, p, view, K):
    """Rows of one camera: indices of the visible Gaussians and their means,
    conics, depths, opacities and extents in the image."""
    W, H = c["width"], c["height"]
    fx, fy, cx, cy = (float(K[i, j]) for i, j in ((0, 0), (1, 1), (0, 2), (1, 2)))
    R, t = view[:3, :3], view[:3, 3]
    cam = (p["means"][:, None, :] * R[None]).sum(dim=-1) + t
    x, y, z = cam.unbind(-1)
    q = p["quats"] / p["quats"].norm(dim=-1, keepdim=True)
    w, i, j, k = q.unbind(-1)
    rot = torch.stack([
        1 - 2 * (j * j + k * k), 2 * (i * j - w * k), 2 * (i * k + w * j),
        2 * (i * j + w * k), 1 - 2 * (i * i + k * k), 2 * (j * k - w * i),
        2 * (i * k - w * j), 2 * (j * k + w * i), 1 - 2 * (i * i + j * j)], dim=-1)
    axes = _mat_mul(R[None], rot.view(-1, 3, 3)) * p["scales"][:, None, :]
    lx0, lx1 = cx / fx + 0.15 * W / fx, (W - cx) / fx + 0.15 * W / fx
    ly0, ly1 = cy / fy + 0.15 * H / fy, (H - cy) / fy + 0.15 * H / fy
    tx = z * (x / z).clamp(-lx0, lx1)
    ty = z * (y / z).clamp(-ly0, ly1)
    rows_x = fx / z[:, None] * axes[:, 0] - (fx * tx / z ** 2)[:, None] * axes[:, 2]
    rows_y = fy / z[:, None] * axes[:, 1] - (fy * ty / z ** 2)[:, None] * axes[:, 2]
    a, b, d = (rows_x * rows_x).sum(-1), (rows_x * rows_y).sum(-1), (rows_y * rows_y).sum(-1)
    A, D = a + 0.3, d + 0.3
    det = A * D - b * b
    opac = p["opacities"]
    if c["antialiased"]:
        opac = opac * ((a * d - b * b) / det).clamp(min=0.005 ** 2).sqrt()
    m2 = torch.stack([fx * x / z + cx, fy * y / z + cy], dim=-1)
    con = torch.stack([D / det, -b / det, A / det], dim=-1)
    with torch.no_grad():
        ext = (2 * (opac * 255).clamp(min=1).log()).sqrt().clamp(max=3.33)
        ex, ey = ext * A.sqrt(), ext * D.sqrt()
        rx, ry = ex.ceil(), ey.ceil()
        u, v = m2.unbind(-1)
        see = (z >= 0.01) & (z <= 1e10) & (det > 0) & (opac * 255 >= 1)
        see &= ~((rx <= c["radius_clip"]) & (ry <= c["radius_clip"]))
        see &= (u + rx > 0) & (u - rx < W) & (v + ry > 0) & (v - ry < H)
        ids = torch.nonzero(see)[:, 0]
    return ids, m2[ids], con[ids], z[ids], opac[ids], torch.stack([ex, ey], dim=-1)[ids] + 1.0


def _features64(c, p, view, ids, depth):
    if c["mode"] in ("D", "ED"):
        return depth[:, None]
    if c["sh"] >= 0:
        center = -(view[:3, :3] * view[:3, 3][:, None]).sum(dim=0)
        d = p["means"][ids] - center
        basis = _sh_basis(c["sh"], d / d.norm(dim=-1, keepdim=True))
        f = ((basis[:, :, None] * p["colors"][ids]).sum(dim=1) + 0.5).clamp(min=0.0)
    else:
        f = p["colors"][ids]
    return torch.cat([f, depth[:, None]], dim=-1) if c["mode"] != "RGB" else f


def _tile_lists64(c, m2, ext, depth):
    """Rows of every tile in depth order: (tile ids, starts, counts, rows)."""
    W, H = c["width"], c["height"]
    tw, th = math.ceil(W / TILE), math.ceil(H / TILE)
    order = torch.sort(depth.float(), stable=True).indices
    m, e = m2[order], ext[order]
    x0 = ((m[:, 0] - e[:, 0]) / TILE).floor().clamp(0, tw).long()
    x1 = ((m[:, 0] + e[:, 0]) / TILE).floor().add(1).clamp(0, tw).long()
    y0 = ((m[:, 1] - e[:, 1]) / TILE).floor().clamp(0, th).long()
    y1 = ((m[:, 1] + e[:, 1]) / TILE).floor().add(1).clamp(0, th).long()
    nx = x1 - x0
    cnt = nx * (y1 - y0)
    row = torch.repeat_interleave(torch.arange(len(cnt), device=DEV), cnt)
    at = torch.arange(len(row), device=DEV) - (cnt.cumsum(0) - cnt)[row]
    tile = (y0[row] + at // nx[row]) * tw + x0[row] + at % nx[row]
    tile, by = torch.sort(tile, stable=True)
    ids, counts = torch.unique_consecutive(tile, return_counts=True)
    return ids, counts.cumsum(0) - counts, counts, order[row[by]]


def _composite64(c, rows, bg, v_rc, v_ra, back, absgrad):
    """Render of one image from its rows (means, conics, opacities, features,
    extents, depths) and, with ``back``, the rows' gradients."""
    m2, con, op, f, ext, depth = rows
    W, H, D = c["width"], c["height"], f.shape[-1]
    tw, th = math.ceil(W / TILE), math.ceil(H / TILE)
    tiles, starts, counts, listed_rows = _tile_lists64(c, m2, ext, depth)
    by = torch.argsort(counts, descending=True)
    tiles, starts, counts = tiles[by], starts[by], counts[by]
    host = counts.tolist()
    if bg is None:
        bg = torch.zeros(D, dtype=torch.float64, device=DEV)
    rc = bg.repeat(th * tw, TILE * TILE, 1)
    ra = torch.zeros(th * tw, TILE * TILE, dtype=torch.float64, device=DEV)

    def tiled(v):
        full = torch.zeros(th * TILE, tw * TILE, v.shape[-1], dtype=torch.float64, device=DEV)
        full[:H, :W] = v
        return full.view(th, TILE, tw, TILE, -1).transpose(1, 2).reshape(th * tw, TILE * TILE, -1)

    def untiled(v):
        full = v.view(th, tw, TILE, TILE, -1).transpose(1, 2).reshape(th * TILE, tw * TILE, -1)
        return full[:H, :W]

    grads = None
    if back:
        up, upa = tiled(v_rc.double()), None if v_ra is None else tiled(v_ra.double())[..., 0]
        grads = [torch.zeros_like(t) for t in (m2, con, op, f)] + [torch.zeros_like(m2)]
    lane = torch.arange(TILE * TILE, device=DEV)
    k = 0
    while k < len(host):
        L = host[k]
        T = max(1, min(len(host) - k, 6_000_000 // (L * TILE * TILE * max(1, D // 8))))
        t, s, n = tiles[k:k + T], starts[k:k + T], counts[k:k + T]
        k += T
        slot = torch.arange(L, device=DEV)
        real = slot[None] < n[:, None]
        g = listed_rows[torch.where(real, s[:, None] + slot[None], s[:, None])]
        px = (t % tw * TILE)[:, None] + lane % TILE + 0.5
        py = (t // tw * TILE)[:, None] + lane // TILE + 0.5
        dx = m2[g][..., 0, None] - px[:, None]
        dy = m2[g][..., 1, None] - py[:, None]
        qa, qb, qc = (con[g][..., i, None] for i in range(3))
        with torch.set_grad_enabled(back):
            sig = (0.5 * (qa * dx * dx + qc * dy * dy) + qb * dx * dy).requires_grad_(back)
            og = op[g].requires_grad_(back)
            fg = f[g].requires_grad_(back)
            alpha = (og[..., None] * torch.exp(-sig)).clamp(max=0.99)
            with torch.no_grad():
                on = real[..., None] & (sig >= 0) & (alpha >= 1 / 255)
            alpha = torch.where(on, alpha, 0.0)
            after = torch.cumprod(1 - alpha, dim=1)
            with torch.no_grad():
                on = after > 1e-4
            alpha = torch.where(on, alpha, 0.0)
            after = torch.cumprod(1 - alpha, dim=1)
            before = torch.cat([torch.ones_like(after[:, :1]), after[:, :-1]], dim=1)
            weight = alpha * before
            left = after[:, -1]
            part = torch.stack([(weight * fg[..., i, None]).sum(dim=1) for i in range(D)], -1)
            part = part + left[..., None] * bg
            cover = 1 - left
            if c["mode"] in ("ED", "RGB+ED"):
                part = torch.cat([part[..., :-1], part[..., -1:] / cover.clamp(min=1e-10)[..., None]],
                                 dim=-1)
            rc[t], ra[t] = part.detach(), cover.detach()
            if not back:
                continue
            loss = (part * up[t]).sum()
            if upa is not None:
                loss = loss + (cover * upa[t]).sum()
            vs, vo, vf = torch.autograd.grad(loss, [sig, og, fg])
        ux, uy = vs * (qa * dx + qb * dy), vs * (qb * dx + qc * dy)
        flat = g.reshape(-1)
        grads[0].index_add_(0, flat, torch.stack([ux.sum(-1), uy.sum(-1)], -1).view(-1, 2))
        grads[1].index_add_(0, flat, torch.stack(
            [0.5 * (vs * dx * dx).sum(-1), (vs * dx * dy).sum(-1),
             0.5 * (vs * dy * dy).sum(-1)], -1).view(-1, 3))
        grads[2].index_add_(0, flat, torch.where(real, vo, 0.0).view(-1))
        grads[3].index_add_(0, flat, vf.reshape(-1, D))
        if absgrad:
            grads[4].index_add_(0, flat, torch.stack([ux.abs().sum(-1), uy.abs().sum(-1)],
                                                     -1).view(-1, 2))
    return untiled(rc), untiled(ra[..., None]), grads


def _scene64(c, p, views, Ks, bg, v_rc, v_ra, back, absgrad=False):
    """All cameras of one scene: renders, alphas, gradients of p, and the
    densification statistics (None without absgrad)."""
    leaves = {k: v.detach().double().requires_grad_(back) for k, v in p.items()}
    views, Ks = views.double(), Ks.double()
    total = {k: torch.zeros_like(v) for k, v in leaves.items()} if back else None
    n = p["means"].shape[0]
    stats = [torch.zeros(n, dtype=torch.float64, device=DEV) for _ in range(2)] if absgrad else None
    rcs, ras = [], []
    for i in range(c["cameras"]):
        with torch.set_grad_enabled(back):
            ids, m2, con, z, op, ext = _project64(c, leaves, views[i], Ks[i])
            f = _features64(c, leaves, views[i], ids, z)
        b = None
        if bg is not None:
            b = bg[i].double()
            if c["mode"] in ("D", "ED"):
                b = None
            elif c["mode"] != "RGB":
                b = torch.cat([b, b.new_zeros(1)])
        rows = [t.detach() for t in (m2, con, op, f, ext, z)]
        rc, ra, grads = _composite64(c, rows, b, None if not back else v_rc[i],
                                     None if v_ra is None else v_ra[i], back, absgrad)
        rcs.append(rc)
        ras.append(ra)
        if back:
            got = torch.autograd.grad([m2, con, op, f], list(leaves.values()), grads[:4],
                                      allow_unused=True)
            for k, v in zip(leaves, got):
                if v is not None:
                    total[k] += v
        if absgrad:
            scale = torch.tensor([c["width"] / 2.0, c["height"] / 2.0], dtype=torch.float64,
                                 device=DEV) * c["cameras"]
            stats[0].index_add_(0, ids, (grads[4] * scale).norm(dim=-1))
            stats[1].index_add_(0, ids, torch.ones_like(grads[2]))
    return torch.stack(rcs), torch.stack(ras), total, stats


def _adam64(raw, moments, grads, visible):
    out = {}
    for k, p in raw.items():
        m, v, g, p = moments[k][0].double(), moments[k][1].double(), grads[k].double(), p.double()
        m1 = _BETAS[0] * m + (1 - _BETAS[0]) * g
        v1 = _BETAS[1] * v + (1 - _BETAS[1]) * g * g
        p1 = p - _LRS[k] * m1 / (v1.sqrt() + _EPS)
        if visible is not None:
            see = visible.view(-1, *[1] * (p.dim() - 1))
            p1, m1, v1 = (torch.where(see, a, b) for a, b in ((p1, p), (m1, m), (v1, v)))
        out[k] = {"param": p1, "exp_avg": m1, "exp_avg_sq": v1}
    return out


def exact(case, seed):
    c = case
    if c["kind"] == "adam":
        return _adam64(*_adam_inputs(c, seed))
    if c["kind"] == "step":
        raw, moments, g = _optimizer_state(c, seed)
        views, Ks = _cameras(c)
        v_rc, _ = _loss_grads(c, g)
        leaves = {k: v.double().requires_grad_() for k, v in raw.items()}
        p = {"means": leaves["means"], "quats": leaves["quats"],
             "scales": leaves["log_scales"].exp(), "opacities": torch.sigmoid(leaves["logits"]),
             "colors": torch.cat([leaves["sh0"], leaves["shN"]], dim=1)
             if "shN" in leaves else leaves["sh0"]}
        rc, ra, total, stats = _scene64(c, p, views.to(DEV), Ks.to(DEV), None, v_rc, None, True,
                                        absgrad=True)
        got = torch.autograd.grad(list(p.values()), list(leaves.values()),
                                  [total[k] for k in p])
        groups = _adam64(raw, moments, dict(zip(leaves, got)), None)
        return {"colors": rc, "alphas": ra, "grad2d": stats[0], "count": stats[1],
                "groups": groups}
    params, views, Ks, bg, g = _inputs(c, seed)
    if c["mode"] in ("D", "ED"):
        params.pop("colors")
    back = c["kind"] != "render"
    v_rc, v_ra = _loss_grads(c, g) if back else (None, None)
    if c["batch"] == 1:
        rc, ra, grads, _ = _scene64(c, params, views, Ks, bg, v_rc, v_ra, back)
    else:
        each = [_scene64(c, {k: v[b] for k, v in params.items()}, views[b], Ks[b],
                         None if bg is None else bg[b], None if v_rc is None else v_rc[b],
                         None if v_ra is None else v_ra[b], back)[:3]
                for b in range(c["batch"])]
        rc, ra = (torch.stack([e[i] for e in each]) for i in range(2))
        grads = {k: torch.stack([e[2][k] for e in each]) for k in params} if back else None
    out = {"colors": rc, "alphas": ra}
    if back:
        out["grads"] = grads
    return out
