"""Workloads of the framework, through its public entry points, over the sizes
that its users give it.

``listed()`` is the fixed list, ``draw(rng)`` one more case of the same ranges.
``prepare`` makes what a program holds before the call (inputs from the seed,
the renderer, plan or layer it keeps), ``run`` is one pass, ``work`` the bytes
and operations that the pass cannot do without, and ``exact`` the same outputs
in 64 bits by plain torch.

Kinds of case
  eval        Microfacet.eval without a gradient: the re-renders written at
              every save point and any preview.
  eval_grad   Microfacet.eval and its adjoint on a given dL/dimages: what a
              loss composed in torch asks of the renderer; optionally the
              light power's gradient too, and lights apart from the cameras.
  fit         FusedStep.run: iterations of the per-pixel optimisation, the
              framework's main loop.
  optim       SvbrdfOptim.optim, the whole call a driver makes: from maps and
              photos to optimised maps and the list of losses.
  batch       BatchedStep: a graph of iterations over materials of uneven size.
  stage       the transition between two resolutions: the 8-bit maps' round
              trip with the Lanczos-4 resize, and the bilinear one in memory.
  conv        a frozen 3x3 layer of the VGG feature loss: forward, or dL/dx
              with the ReLU gate.
  modconv     a modulated 3x3 layer of the generator: forward with noise, bias
              and leaky ReLU, and dL/dx, dL/dweight, dL/dstyle of it.
  features    the VGG feature vector of a set of images.
  synthesis   the generator's maps from a latent and its noise.

Layers are measured one by one in the backward direction, on a given output
and a given gradient: through a stack of ReLUs the gradient is not a
continuous function of the rounding.
"""
import math

import numpy as np
import torch
import torch.nn.functional as F

from __graft_entry__ import load_package

DEV = "cuda"
SIZE = 17.0             # plane side, cm
EPS = 1e-6
BETAS, ADAM_EPS = (0.9, 0.999), 1e-8
STYLE_STD = 0.3
VGG_FLOPS_PLAN = [(3, 64, 1), (64, 64, 1), (64, 128, 2), (128, 128, 2), (128, 256, 4), (256, 256, 4), (256, 256, 4),
                  (256, 256, 4), (256, 512, 8), (512, 512, 8)]


def listed():
    return [
        # a preview render at the size MaterialGAN and the first stage work at
        {"name": "eval_256x9", "kind": "eval", "res": 256, "views": 9, "apart": False},
        # the renderer inside a composed loss, at the full map size
        {"name": "eval_grad_1024x9", "kind": "eval_grad", "res": 1024, "views": 9, "apart": False, "light": False},
        # the first (coarse) stage of a fit: 256 x 256 maps, 9 photos
        {"name": "fit_256x9_logl2", "kind": "fit", "res": 256, "views": 9, "loss": "log_l2", "steps": 10},
        # the last stage, the framework's headline configuration
        {"name": "fit_1024x9_logl2", "kind": "fit", "res": 1024, "views": 9, "loss": "log_l2", "steps": 10},
        # a short run of the whole optimisation call, light power included
        {"name": "optim_512x9_light", "kind": "optim", "res": 512, "views": 9, "loss": "l2", "steps": 50,
         "light": True},
        # materials of uneven size and view count stepping together
        {"name": "batch_6", "kind": "batch", "materials": "256x9,512x9,333x5,384x12,768x9,1024x4", "steps": 5},
        # coarse-to-fine: the maps go from 512 to 1024
        {"name": "stage_512_1024", "kind": "stage", "res": 512, "to": 1024},
        # conv1_2 of the feature loss on the 9 re-renders, the costliest layer shape of the stack
        {"name": "conv_64_64_256_fwd", "kind": "conv", "n": 9, "cin": 64, "cout": 64, "h": 256, "w": 256,
         "grad": False},
        # the input gradient of conv3_2
        {"name": "conv_256_256_64_dx", "kind": "conv", "n": 9, "cin": 256, "cout": 256, "h": 64, "w": 64,
         "grad": True},
        # the generator's 512-channel layer at 32 x 32, both directions
        {"name": "modconv_512_512_32", "kind": "modconv", "cin": 512, "cout": 512, "side": 32},
        # the feature vector of the 9 re-renders
        {"name": "features_256x9", "kind": "features", "n": 9, "side": 256},
        # latent and noise to maps
        {"name": "synthesis_256", "kind": "synthesis", "res": 256},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["eval", "eval_grad", "fit", "fit", "optim", "batch", "stage", "conv", "conv", "modconv",
                       "features"])
    res = _log_int(rng, 40, 1024)
    views = rng.randint(1, 12)
    if kind == "eval":
        return {"kind": kind, "res": res, "views": views, "apart": rng.random() < 0.3}
    if kind == "eval_grad":
        return {"kind": kind, "res": res, "views": views, "apart": rng.random() < 0.3, "light": rng.random() < 0.4}
    if kind == "fit":
        return {"kind": kind, "res": res, "views": views, "loss": rng.choice(["l2", "log_l2"]),
                "steps": rng.randint(3, 12)}
    if kind == "optim":
        return {"kind": kind, "res": min(res, 700), "views": views, "loss": rng.choice(["l2", "log_l2"]),
                "steps": rng.randint(8, 50), "light": rng.random() < 0.5}
    if kind == "batch":
        n = rng.randint(2, 8)
        return {"kind": kind, "steps": rng.randint(2, 5),
                "materials": ",".join(f"{_log_int(rng, 48, 768)}x{rng.randint(1, 12)}" for _ in range(n))}
    if kind == "stage":
        r = _log_int(rng, 64, 600)
        return {"kind": kind, "res": r, "to": 2 * r}
    if kind == "conv":
        while True:
            c = {"kind": kind, "n": rng.randint(1, 9), "cin": _log_int(rng, 3, 512), "cout": _log_int(rng, 16, 512),
                 "h": _log_int(rng, 6, 256), "w": _log_int(rng, 6, 256), "grad": rng.random() < 0.5}
            if rng.random() < 0.5:      # the stack's own channel counts, on square images
                c["cin"], c["cout"] = rng.choice([(64, 64), (64, 128), (128, 128), (128, 256), (256, 512), (512, 512)])
                c["w"] = c["h"]
            if work(c)["flops"] <= 4.4e10:
                return c
    if kind == "modconv":
        side = _log_int(rng, 4, 160)
        cin = min(512, rng.choice([512, 256, 128, 96]), 32768 // side)
        return {"kind": kind, "cin": cin, "cout": rng.choice([cin, max(32, cin // 2)]), "side": side}
    return {"kind": "features", "n": rng.randint(1, 9), "side": _log_int(rng, 32, 250)}


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _smooth(g, channels, res, cells, amount):
    """Smooth random maps: noise on a coarse grid, interpolated."""
    a = torch.randn((1, channels, cells, cells), generator=g, device=DEV)
    return F.interpolate(a, size=(res, res), mode="bicubic", align_corners=True) * amount


def _maps(g, res):
    """[1, 9, R, R] maps in [-1, 1]: smooth normals, coloured albedos with
    per-texel detail, roughness over its usual range."""
    cells = max(4, min(res, 24))
    detail = torch.rand((1, 9, res, res), generator=g, device=DEV)
    base = torch.rand((9,), generator=g, device=DEV)
    t = torch.empty((1, 9, res, res), device=DEV)
    t[:, 0:3] = 0.1 + 0.6 * base[0:3].view(1, 3, 1, 1) + 0.2 * detail[:, 0:3]
    t[:, 5] = 0.2 + 0.4 * base[5] + 0.3 * detail[:, 5]
    t[:, 6:9] = 0.02 + 0.15 * base[6:9].view(1, 3, 1, 1) + 0.1 * detail[:, 6:9]
    t = t * 2 - 1
    t[:, 3:5] = _smooth(g, 2, res, cells, 0.15).clamp(-0.8, 0.8)
    return t


def _flash(g, views, apart):
    """Cameras on the 3 x 3 flash grid, repeated and jittered; the light at
    the camera, or a few cm beside it."""
    grid = torch.tensor([[x, y, 30.0] for y in (8.0, 0.0, -8.0) for x in (-8.0, 0.0, 8.0)], device=DEV)
    cam = grid[torch.arange(views, device=DEV) % 9].clone()
    cam[:, :2] += torch.rand((views, 2), generator=g, device=DEV) * 2 - 1
    light = cam.clone()
    if apart:
        light[:, :2] += torch.rand((views, 2), generator=g, device=DEV) * 4 - 2
    return cam, light, torch.full((3,), 1500.0, device=DEV)


def _photos(maps, cl):
    """8-bit photos of the maps, as floats in [0, 1]."""
    with torch.no_grad():
        return (_render(maps, *cl) * 255).round() / 255


def _problem(g, res, views, apart=False):
    truth = _maps(g, res)
    cl = _flash(g, views, apart)
    start = (truth + 0.1 * torch.randn(truth.shape, generator=g, device=DEV)).clamp(-1, 1)
    return start, _photos(truth, cl), cl


def _materials(case):
    return [tuple(int(v) for v in m.split("x")) for m in case["materials"].split(",")]


def _conv_inputs(case, g):
    n, ci, co, h, w = (case[k] for k in ("n", "cin", "cout", "h", "w"))
    weight = torch.randn((co, ci, 3, 3), generator=g, device=DEV) * math.sqrt(2.0 / (ci * 9))
    bias = 0.1 * torch.randn((co,), generator=g, device=DEV)
    if not case["grad"]:
        # activations behind a ReLU (conv1_1 reads normalised colours)
        x = torch.randn((n, ci, h, w), generator=g, device=DEV)
        return weight, bias, x if ci == 3 else x.relu()
    y = torch.randn((n, co, h, w), generator=g, device=DEV).relu()
    return weight, y, 1e-4 * torch.randn((n, co, h, w), generator=g, device=DEV)


def _modconv_inputs(case, g):
    ci, co, s = case["cin"], case["cout"], case["side"]
    rnd = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    x = F.leaky_relu(rnd(1, ci, s, s), 0.2) * math.sqrt(2.0)
    return {"x": x, "style": 1.0 + STYLE_STD * rnd(1, ci), "weight": rnd(co, ci, 3, 3),
            "scale": 1.0 / math.sqrt(ci * 9), "bias": 0.1 * rnd(co), "noise": rnd(1, 1, s, s), "strength": 0.1,
            "gz": 1e-3 * rnd(1, co, s, s)}


def prepare(case, seed):
    pkg = load_package()
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("eval", "eval_grad"):
        cl = _flash(g, case["views"], case["apart"])
        s = {"maps": _maps(g, case["res"]), "cl": cl,
             "renderer": pkg.Microfacet(case["res"], case["views"], SIZE, list(cl), DEV)}
        if kind == "eval_grad":
            # dL/dimages of a mean over all pixels
            s["grad"] = torch.randn((case["views"], 3, case["res"], case["res"]), generator=g, device=DEV)
            s["grad"] /= s["grad"].numel()
            s["maps"].requires_grad_(True)
            if case["light"]:
                s["renderer"].update_light(cl[2].clone().requires_grad_(True))
    elif kind in ("fit", "optim"):
        start, photos, cl = _problem(g, case["res"], case["views"])
        r = pkg.Microfacet(case["res"], case["views"], SIZE, list(cl), DEV)
        if kind == "fit":
            s = {"step": pkg.FusedStep(r, start, photos, 0.01, loss=case["loss"], history=case["steps"],
                                       own_textures=True)}
        else:
            s = {"optim": pkg.SvbrdfOptim(DEV, r), "renderer": r}
            s["optim"].init_from_tex(start)
            s["optim"].load_targets(photos)
    elif kind == "batch":
        problems = []
        for res, views in _materials(case):
            start, photos, cl = _problem(g, res, views)
            problems.append((pkg.Microfacet(res, views, SIZE, list(cl), DEV), start, photos))
        s = {"batch": pkg.BatchedStep(problems, 0.01, loss="log_l2", own_textures=True)}
        s["batch"].capture(case["steps"])
    elif kind == "stage":
        s = {"maps": _maps(g, case["res"]), "pkg": pkg}
    elif kind == "conv":
        s = {"convnet": pkg.materialgan.convnet}
        weight, a, b = _conv_inputs(case, g)
        if case["grad"]:
            s.update(layer=s["convnet"].Conv3x3(weight), y=a, gy=b)
        else:
            s.update(layer=s["convnet"].Conv3x3(weight, a), x=b)
    elif kind == "modconv":
        s = dict(_modconv_inputs(case, g), convnet=pkg.materialgan.convnet)
    elif kind == "features":
        s = {"net": pkg.materialgan.VGGLoss(torch.device(DEV), np.array([1, 1, 4, 8]) / 14),
             "images": torch.rand((case["n"], 3, case["side"], case["side"]), generator=g, device=DEV)}
    else:
        net = pkg.materialgan.StyleGAN2Generator(case["res"], 9, seed=7, device=DEV)
        s = {"net": net, "noises": [torch.randn((1, 1, r, r), generator=g, device=DEV) for r in net.conv_res],
             "latent": torch.randn((1, net.num_layers, 512), generator=g, device=DEV)}
    s["case"] = case
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "eval":
        with torch.no_grad():
            return s["renderer"].eval(s["maps"])
    if kind == "eval_grad":
        images = s["renderer"].eval(s["maps"])
        wrt = [s["maps"]] + ([s["renderer"].light_pow] if case["light"] else [])
        return [images.detach(), *torch.autograd.grad(images, wrt, s["grad"])]
    if kind == "fit":
        f = s["step"]
        f.run(case["steps"])
        f.flush()
        return [f.textures, f.exp_avg, f.exp_avg_sq, f.history]
    if kind == "optim":
        o = s["optim"]
        losses = o.optim(case["steps"], 0.01, optim_light=case["light"], loss=case["loss"])
        return [o.textures.detach(), torch.tensor(losses), s["renderer"].light_pow]
    if kind == "batch":
        s["batch"].replay()
        return [*s["batch"].textures, s["batch"].losses_dev]
    if kind == "stage":
        pkg = s["pkg"]
        return [pkg.reload_textures(s["maps"], case["to"]), pkg.upsample_textures(s["maps"])]
    if kind == "conv":
        if case["grad"]:
            layer = s["layer"]
            return s["convnet"].conv3x3_input_grad(s["gy"], s["y"], layer.packed_t, layer.cin, layer.act)
        with torch.no_grad():
            return s["layer"](s["x"])
    if kind == "modconv":
        c, cin, cout = s["convnet"], case["cin"], case["cout"]
        with torch.no_grad():
            y = c.modulated_conv3x3(s["x"], s["style"], s["weight"], s["scale"], True, s["bias"], s["noise"],
                                    s["strength"], "lrelu")
            packed_t = c.pack3x3(s["weight"], s["style"], s["scale"], True, transpose=True)
            gx = c.conv3x3_packed(s["gz"], packed_t, cin)
            gw = c.conv3x3_wgrad(s["x"], s["gz"], cout)
            gs = c.modulation_grad(s["weight"], s["style"], s["scale"], True, gw)
        return [y, gx, gw, gs]
    with torch.no_grad():
        if kind == "features":
            return s["net"].compute_feature_vector(s["net"].normalize(s["images"]))
        return s["net"].synthesis(s["latent"], s["noises"])


# ---------------------------------------------------------------- work
def _vgg(n, side):
    """(values of activations written, weights, flops) of the stack to relu4_2."""
    acts = weights = flops = 0
    for cin, cout, f in VGG_FLOPS_PLAN:
        hw = n * (side // f) ** 2
        acts += cout * hw
        weights += 9 * cin * cout
        flops += 18 * cin * cout * hw
    return acts, weights, flops


def work(case):
    kind = case["kind"]
    if kind == "stage":
        src, dst = case["res"] ** 2, case["to"] ** 2
        return {"bytes": 2 * 36 * (src + dst), "flops": 2 * 9 * 40 * dst}
    if kind == "conv":
        n, ci, co, hw = case["n"], case["cin"], case["cout"], case["h"] * case["w"]
        values = n * hw * (ci + co + (co if case["grad"] else 0)) + 9 * ci * co
        return {"bytes": 4 * values, "flops": 18 * n * hw * ci * co}
    if kind == "modconv":
        ci, co, hw = case["cin"], case["cout"], case["side"] ** 2
        return {"bytes": 4 * (hw * (2 * ci + 2 * co) + 2 * 9 * ci * co), "flops": 3 * 18 * hw * ci * co}
    if kind == "features":
        acts, weights, flops = _vgg(case["n"], case["side"])
        n, s = case["n"], case["side"]
        out = n * (2 * 64 * s * s + 256 * (s // 4) ** 2 + 512 * (s // 8) ** 2)
        return {"bytes": 4 * (3 * n * s * s + weights + out), "flops": flops}
    if kind == "synthesis":
        nf = lambda r: min(32768 // r, 512)  # noqa: E731
        weights, flops, r = 9 * 512 * 512, 18 * 512 * 512 * 16, 8
        while r <= case["res"]:
            for ci in (nf(r // 2), nf(r)):
                weights += 9 * ci * nf(r)
                flops += 18 * ci * nf(r) * r * r
            r *= 2
        return {"bytes": 4 * (weights + 9 * case["res"] ** 2), "flops": flops}
    if kind == "batch":
        px = [(r * r, v) for r, v in _materials(case)]
        return {"bytes": case["steps"] * sum(p * (216 + 12 * v) for p, v in px),
                "flops": case["steps"] * sum(p * (400 + 170 * v) for p, v in px)}
    p, v = case["res"] ** 2, case["views"]
    if kind == "eval":
        return {"bytes": p * (36 + 12 * v), "flops": p * (60 + 80 * v)}
    if kind == "eval_grad":
        return {"bytes": p * (108 + 24 * v), "flops": p * (200 + 230 * v)}
    return {"bytes": case["steps"] * p * (216 + 12 * v), "flops": case["steps"] * p * (400 + 170 * v)}


# ---------------------------------------------------------------- in 64 bits
def _render(maps, cam, light, power):
    """The microfacet render of maps [1, 9, R, R] in their own precision."""
    dt, res = maps.dtype, maps.shape[-1]
    t = ((torch.arange(res, dtype=torch.float32, device=maps.device) + 0.5) / res - 0.5) * SIZE
    t = t.to(dt)
    yy, xx = torch.meshgrid(t, t, indexing="ij")
    pos = torch.stack((xx, -yy, torch.zeros_like(xx)))[None]
    cam, light, power = (a.to(dt) for a in (cam, light, power))
    lin = lambda a: ((a + 1) / 2) ** 2.2  # noqa: E731
    dif, rough, spe = lin(maps[:, 0:3]), lin(maps[:, 5:6]), lin(maps[:, 6:9])
    nx, ny = maps[:, 3:4].clamp(-1, 1), maps[:, 4:5].clamp(-1, 1)
    # 1 - 1e-6 is a number of the maps' precision here; it only binds for normals at the horizon
    nz = (1 - (nx ** 2 + ny ** 2).clamp(0, 1 - EPS)).sqrt()
    unit = lambda a: a / a.norm(dim=1, keepdim=True)  # noqa: E731
    dot = lambda a, b: (a * b).sum(1, keepdim=True)  # noqa: E731
    nrm = unit(torch.cat((nx, ny, nz), 1))
    out = []
    for k in range(cam.shape[0]):
        to_cam, to_light = cam[k].view(1, 3, 1, 1) - pos, light[k].view(1, 3, 1, 1) - pos
        v, l = unit(to_cam), unit(to_light)
        h = unit(v + l)
        nv, nl, nh, vh = (dot(*p).clamp(min=0) for p in ((nrm, v), (nrm, l), (nrm, h), (v, h)))
        alpha = rough ** 2
        c2, a2, kk = nh ** 2, alpha ** 2, alpha / 2 + EPS
        ggx = a2 / (math.pi * (c2 * a2 + (1 - c2)) ** 2 + EPS)
        fres = spe + (1 - spe) * torch.pow(2.0, (-5.55473 * vh - 6.98316) * vh)
        smith = (nv / (nv * (1 - kk) + kk)) * (nl / (nl * (1 - kk) + kk))
        f = dif / math.pi * (1 - spe) + ggx * fres * smith / (4 * nv * nl + EPS)
        img = power.view(1, 3, 1, 1) * f * nl / dot(to_light, to_light)
        out.append(img.clamp(EPS, 1) ** (1 / 2.2))
    return torch.cat(out)


def _fit64(start, photos, cl, steps, loss, light):
    """Adam on the maps (and the light power) in 64 bits."""
    maps, target = start.double(), photos.double()
    cam, lpos, power = cl[0].double(), cl[1].double(), cl[2].double()
    if loss == "log_l2":
        target = target.clamp(EPS ** (1 / 2.2), 1).log()
    params = [maps] + ([power] if light else [])
    params = [p.clone().requires_grad_(True) for p in params]
    m = [torch.zeros_like(p) for p in params]
    v = [torch.zeros_like(p) for p in params]
    losses = []
    for k in range(1, steps + 1):
        total, n = 0.0, target.numel()
        grads = [torch.zeros_like(p) for p in params]
        for i in range(cam.shape[0]):      # view by view, to bound the graph's memory
            out = _render(params[0].clamp(-1, 1), cam[i:i + 1], lpos[i:i + 1], params[1] if light else power)
            out = out.log() if loss == "log_l2" else out
            part = ((out - target[i:i + 1]) ** 2).sum() / n
            total += float(part.detach())
            for a, b in zip(grads, torch.autograd.grad(part, params)):
                a += b
        losses.append(total)
        with torch.no_grad():
            for p, g, a, b in zip(params, grads, m, v):
                a.mul_(BETAS[0]).add_(g, alpha=1 - BETAS[0])
                b.mul_(BETAS[1]).addcmul_(g, g, value=1 - BETAS[1])
                denom = b.sqrt() / math.sqrt(1 - BETAS[1] ** k) + ADAM_EPS
                p.addcdiv_(a, denom, value=-0.01 / (1 - BETAS[0] ** k))
    return [p.detach() for p in params], m, v, losses


def _conv64(x, weight):
    return torch.cat([F.conv2d(x[i:i + 1].double(), weight.double(), padding=1) for i in range(x.shape[0])])


def _up64(x):
    """x2 by zero insertion and the [1, 3, 3, 1] filter per axis, gain 4."""
    f = torch.tensor([1.0, 3.0, 3.0, 1.0], dtype=torch.float64, device=x.device) / 4
    k = (f.view(4, 1) * f.view(1, 4)).view(1, 1, 4, 4)
    n, c, h, w = x.shape
    z = torch.zeros((n * c, 1, 2 * h, 2 * w), dtype=x.dtype, device=x.device)
    z[:, :, ::2, ::2] = x.reshape(n * c, 1, h, w)
    return F.conv2d(F.pad(z, (2, 1, 2, 1)), k).view(n, c, 2 * h, 2 * w)


def _modulate64(weight, style, scale, demodulate=True):
    w = weight.double() * scale * style.double().reshape(1, -1, 1, 1)
    return w * torch.rsqrt((w * w).sum(dim=(1, 2, 3), keepdim=True) + 1e-8) if demodulate else w


def _lrelu64(x):
    return F.leaky_relu(x, 0.2) * math.sqrt(2.0)


def exact(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "eval":
        cl = _flash(g, case["views"], case["apart"])
        return _render(_maps(g, case["res"]).double(), *cl)
    if kind == "eval_grad":
        s = prepare(case, seed)
        maps = s["maps"].detach().double().requires_grad_(True)
        power = s["cl"][2].double().requires_grad_(True)
        images, grads = [], [torch.zeros_like(maps), torch.zeros_like(power)]
        for i in range(case["views"]):
            out = _render(maps, s["cl"][0][i:i + 1], s["cl"][1][i:i + 1], power)
            images.append(out.detach())
            for a, b in zip(grads, torch.autograd.grad(out, [maps, power], s["grad"][i:i + 1].double())):
                a += b
        return [torch.cat(images), *grads[:2 if case["light"] else 1]]
    if kind == "fit":
        params, m, v, losses = _fit64(*_problem(g, case["res"], case["views"]), case["steps"], case["loss"], False)
        return [params[0], m[0], v[0], torch.tensor(losses, dtype=torch.float64)]
    if kind == "optim":
        start, photos, cl = _problem(g, case["res"], case["views"])
        params, _, _, losses = _fit64(start, photos, cl, case["steps"], case["loss"], case["light"])
        return [params[0], torch.tensor(losses, dtype=torch.float64), params[1] if case["light"] else cl[2].double()]
    if kind == "batch":
        maps, last = [], []
        for res, views in _materials(case):
            params, _, _, losses = _fit64(*_problem(g, res, views), case["steps"], "log_l2", False)
            maps.append(params[0])
            last.append(losses[-1])
        return [*maps, torch.tensor(last, dtype=torch.float64)]
    if kind == "stage":
        # the 8-bit route is whole numbers by nature; the bilinear one is computed
        up = F.interpolate(_maps(g, case["res"]).double(), scale_factor=2, mode="bilinear", align_corners=False)
        return [None, up]
    if kind == "conv":
        weight, a, b = _conv_inputs(case, g)
        if case["grad"]:
            return _conv64(b * (a > 0), weight.flip(2, 3).transpose(0, 1))
        return (_conv64(b, weight) + a.double().view(1, -1, 1, 1)).relu()
    if kind == "modconv":
        i = _modconv_inputs(case, g)
        s = case["side"]
        w = _modulate64(i["weight"], i["style"], i["scale"])
        y = _lrelu64(_conv64(i["x"], w) + i["strength"] * i["noise"].double() + i["bias"].double().view(1, -1, 1, 1))
        gx = _conv64(i["gz"], w.flip(2, 3).transpose(0, 1))
        # dL/dweight: one product over the pixels per tap
        xp, gz = F.pad(i["x"][0].double(), (1, 1, 1, 1)), i["gz"][0].double().flatten(1)
        taps = [gz @ xp[:, a:a + s, b:b + s].flatten(1).t() for a in range(3) for b in range(3)]
        gw = torch.stack(taps, -1).view(case["cout"], case["cin"], 3, 3)
        style = i["style"].double().requires_grad_(True)
        (gs,) = torch.autograd.grad(_modulate64(i["weight"], style, i["scale"]), style, gw)
        return [y, gx, gw, gs.flatten()]
    if kind == "features":
        net = prepare(case, seed)
        x = net["images"].double()
        x = (x - net["net"].mean.double()) / net["net"].std.double()
        feats, k = [], 0
        for item in net["net"].plan:
            if item == "P":
                x = F.avg_pool2d(x, 2)
                continue
            x = _conv64(x, net["net"].convs[item].weight).relu()
            if item in net["net"].HOOKS:
                feats.append(x.flatten() * net["net"].weights[k])
                k += 1
        return torch.cat(feats)
    s = prepare(case, seed)
    net, ws = s["net"], s["latent"].double()[0]
    x, rgb, wi = net.const.double(), None, 0
    style = lambda conv, w: w @ conv.affine.weight.double().t() * conv.affine.scale + conv.affine.bias.double()  # noqa: E731
    for i, conv in enumerate(net.convs):
        x = _up64(x) if conv.upsample else x
        x = _conv64(x, _modulate64(conv.weight, style(conv, ws[min(wi, net.num_layers - 1)]), conv.scale))
        x = _lrelu64(x + net.noise_strength[i].double() * s["noises"][i].double())
        wi += 1
        if i % 2 == 0:
            rgb_conv = net.to_rgb[(i + 1) // 2]
            w = _modulate64(rgb_conv.weight, style(rgb_conv, ws[min(wi, net.num_layers - 1)]), rgb_conv.scale, False)
            t = F.conv2d(x, w)
            rgb = t if rgb is None else _up64(rgb) + t
    return rgb
