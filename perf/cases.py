"""What a user of this framework has it do, as cases that can be timed.

Seven kinds, each through the package's public entry points:

  render   Context.render: one whole frame (warmup, draws, density
           estimation, tonemap) with the image on the host.
  draw     FlameHandle.draw_to_bins into a histogram that lives on the GPU,
           the loop of an offline render or of a progressive preview.
  density  Context.density_tonemap of a finished histogram.
  display  Context.tonemap and Context.rgba8 of a float image: what a viewer
           repeats when the gamma or the brightness is changed.
  batch    Batch.run and the images of an animation's frames.
  denoise  denoise_histogram: the U-Net on a low-sample histogram.
  train    Denoiser.train_step over a few batches, then the weights.

A flame's structure (its variations, post-affines, final xform) comes from
the case's "flame" number and its coefficients from the input seed, as in an
animation or an editor, where values change and the structure stays.
"""
import math

import numpy as np
import torch

import refrakt_amd as rf
from refrakt_amd import configs
from refrakt_amd.denoise import WEIGHTS, denoise_histogram, load_weights

SCALE = 1e-4          # the tonemap's density scale, Context.render's default
FUSE = 19             # warmup passes after the first run


# ------------------------------------------------------------------ cases
def listed():
    return [
        # the editor's thumbnail: the smallest call, where launches and host work count
        {"name": "render_thumbnail", "kind": "render", "width": 320, "height": 240, "particles": 1 << 14, "temporal": 1,
         "passes": 16, "calls": 1, "flame": 11, "motion": False, "radius": 9},
        # one frame of an animation with motion blur at full HD, 65 samples per pixel
        {"name": "render_hd_motion", "kind": "render", "width": 1920, "height": 1080, "particles": 1 << 20,
         "temporal": 512, "passes": 64, "calls": 2, "flame": 5030, "motion": True, "radius": 9},
        # a progressive preview's next step: one pass, one sample per pixel
        {"name": "draw_preview", "kind": "draw", "width": 2048, "height": 2048, "particles": 1 << 22, "temporal": 1,
         "passes": 1, "flame": 5070, "family": "random", "opacity": 1.0},
        # one call of the full-size offline render: 3840x2160 at supersample 2
        {"name": "draw_8k", "kind": "draw", "width": 7680, "height": 4320, "particles": 1 << 24, "temporal": 512,
         "passes": 16, "flame": 2, "family": "cfg2", "opacity": 1.0},
        # a flame some of whose xforms are translucent or hidden (flam3's opacity)
        {"name": "draw_translucent", "kind": "draw", "width": 1920, "height": 1080, "particles": 1 << 22,
         "temporal": 512, "passes": 16, "flame": 5030, "family": "random", "opacity": 0.5},
        # a concentrated attractor in a large frame: nearly every sample in a few hundred bins
        {"name": "draw_contention", "kind": "draw", "width": 8192, "height": 8192, "particles": 1 << 24,
         "temporal": 512, "passes": 16, "flame": 3, "family": "cfg3", "opacity": 1.0},
        # the full-size accumulator with the usual estimator
        {"name": "density_8k", "kind": "density", "width": 7680, "height": 4320, "radius": 9, "rmin": 0, "curve": 0.4,
         "spp": 8.0},
        # a wide estimator on an odd-sized frame of few samples
        {"name": "density_wide", "kind": "density", "width": 1919, "height": 1083, "radius": 24, "rmin": 0,
         "curve": 0.45, "spp": 2.0},
        # a viewer's gamma slider on a 4K image
        {"name": "display_4k", "kind": "display", "width": 3840, "height": 2160},
        # sixteen animation frames of uneven size in one replay
        {"name": "batch_animation", "kind": "batch", "frames": 16, "flame": 4, "density": 0.125, "mode": rf.RF_HIST_SORT,
         "iters": 256},
        # the denoised preview of a 2048x2048 frame
        {"name": "denoise_2k", "kind": "denoise", "width": 2048, "height": 2048, "spp": 4.0},
        # training as the package's own training loop runs it: 8 crops of 256x256 per step
        {"name": "train_8x256", "kind": "train", "batch": 8, "crop": 256, "steps": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["render", "draw", "draw", "density", "density", "display", "batch", "denoise", "train"])
    if kind == "render":
        w = _log_int(rng, 200, 1920)
        motion = rng.random() < 0.5
        return {"kind": kind, "width": w, "height": max(120, int(w * rng.uniform(0.5, 0.5625))),
                "particles": 1 << rng.randint(14, 20), "temporal": rng.choice([1, 16, 32]) if motion else 1,
                "passes": rng.randint(8, 64), "calls": rng.randint(1, 2), "flame": rng.randint(1, 9999),
                "motion": motion, "radius": rng.choice([0, 5, 9, 9, 11])}
    if kind == "draw":
        family = rng.choice(["random", "random", "random", "cfg1", "cfg3"])
        w = _log_int(rng, 512, 4096)
        return {"kind": kind, "width": w, "height": max(256, int(w * rng.uniform(0.5, 1.0))),
                "particles": 1 << rng.randint(18, 24), "temporal": 1, "passes": _log_int(rng, 1, 16),
                "flame": rng.randint(1, 9999), "family": family,
                "opacity": 0.5 if family == "random" and rng.random() < 0.35 else 1.0}
    if kind == "density":
        wide = rng.random() < 0.5
        w = _log_int(rng, 256, 1900 if wide else 6000)
        r = rng.randint(16, 24) if wide else rng.randint(0, 15)
        return {"kind": kind, "width": w, "height": max(200, int(w * rng.uniform(0.5, 0.5625))), "radius": r,
                "rmin": rng.choice([0, 0, 0, 1, 2]), "curve": round(rng.uniform(0.3, 0.6), 3),
                "spp": round(math.exp(rng.uniform(math.log(2.0), math.log(8.0))), 2)}
    if kind == "display":
        w = _log_int(rng, 300, 3840)
        return {"kind": kind, "width": w, "height": max(200, int(w * rng.uniform(0.5, 0.5625)))}
    if kind == "batch":
        lds = rng.random() < 0.3
        return {"kind": kind, "frames": rng.randint(3, 12), "flame": rng.randint(1, 9999),
                "density": round(rng.uniform(0.02, 0.12), 3), "mode": rf.RF_HIST_LDS if lds else rf.RF_HIST_SORT,
                "iters": 64 if lds else rng.choice([64, 256])}
    if kind == "denoise":
        w = 8 * _log_int(rng, 32, 256)
        return {"kind": kind, "width": w, "height": 8 * max(8, int(w / 8 * rng.uniform(0.5, 1.0))),
                "spp": round(math.exp(rng.uniform(0.0, math.log(32.0))), 2)}
    return {"kind": kind, "batch": rng.randint(1, 8), "crop": 8 * rng.randint(8, 32), "steps": rng.randint(2, 8)}


# ----------------------------------------------------------------- inputs
def _edit(flame, rng, xforms=None):
    """New coefficients for a flame of the same structure."""
    for x in xforms if xforms is not None else flame.xforms:
        x.affine = [float(v * rng.uniform(0.97, 1.03)) for v in x.affine]
        x.color = float(rng.uniform(0.0, 1.0))
        x.weight = float(x.weight * rng.uniform(0.9, 1.1))
    flame.palette = configs.smooth_palette(rng)
    return flame


def _flame(family, number, size, seed):
    structure = np.random.Generator(np.random.PCG64(number))
    if family == "random":
        f = configs.random_flame(structure, 1024)
    else:
        f = {"cfg1": configs.cfg1, "cfg2": configs.cfg2, "cfg3": configs.cfg3}[family](number).flame
    view = f.size[1] / f.scale  # view height in flame units
    f = _edit(f, np.random.Generator(np.random.PCG64([seed, number])))
    f.size, f.scale = list(size), size[1] / view
    return f


def _set_opacity(flame, opacity):
    """Every second xform translucent, and one of five hidden."""
    for i, x in enumerate(flame.xforms):
        x.opacity = 0.0 if i % 5 == 4 else opacity * (0.8 + 0.1 * (i % 3)) if i % 2 == 0 else 1.0


def _histogram(width, height, spp, seed):
    """A flame-like RGBA histogram (height, width, 4) from a plain chaos game
    of four bent affine maps: integer counts, colours that sum palette entries."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = np.random.Generator(np.random.PCG64([seed, width, height]))
    maps = [(configs._rot_scale(r, 0.45, 0.8), r.uniform(-1, 1, 2), r.uniform(0, 1), r.uniform(0.2, 0.9))
            for _ in range(4)]
    pal = torch.as_tensor(np.round(configs.smooth_palette(r)[:, :3] * 4096).astype(np.int32), device="cuda")
    n = 1 << 20
    steps = max(1, int(round(spp * width * height / n)))
    p = torch.rand((n, 3), generator=g, device="cuda", dtype=torch.float32) * 2 - 1
    count = torch.zeros(width * height, dtype=torch.int32, device="cuda")
    rgb = torch.zeros((width * height, 3), dtype=torch.int32, device="cuda")
    ones = torch.ones(n, dtype=torch.int32, device="cuda")
    scale = height / 3.2
    coef = torch.tensor([[*m[0], *m[1], m[2], m[3]] for m in maps], dtype=torch.float32, device="cuda")
    for k in range(16 + steps):
        c = coef[torch.randint(0, 4, (n,), generator=g, device="cuda")]
        x = c[:, 0] * p[:, 0] + c[:, 2] * p[:, 1] + c[:, 4]
        y = c[:, 1] * p[:, 0] + c[:, 3] * p[:, 1] + c[:, 5]
        bend = c[:, 7]
        p = torch.stack([x + bend * 0.3 * torch.sin(2 * y), y + bend * 0.3 * torch.sin(2 * x),
                         0.5 * (p[:, 2].abs() + c[:, 6])], 1)
        if k < 16:
            continue
        ix = torch.floor(p[:, 0] * scale + width / 2).long()
        iy = torch.floor(p[:, 1] * scale + height / 2).long()
        ok = (ix >= 0) & (ix < width) & (iy >= 0) & (iy < height)
        b = (iy * width + ix)[ok]
        count.index_add_(0, b, ones[:b.numel()])
        rgb.index_add_(0, b, pal[(p[:, 2][ok] * 255).long().clamp(0, 255)])
    h = torch.empty((height, width, 4), dtype=torch.float32, device="cuda")
    h[..., :3] = rgb.view(height, width, 3).float() / 4096
    h[..., 3] = count.view(height, width).float()
    return h


def _training_images(batch, crop, seed):
    """Network input and target (batch, crop, crop, 16 and 16 channels, bf16):
    smooth log-densities seen at a few samples per pixel, and at a thousand."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    c = max(2, crop // 16)
    field = torch.randn((batch, 4, c, c), generator=g, device="cuda")
    field = torch.nn.functional.interpolate(field, size=(crop, crop), mode="bilinear", align_corners=False)
    rate = torch.exp(1.5 * field).permute(0, 2, 3, 1)
    spp = torch.exp(torch.rand((batch, 1, 1, 1), generator=g, device="cuda") * math.log(32.0))
    x = torch.zeros((batch, crop, crop, 16), device="cuda")
    t = torch.zeros_like(x)
    x[..., :4] = torch.log10(1 + torch.poisson(rate * spp, generator=g) / spp)
    x[..., 4:5] = torch.log10(1 + 1 / spp)
    t[..., :4] = torch.log10(1 + torch.poisson(rate * 1024, generator=g) / 1024)
    return x.to(torch.bfloat16), t.to(torch.bfloat16)


# the network's layers: input and output channels, ReLU
LAYERS = [(16, 32, 1), (32, 32, 1), (32, 64, 1), (64, 64, 1), (64, 128, 1), (128, 128, 1), (128, 256, 1),
          (384, 128, 1), (192, 64, 1), (96, 32, 1), (32, 32, 1), (32, 16, 0)]
LR = 1e-4


def _initial_weights(seed):
    """He initialisation, the last layer small: a network near the identity."""
    r = np.random.Generator(np.random.PCG64([seed, 7]))
    parts = []
    for k, (cin, cout, _) in enumerate(LAYERS):
        s = math.sqrt(2.0 / (9 * cin)) * (0.1 if k == len(LAYERS) - 1 else 1.0)
        parts += [r.normal(0.0, s, 9 * cin * cout), np.zeros(cout)]
    return np.concatenate(parts).astype(np.float32)


def _tonemap_params():
    return rf.TonemapParams(2.2, 4.0, 0.8, SCALE)


def _batch_frames(case, seed):
    frames = configs.cfg4(case["flame"], case["frames"])
    r = np.random.Generator(np.random.PCG64([seed, case["flame"]]))
    out = []
    for f in frames:
        out.append((_edit(f.flame, r), f.width, f.height, max(1, int(f.samples * case["density"]))))
    return out


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "render":
        w, h = case["width"], case["height"]
        f = _flame("random", case["flame"], (w, h), seed)
        if case["motion"]:
            for i, x in enumerate(f.xforms):
                x.rotation_frequency = 1.0 - 0.5 * (i % 3)
        s["ctx"] = rf.Context(case["particles"], case["temporal"], 64, seed=seed)
        s["flame"] = s["ctx"].flame(f)
        s["params"] = rf.RenderParams(w, h, FUSE, case["passes"], case["calls"], 1.2 / 60.0, int(case["radius"] > 0),
                                      rf.DEParams(case["radius"], 0, 0.4), _tonemap_params())
    elif kind == "draw":
        w, h = case["width"], case["height"]
        f = _flame(case["family"], case["flame"], (w, h), seed)
        if case["opacity"] != 1.0:
            _set_opacity(f, case["opacity"])
        s["ctx"] = rf.Context(case["particles"], case["temporal"], 64, seed=seed)
        s["flame"] = s["ctx"].flame(f)
        s["bins"] = torch.zeros((h, w, 4), dtype=torch.float32, device="cuda")
        s["hist"] = s["ctx"].histogram(w, h, s["bins"].data_ptr())
        s["flame"].warmup(FUSE)
    elif kind == "density":
        s["ctx"] = rf.Context(1 << 12, 1, 16, seed=seed)
        s["bins"] = _histogram(case["width"], case["height"], case["spp"], seed)
        s["hist"] = s["ctx"].histogram(case["width"], case["height"], s["bins"].data_ptr())
        s["de"] = rf.DEParams(case["radius"], case["rmin"], case["curve"])
        s["tm"] = _tonemap_params()
        s["image"] = torch.empty_like(s["bins"])
    elif kind == "display":
        s["ctx"] = rf.Context(1 << 12, 1, 16, seed=seed)
        s["density"] = _histogram(case["width"], case["height"], 8.0, seed)
        s["tm"] = _tonemap_params()
        s["image"] = torch.empty_like(s["density"])
        s["bytes"] = torch.empty(s["density"].shape, dtype=torch.uint8, device="cuda")
    elif kind == "batch":
        s["ctx"] = rf.Context(1 << 12, 1, 16, seed=seed)
        s["batch"] = s["ctx"].batch(_batch_frames(case, seed))
        s["batch"].set_config(8, case["mode"], case["iters"], 20)
    elif kind == "denoise":
        w, h = case["width"], case["height"]
        s["ctx"] = rf.Context(1 << 12, 1, 16, seed=seed)
        s["net"] = s["ctx"].denoiser(1)
        load_weights(s["net"])
        s["bins"] = _histogram(w, h, case["spp"], seed)
        s["samples"] = int(s["bins"][..., 3].double().sum())
        s["x"] = torch.empty((1, h, w, 16), dtype=torch.bfloat16, device="cuda")
        s["y"] = torch.empty((1, h, w, 4), dtype=torch.float32, device="cuda")
    else:
        s["ctx"] = rf.Context(1 << 12, 1, 16, seed=seed)
        s["net"] = s["ctx"].denoiser(1)
        s["net"].set_params(_initial_weights(seed))
        s["data"] = [_training_images(case["batch"], case["crop"], 100 * seed + k) for k in range(case["steps"])]
    return s


# ------------------------------------------------------------------- pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "render":
        _, image, stats = s["ctx"].render(s["flame"], s["params"], want_hist=False)
        return {"image": image, "drawn": int(stats.drawn)}
    if kind == "draw":
        drawn = s["flame"].draw_to_bins(s["hist"], case["passes"])
        return {"bins": s["bins"], "drawn": int(drawn)}
    if kind == "density":
        s["ctx"].density_tonemap(s["hist"], s["de"], s["tm"], s["image"].data_ptr())
        return {"image": s["image"]}
    if kind == "display":
        w, h = case["width"], case["height"]
        s["ctx"].tonemap(s["density"].data_ptr(), s["image"].data_ptr(), w, h, s["tm"])
        s["ctx"].rgba8(s["image"].data_ptr(), s["bytes"].data_ptr(), w, h)
        return {"image": s["image"], "bytes": s["bytes"]}
    if kind == "batch":
        b = s["batch"]
        b.run()
        return {"images": [b.image(i) for i in range(case["frames"])],
                "drawn": b.frame_stats()["drawn"].astype(np.int64)}
    if kind == "denoise":
        return {"y": denoise_histogram(s["ctx"], s["net"], s["bins"].data_ptr(), case["width"], case["height"],
                                       s["samples"], s["x"], s["y"])}
    n, c = case["batch"], case["crop"]
    loss = None
    for k, (x, t) in enumerate(s["data"]):
        loss = s["net"].train_step(x.data_ptr(), t.data_ptr(), n, c, c, LR, want_loss=k == case["steps"] - 1)
    return {"loss": loss, "weights": s["net"].params()}


# ------------------------------------------------------------------- work
# one chaos-game iteration: an affine, a handful of variations of about
# fifteen operations each, a post-affine, the colour and the screen affine
OPS_PER_ITERATION = 100
NET_FLOPS = 2 * 9 * sum(ci * co / 4 ** l for (ci, co, _), l in zip(LAYERS, (0, 0, 1, 1, 2, 2, 3, 2, 1, 0, 0, 0)))


def _disc(r):
    """Average taps per texel an estimator of radius r cannot do without: one disc per source."""
    return math.pi * r * r / 4 + 1


def work(case):
    kind = case["kind"]
    if kind == "render":
        px, p = case["width"] * case["height"], case["particles"]
        n = p * (FUSE + 1 + case["passes"] * case["calls"])
        return {"bytes": 16 * px, "flops": n * OPS_PER_ITERATION + 8 * px * _disc(case["radius"])}
    if kind == "draw":
        px, p = case["width"] * case["height"], case["particles"]
        n = p * case["passes"]
        if case["family"] == "cfg3":
            px //= 100  # its attractor covers well under a hundredth of the frame
        return {"bytes": 32 * min(px, n) + 24 * p, "flops": n * OPS_PER_ITERATION}
    if kind == "density":
        px = case["width"] * case["height"]
        return {"bytes": 32 * px, "flops": 8 * px * _disc(case["radius"])}
    if kind == "display":
        px = case["width"] * case["height"]
        return {"bytes": 36 * px, "flops": 60 * px}
    if kind == "batch":
        fr = configs.cfg4(case["flame"], case["frames"])
        px = sum(f.width * f.height for f in fr)
        n = sum(int(f.samples * case["density"]) for f in fr)
        return {"bytes": 16 * px, "flops": n * OPS_PER_ITERATION + 8 * px * _disc(9)}
    if kind == "denoise":
        px = case["width"] * case["height"]
        return {"bytes": 32 * px, "flops": px * NET_FLOPS}
    px = case["batch"] * case["crop"] ** 2
    n = sum(9 * ci * co + co for ci, co, _ in LAYERS)
    return {"bytes": case["steps"] * (64 * px + 24 * n) + 4 * n, "flops": 3 * case["steps"] * px * NET_FLOPS}


# ------------------------------------------------------------------ exact
def _f32(v):
    return float(np.float32(v))


def _tonemap64(v):
    g, b, vib, k = (_f32(x) for x in (2.2, 4.0, 0.8, SCALE))
    a = v[..., 3]
    some = a > 0
    ls = torch.where(some, 0.5 * b * torch.log1p(a * k) / math.log(10.0) / torch.where(some, a, 1.0), 0.0)
    v = v * ls[..., None]
    z = torch.where(some, v[..., 3], 1.0)
    gf = z ** (1 / g) / z
    rgb = v[..., :3]
    o = rgb.clamp_min(0) ** (1 / g) * (1 - vib) + gf[..., None] * rgb * vib
    out = torch.ones_like(v)
    out[..., :3] = torch.where(some[..., None], o.clamp(0, 1), 0.0)
    return out


def _density64(h, radius, rmin, curve):
    """The estimator as a gather: each bin a sprite of its own radius."""
    H, W, _ = h.shape
    v = torch.zeros((H, W, 4), dtype=torch.float64, device=h.device)
    # bin (px, py) is centred on texel (px - 1, H - 1 - py); column 0 is dropped
    v[:, :W - 1] = h.flip(0)[:, 1:].double()
    a = v[..., 3]
    q = radius / torch.where(a > 0, a, 1.0) ** _f32(curve)
    r = torch.where(a > 0, torch.clamp(torch.floor(q).clamp(max=radius), min=rmin), -1.0)
    span = max(radius, rmin)
    S = 2 * r + 1
    norm = torch.where(r > 0, (2 / math.pi) / torch.where(r > 0, r * r, 1.0), 0.0)
    out = torch.where((r == 0)[..., None], v, 0.0)
    for i in range(-span, span + 1):
        ny2 = ((2 * i + 1 / S) / S) ** 2
        for j in range(-span, span + 1):
            if i * i + j * j > (span + 1) ** 2:
                continue
            d = ((2 * j + 1 / S) / S) ** 2 + ny2
            w = torch.where((r >= max(abs(i), abs(j))) & (r > 0) & (d <= 1), (1 - d) * norm, 0.0)
            y0, y1, x0, x1 = max(0, -i), min(H, H - i), max(0, -j), min(W, W - j)
            if y1 <= y0 or x1 <= x0:
                continue
            out[y0 + i:y1 + i, x0 + j:x1 + j] += v[y0:y1, x0:x1] * w[y0:y1, x0:x1, None]
    return out


def _conv64(x, w, b, relu):
    """x (N, H, W, Cin), w (3, 3, Cout, Cin): nine shifted products."""
    n, h, wd, ci = x.shape
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    y = b.expand(n * h * wd, -1)
    for r in range(3):
        for s in range(3):
            y = y + p[:, r:r + h, s:s + wd].reshape(-1, ci) @ w[r, s].t().contiguous()
    y = y.view(n, h, wd, -1)
    return torch.relu(y) if relu else y


def _net64(params, x):
    ls, off = [], 0
    for ci, co, relu in LAYERS:
        w = params[off:off + 9 * ci * co].view(3, 3, co, ci)
        off += 9 * ci * co
        ls.append((w, params[off:off + co], relu))
        off += co

    def conv(k, t):
        return _conv64(t, *ls[k])

    def pool(t):
        n, h, w, c = t.shape
        return t.view(n, h // 2, 2, w // 2, 2, c).mean((2, 4))

    def up(t):
        return t.repeat_interleave(2, 1).repeat_interleave(2, 2)

    e0 = conv(1, conv(0, x))
    e1 = conv(3, conv(2, pool(e0)))
    e2 = conv(5, conv(4, pool(e1)))
    d2 = conv(7, torch.cat([up(conv(6, pool(e2))), e2], 3))
    d1 = conv(8, torch.cat([up(d2), e1], 3))
    d0 = conv(10, conv(9, torch.cat([up(d1), e0], 3)))
    return x[..., :4] + conv(11, d0)[..., :4]


def exact(case, seed):
    kind = case["kind"]
    if kind == "density":
        h = _histogram(case["width"], case["height"], case["spp"], seed)
        return {"image": _tonemap64(_density64(h, case["radius"], case["rmin"], case["curve"]))}
    if kind == "display":
        return {"image": _tonemap64(_histogram(case["width"], case["height"], 8.0, seed).double()), "bytes": None}
    if kind == "denoise":
        h = _histogram(case["width"], case["height"], case["spp"], seed).double()
        scale = case["width"] * case["height"] / int(h[..., 3].sum())
        x = torch.zeros((1, case["height"], case["width"], 16), dtype=torch.float64, device="cuda")
        x[0, ..., :4] = torch.log10(1 + h * scale)
        x[..., 4] = math.log10(1 + scale)
        with np.load(WEIGHTS, allow_pickle=False) as z:
            p = torch.as_tensor(z["params"], device="cuda").double()
        with torch.no_grad():
            return {"y": _net64(p, x)[0]}
    if kind == "train":
        p = torch.as_tensor(_initial_weights(seed), device="cuda").double().requires_grad_(True)
        m, v, loss = torch.zeros_like(p), torch.zeros_like(p), None
        for k in range(case["steps"]):
            x, t = _training_images(case["batch"], case["crop"], 100 * seed + k)
            e = ((_net64(p, x.double()) - t[..., :4].double()) ** 2).mean()
            (g,) = torch.autograd.grad(e, p)
            loss = float(e)
            with torch.no_grad():
                m = 0.9 * m + 0.1 * g
                v = 0.999 * v + 0.001 * g * g
                p -= LR * (m / (1 - 0.9 ** (k + 1))) / (torch.sqrt(v / (1 - 0.999 ** (k + 1))) + 1e-8)
        return {"loss": loss, "weights": p.detach().clone()}
    return None  # the chaos game amplifies every rounding: its outputs have no 64-bit value to hold them to
