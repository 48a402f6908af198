"""Performance cases of the Gaussian-splat rasterizer and its training step.

Each case is one call sequence that a program using this package makes per
frame or per training step, through the public entry points
``gaussian_splats_hip.splats.rasterize`` / ``rasterize_views`` and
``gaussian_splats_hip.training``.  The workloads are this repository's own
configurations (``gaussian_splats_hip/scenes.py``), its trajectory benchmark's
defaults and generic sizes between them.  ``exact`` restates the same functions
in float64 with plain torch operations.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = Path(__file__).resolve().parents[1] / "gaussian-splats_amd"
if str(_PACKAGE) not in sys.path:
    sys.path.insert(0, str(_PACKAGE))

PARAMS = ("mean", "rotation", "scale", "opacity", "color")

# Weights and learning rates of the training step (those of bench.py's
# --train-step: L1 + 0.2 D-SSIM + two regularisers, Adam).
LAMBDA_DSSIM, OPACITY_REG, SCALE_REG = 0.2, 1e-2, 1e-2
RATES = {"mean": 1.6e-4, "rotation": 1e-3, "scale": 5e-3, "opacity": 5e-2, "color": 2.5e-3}


def _case(name, kind, scene, n, sh, width, height, tile=None, mode="gaussian", near=0.2, views=1,
          subset=False):
    """``tile`` None leaves the entry point's default tile size; ``subset``
    renders a seeded half of the Gaussians through ``indices``."""
    case = {"kind": kind, "scene": scene, "n": n, "sh": sh, "width": width, "height": height,
            "tile": tile, "mode": mode, "near": near, "views": views, "subset": subset}
    return {"name": name, **case} if name else case


def listed():
    return [
        # The smallest call: one preview frame of a toy scene (config 1).
        _case("preview frame", "render", "ball", 10_000, 0, 256, 256, tile=16, near=0.01),
        # A viewer's frame with the entry point's default arguments: the
        # trajectory benchmark's scene and image.
        _case("viewer frame", "render", "slab", 10_000, 1, 640, 480),
        # The same benchmark's forward + backward of a mean square.
        _case("viewer step", "step", "slab", 10_000, 1, 640, 480),
        # A small fit at an odd size: early training, few Gaussians, SH 2.
        _case("small odd step", "step", "cloud", 20_011, 2, 403, 307, tile=8),
        # The viewer's ellipsoid display of an evenly drawn subset, default tile.
        _case("ellipsoid subset", "render", "cloud", 200_000, 3, 1272, 716, mode="ellipsoid",
              subset=True),
        # A full-HD frame (config 2).
        _case("frame 1080p", "render", "cloud", 200_000, 3, 1920, 1080, tile=16),
        # A full-HD step of the same scene with the default arguments.
        _case("default step 1080p", "step", "cloud", 200_000, 3, 1920, 1080),
        # The headline training step (config 3).
        _case("step 1080p 1M", "step", "cloud", 1_000_000, 3, 1920, 1080, tile=16),
        # Very long lists: 4M Gaussians in a small cube (config 4).
        _case("dense step 4M", "step", "dense", 4_000_000, 3, 1600, 1600, tile=16),
        # A baked mesh seen by 16 cameras in one batch (config 5).
        _case("mesh step 16 views", "step", "shell", 500_000, 3, 800, 800, tile=16, views=16),
        # A whole optimisation step: render, L1 + SSIM + regularisers,
        # backward, Adam; a ragged image.
        _case("optimisation step", "train", "cloud", 300_000, 3, 1237, 822, tile=16),
        # The image losses alone, forward + backward, on a ragged image.
        _case("image losses", "loss", "none", 0, 0, 1297, 840),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["render", "render", "step", "step", "step", "train", "loss"])
    width = _log_int(rng, 200, 1920)
    height = max(64, min(1600, int(width * rng.uniform(0.5, 1.1))))
    if kind == "loss":
        return _case(None, kind, "none", 0, 0, width, height)
    scene = rng.choice(["ball", "slab", "cloud", "cloud", "cloud", "dense", "shell"])
    tile = rng.choice([None, 4, 8, 16, 16, 16, 32])
    views, most = 1, 800_000
    if scene == "slab":
        most = 40_000
    elif scene == "ball":
        most = 30_000
    elif scene == "dense":
        tile = rng.choice([16, 16, 32])
    elif scene == "shell" and kind != "train":
        views = rng.choice([1, 2, 3, 4, 6, 8])
        width, height = min(width, 900), min(height, 900)
        most = 200_000
    if views > 1 and tile is not None:
        tile = rng.choice([8, 16, 16, 32])
    mode = "ellipsoid" if kind == "render" and rng.random() < 0.25 else "gaussian"
    subset = kind == "render" and rng.random() < 0.3
    return _case(None, kind, scene, _log_int(rng, 3_000, most), rng.choice([0, 1, 2, 3, 3]), width,
                 height, tile=tile, mode=mode, near=rng.choice([0.01, 0.2]), views=views,
                 subset=subset)


# ---------------------------------------------------------------------------
# Inputs.
# ---------------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _parameters(case, g):
    """The five float32 parameter tensors of the case's scene (the
    distributions of scenes.py and of the trajectory benchmark)."""
    n, k = case["n"], (case["sh"] + 1) ** 2

    def randn(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    def rand(*shape):
        return torch.rand(*shape, generator=g, device="cuda")

    scene = case["scene"]
    rotation = randn(n, 4)
    rotation = rotation / rotation.norm(dim=-1, keepdim=True).clamp_min(1e-12)
    color = torch.cat((randn(n, 1, 3) * 0.5, randn(n, k - 1, 3) * 0.05), 1)
    if scene == "ball":
        mean, scale, opacity = rand(n, 3) * 2 - 1, randn(n, 3) * 0.5 - 3, randn(n, 1)
    elif scene == "slab":
        mean = torch.cat((randn(n, 2) * 0.5, rand(n, 1) * 4 + 2), 1)
        # The benchmark's isotropic e^-2 with the spread that fitting gives.
        scale, opacity = randn(n, 3) * 0.3 - 2, randn(n, 1)
    elif scene == "cloud":
        mean = randn(n, 3) * torch.tensor([2.0, 1.0, 2.0], device="cuda")
        scale, opacity = randn(n, 3) * 0.7 - 4, randn(n, 1) * 1.5
    elif scene == "dense":
        mean, scale, opacity = rand(n, 3) * 0.5 - 0.25, randn(n, 3) * 0.5 - 3.5, randn(n, 1) - 1
    else:  # "shell": flat splats on the unit sphere, the thin axis turned to a random normal
        mean = randn(n, 3)
        mean = mean / mean.norm(dim=-1, keepdim=True).clamp_min(1e-12)
        scale = randn(n, 3) * 0.3 - 4
        scale[:, 2] = -9.2
        normal = randn(n, 3)
        normal = normal / normal.norm(dim=-1, keepdim=True).clamp_min(1e-12)
        x, y, z = normal.unbind(-1)
        rotation = torch.stack((1 + z, -y, x, torch.zeros_like(z)), -1)
        rotation = rotation / rotation.norm(dim=-1, keepdim=True).clamp_min(1e-6)
        opacity = randn(n, 1) * 1.5
    return tuple(t.contiguous() for t in (mean, rotation, scale, opacity, color))


def _cameras(case, seed):
    """The case's cameras: scenes.py's distance and focal length per scene,
    at a seeded place on a ring (a viewer's or a trainer's next camera)."""
    from gaussian_splats_hip.splats import PinholeCamera

    w, h, views = case["width"], case["height"], case["views"]
    # Distance, focal length per pixel of width, target, elevation.
    distance, focal, target, lift = {
        "ball": (3.0, 1.0, (0.0, 0.0, 0.0), 0.0),
        "slab": (8.6, 0.75, (0.0, 0.0, 4.0), math.pi / 4),
        "cloud": (6.0, 1500 / 1920, (0.0, 0.0, 0.0), 0.0),
        "dense": (3.0, 1.0, (0.0, 0.0, 0.0), 0.0),
        "shell": (3.0, 1.25, (0.0, 0.0, 0.0), 0.0),
    }[case["scene"]]
    f = float(focal * w)
    start = 0.1 * (seed % 61)
    cameras = []
    for v in range(views):
        angle = 0.3 * math.sin(start) + 2 * math.pi * v / views
        position = (target[0] + distance * math.cos(lift) * math.sin(angle),
                    target[1] + distance * math.sin(lift),
                    target[2] + distance * math.cos(lift) * math.cos(angle))
        cameras.append(PinholeCamera.look_at(
            position, target, image_size=(w, h), focal_length=(f, f),
            principal_point=(w / 2, h / 2)))
    return cameras


def _images(case, g):
    shape = (case["height"], case["width"], 3)
    if case["views"] > 1:
        shape = (case["views"], *shape)
    return torch.rand(*shape, generator=g, device="cuda")


def _loss_inputs(case, g):
    """A rendered-looking image (it leaves [0, 1] at places, as renders do)
    and the photograph it is compared with."""
    target = _images(case, g)
    image = target + 0.1 * torch.randn(*target.shape, generator=g, device="cuda") + 0.02
    return image, target


def _draw_subset(case, g):
    if not case["subset"]:
        return None
    return torch.randperm(case["n"], generator=g, device="cuda")[: max(1, case["n"] // 2)]


def prepare(case, seed):
    g = _generator(seed)
    if case["kind"] == "loss":
        image, target = _loss_inputs(case, g)
        return {"case": case, "image": image.requires_grad_(True), "target": target}

    from gaussian_splats_hip.splats import GaussianSplat
    from gaussian_splats_hip.training import FusedAdam

    splats = GaussianSplat.from_tensors(*_parameters(case, g))
    state = {"case": case, "splats": splats, "cameras": _cameras(case, seed),
             "indices": _draw_subset(case, g)}
    options = {"near": case["near"]}
    if case["tile"] is not None:
        options["tile_size"] = case["tile"]
    if case["mode"] != "gaussian":
        options["rendering_mode"] = case["mode"]
    state["options"] = options
    if case["kind"] in ("step", "train"):
        state["target"] = _images(case, g)
    if case["kind"] == "train":
        state["optimizer"] = FusedAdam(
            [{"params": [getattr(splats, name)], "lr": rate} for name, rate in RATES.items()],
            eps=1e-15)
    return state


# ---------------------------------------------------------------------------
# One pass.
# ---------------------------------------------------------------------------


def _render(state):
    from gaussian_splats_hip.splats import rasterize, rasterize_views

    if state["case"]["views"] > 1:
        return rasterize_views(state["splats"], state["cameras"], indices=state["indices"],
                               **state["options"])
    return rasterize(state["splats"], state["cameras"][0], indices=state["indices"],
                     **state["options"])


def run(state):
    from gaussian_splats_hip.training import l1_loss, splat_regularizers, ssim

    case = state["case"]
    if case["kind"] == "render":
        with torch.no_grad():
            return {"image": _render(state)}
    if case["kind"] == "loss":
        image, target = state["image"], state["target"]
        image.grad = None
        loss = (1 - LAMBDA_DSSIM) * l1_loss(image, target, clamp=True)
        loss = loss + LAMBDA_DSSIM * (1 - ssim(image, target))
        loss.backward()
        return {"loss": loss.detach(), "grad": image.grad}
    splats, target = state["splats"], state["target"]
    params = [getattr(splats, name) for name in PARAMS]
    if case["kind"] == "step":
        for p in params:
            p.grad = None
        image = _render(state)
        loss = image.square().mean() if case["scene"] == "slab" else l1_loss(image, target)
        loss.backward()
        return {"image": image.detach(), "loss": loss.detach(),
                **{name: p.grad for name, p in zip(PARAMS, params)}}
    optimizer = state["optimizer"]
    image = _render(state)
    regs = splat_regularizers(splats.opacity, splats.scale)
    loss = ((1 - LAMBDA_DSSIM) * l1_loss(image, target, clamp=True)
            + LAMBDA_DSSIM * (1 - ssim(image.clamp(0, 1), target))
            + OPACITY_REG * regs[0] + SCALE_REG * regs[1])
    loss.backward()
    grads = {"grad_" + name: p.grad for name, p in zip(PARAMS, params)}
    optimizer.step()
    optimizer.zero_grad()
    return {"image": image.detach(), "loss": loss.detach(), **grads,
            **{name: p.detach() for name, p in zip(PARAMS, params)}}


# ---------------------------------------------------------------------------
# What a pass cannot do without.
# ---------------------------------------------------------------------------

# (Gaussian, pixel) pairs that change a pixel (alpha of 1/255 or more, in
# front of where the pixel saturates): the smaller of the Gaussians' footprints
# and this many per pixel, counted with the float64 code below on the listed
# sizes.
_PAIRS_PER_PIXEL = {"ball": 46.0, "slab": 8.0, "cloud": 52.0, "dense": 30.0, "shell": 74.0}
# Mean footprint (pixels with alpha >= 1/255) of a Gaussian, as a share of the
# squared focal length in pixels.
_FOOTPRINT = {"ball": 1.3e-2, "slab": 7.7e-3, "cloud": 1.25e-3, "dense": 3.6e-3, "shell": 7e-4}
# Floating operations per such pair: exponent, alpha and blend; its reverse;
# and per Gaussian and view: projection, covariance and colour.
_PAIR_FORWARD, _PAIR_BACKWARD = 20.0, 45.0
_GAUSSIAN_FORWARD, _GAUSSIAN_BACKWARD = 400.0, 1200.0


def work(case):
    pixels = case["width"] * case["height"] * case["views"]
    if case["kind"] == "loss":
        # Image and target in, image gradient out; the 11-tap separable
        # window over five moments forward and three maps backward.
        return {"bytes": 12.0 * pixels * 3, "flops": pixels * 3 * (5 + 3) * 2 * 11 * 2.0}
    n = case["n"] // 2 if case["subset"] else case["n"]
    params = n * 4.0 * (11 + 3 * (case["sh"] + 1) ** 2)
    focal = {"cloud": 1500 / 1920, "slab": 0.75, "shell": 1.25}.get(case["scene"], 1.0) * case["width"]
    pairs = min(n * case["views"] * _FOOTPRINT[case["scene"]] * focal * focal,
                pixels * _PAIRS_PER_PIXEL[case["scene"]])
    moved = params + 12.0 * pixels
    flops = pairs * _PAIR_FORWARD + n * case["views"] * _GAUSSIAN_FORWARD
    if case["kind"] != "render":
        # The target in, the parameter gradients out.
        moved += 12.0 * pixels + params
        flops += pairs * _PAIR_BACKWARD + n * case["views"] * _GAUSSIAN_BACKWARD
    if case["kind"] == "train":
        # Both moments in and out, the parameters out.
        moved += 5 * params
        flops += pixels * 3 * (5 + 3) * 2 * 11 * 2.0 + params / 4 * 12
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """32-bit sums over up to thousands of terms per value, and pairs whose
    alpha lies within rounding of the 1/255 cut (or of the ellipsoid's edge,
    where the full alpha appears at once) and may fall on either side of it.
    About four times the differences from ``exact``: images 1.2e-5 (ellipsoid
    5e-4), gradients up to 4.5e-4, up to 1.2e-3 in small scenes, where one such
    pair weighs more; losses 2e-7."""
    if case["kind"] == "loss":
        return {"rel": 1e-6, "max": 1e-4}
    if case["mode"] == "ellipsoid":
        return {"rel": 2e-3, "max": 0.9}
    if case["kind"] == "render":
        return {"rel": 5e-5, "max": 0.05}
    return {"rel": 4e-3 if case["n"] < 50_000 else 1.5e-3, "max": 0.9}


# ---------------------------------------------------------------------------
# The same functions in float64 with plain torch operations.
# ---------------------------------------------------------------------------


def _sh_basis(d, degree):
    x, y, z = d.unbind(-1)
    one = torch.ones_like(x)
    c = [math.sqrt(1 / (4 * math.pi)) * one]
    if degree > 0:
        k = math.sqrt(3 / (4 * math.pi))
        c += [-k * y, k * z, -k * x]
    if degree > 1:
        k = math.sqrt(15 / (4 * math.pi))
        c += [k * x * y, -k * y * z, math.sqrt(5 / (16 * math.pi)) * (2 * z * z - x * x - y * y),
              -k * x * z, k / 2 * (x * x - y * y)]
    if degree > 2:
        a = math.sqrt(35 / (32 * math.pi))
        b = math.sqrt(105 / (4 * math.pi))
        e = math.sqrt(21 / (32 * math.pi))
        c += [-a * y * (3 * x * x - y * y), b * x * y * z, -e * y * (4 * z * z - x * x - y * y),
              math.sqrt(7 / (16 * math.pi)) * z * (2 * z * z - 3 * x * x - 3 * y * y),
              -e * x * (4 * z * z - x * x - y * y), b / 2 * z * (x * x - y * y),
              -a * x * (x * x - 3 * y * y)]
    return torch.stack(c, -1)


def _rotation(q):
    q = q / q.norm(dim=-1, keepdim=True).clamp_min(1e-12)
    w, x, y, z = q.unbind(-1)
    return (1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
            2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
            2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y))


def _exact_project(params, camera, degree):
    """Per Gaussian: pixel mean, depth, inverse covariance, colour, opacity
    (differentiable) and the covariance's diagonal."""
    mean, rotation, scale, opacity, color = params
    r = [float(v) for v in _rotation(camera.rotation.detach().double().cpu())]
    t = [float(v) for v in camera.translation.detach().double().cpu()]
    (fx, fy), (cx, cy), (width, height) = camera.focal_length, camera.principal_point, camera.image_size
    mx, my, mz = mean.unbind(-1)
    px, py, pz = (r[3 * i] * mx + r[3 * i + 1] * my + r[3 * i + 2] * mz + t[i] for i in range(3))
    d = -pz
    dc = torch.where(d.abs() >= 1e-4, d, torch.copysign(torch.full_like(d, 1e-4), d))
    u, v = fx * px / d + cx, -fy * py / d + cy
    lim_x, lim_y = 1.3 * width / (2 * fx), 1.3 * height / (2 * fy)
    nx, ny = (px / dc).clamp(-lim_x, lim_x), (py / dc).clamp(-lim_y, lim_y)
    rows = []
    for j0, j2, base in ((fx / dc, fx * nx / dc, 0), (-fy / dc, -fy * ny / dc, 3)):
        w = [j0 * r[base + i] + j2 * r[6 + i] for i in range(3)]
        q = _rotation(rotation)
        s = scale.exp().unbind(-1)
        rows.append([(w[0] * q[i] + w[1] * q[3 + i] + w[2] * q[6 + i]) * s[i] for i in range(3)])
    c00 = sum(m * m for m in rows[0]) + 0.03
    c01 = sum(a * b for a, b in zip(*rows))
    c11 = sum(m * m for m in rows[1]) + 0.03
    det = c00 * c11 - c01 * c01
    centre = torch.tensor([-(r[i] * t[0] + r[3 + i] * t[1] + r[6 + i] * t[2]) for i in range(3)],
                          dtype=mean.dtype, device=mean.device)
    ray = centre - mean
    ray = ray / ray.norm(dim=-1, keepdim=True).clamp_min(1e-12)
    basis = _sh_basis(ray, degree)
    rgb = ((basis[..., None] * color).sum(-2) + 0.5).clamp_min(0)
    return (u, v, c11 / det, -c01 / det, c00 / det, rgb, opacity.sigmoid()[:, 0]), dc, c00, c11


_TILE = 16
_CHUNK = 128  # list entries composited at a time
_GROUP = 128  # tiles composited at a time
_MOST_ENTRIES = 20_000_000  # (Gaussian, 16-pixel tile) entries of one view: above, exact() is None


def _exact_lists(splat, depth, c00, c11, case):
    """Gaussians per 16-pixel tile in (depth, index) order: ids, starts, lengths."""
    u, v, _, _, _, _, opacity = splat
    w, h = case["width"], case["height"]
    visible = (depth > case["near"]) & (depth < 100.0) & (opacity >= 1 / 255)
    if case["mode"] == "ellipsoid":
        reach = torch.full_like(depth, -2 * math.log1p(-0.95))
    else:
        reach = 2 * (opacity * 255).clamp_min(1).log()
    ex, ey = (reach * c00).sqrt() + 1e-3, (reach * c11).sqrt() + 1e-3
    visible &= (u + ex >= 0) & (u - ex <= w - 1) & (v + ey >= 0) & (v - ey <= h - 1)
    order = depth.float().argsort(stable=True)
    order = order[visible[order]]
    tw, th = -(-w // _TILE), -(-h // _TILE)

    def span(c, e, size, tiles):
        lo = ((c - e)[order].clamp(0, size - 1) / _TILE).floor().long()
        hi = ((c + e)[order].clamp(0, size - 1) / _TILE).floor().long().clamp(max=tiles - 1)
        return lo, hi - lo + 1

    x0, nx = span(u, ex, w, tw)
    y0, ny = span(v, ey, h, th)
    counts = nx * ny
    total = int(counts.sum())
    if total > _MOST_ENTRIES:
        return None
    owner = torch.repeat_interleave(torch.arange(len(order), device=u.device), counts)
    local = torch.arange(total, device=u.device) - (counts.cumsum(0) - counts)[owner]
    tile = (y0[owner] + local // nx[owner]) * tw + x0[owner] + local % nx[owner]
    tile, place = tile.sort(stable=True)
    ids = order[owner[place]]
    lengths = torch.bincount(tile, minlength=tw * th)
    return ids, lengths.cumsum(0) - lengths, lengths, tw


def _chunk_terms(splat, ids, valid, px, py, ellipsoid):
    """alpha of G tiles x L entries x P pixels and what its gradient needs."""
    u, v, a, b, c, _, opacity = (f[ids] for f in splat)
    dx = px[:, None, :] - u[..., None]
    dy = py[:, None, :] - v[..., None]
    form = a[..., None] * dx * dx + 2 * b[..., None] * dx * dy + c[..., None] * dy * dy
    if ellipsoid:
        fall = (form <= -2 * math.log1p(-0.95)).double()
    else:
        fall = (-0.5 * form).exp()
    raw = opacity[..., None] * fall
    alpha = raw.clamp_max(0.99)
    alpha = torch.where((alpha >= 1 / 255) & valid[..., None], alpha, torch.zeros_like(alpha))
    return alpha, raw, fall, dx, dy


def _exact_composite(splat, lists, case, grad_of=None):
    """The image; with ``grad_of(image)`` (the loss's gradient) also the
    gradients of the seven projected quantities."""
    ids, starts, lengths, tw = lists
    w, h = case["width"], case["height"]
    ellipsoid = case["mode"] == "ellipsoid"
    device = lengths.device
    splat = tuple(f.detach() for f in splat)
    color = splat[5]
    image = torch.zeros(h, w, 3, dtype=torch.float64, device=device)
    tiles = lengths.argsort(descending=True)
    tiles = tiles[lengths[tiles] > 0]
    q = torch.arange(_TILE * _TILE, device=device)
    groups = []
    for g in tiles.split(_GROUP):
        x = (g % tw * _TILE)[:, None] + q % _TILE
        y = (g // tw * _TILE)[:, None] + q // _TILE
        inside = (x < w) & (y < h)
        px, py = x.double(), y.double()
        T = inside.double()
        acc = torch.zeros(*T.shape, 3, dtype=torch.float64, device=device)
        saved = []
        for first in range(0, int(lengths[g].max()), _CHUNK):
            if not bool((T > 1 - 0.999).any()):
                break
            j = first + torch.arange(_CHUNK, device=device)
            valid = j < lengths[g][:, None]
            entry = ids[(starts[g][:, None] + j).clamp(max=len(ids) - 1)]
            alpha = _chunk_terms(splat, entry, valid, px, py, ellipsoid)[0]
            after = T[:, None] * (1 - alpha).cumprod(1)
            before = torch.cat((T[:, None], after[:, :-1]), 1)
            weight = before * alpha * (before > 1 - 0.999)
            acc += (weight[..., None, :] * color[entry][..., None]).sum(1).transpose(1, 2)
            saved.append((entry, valid, T))
            # Past the threshold nothing is blended: T stays where it crossed.
            T = after[:, -1]
        image[y[inside], x[inside]] = acc[inside]
        if grad_of is not None:
            groups.append((x, y, inside, px, py, saved))
    if grad_of is None:
        return image, None
    grad_image = grad_of(image)
    grads = [torch.zeros_like(f) for f in splat]
    for x, y, inside, px, py, saved in groups:
        gi = grad_image[y.clamp(max=h - 1), x.clamp(max=w - 1)] * inside[..., None]
        behind = torch.zeros(x.shape, dtype=torch.float64, device=device)  # sum of later g.c weight
        for entry, valid, T in reversed(saved):
            alpha, raw, fall, dx, dy = _chunk_terms(splat, entry, valid, px, py, False)
            after = T[:, None] * (1 - alpha).cumprod(1)
            before = torch.cat((T[:, None], after[:, :-1]), 1)
            active = (before > 1 - 0.999).double()
            weight = before * alpha * active
            shade = (gi[:, None] * color[entry][:, :, None]).sum(-1)
            term = weight * shade
            later = behind[:, None] + term.flip(1).cumsum(1).flip(1) - term
            behind = behind + term.sum(1)
            grad_alpha = (before * shade - later / (1 - alpha)) * active
            grad_raw = grad_alpha * ((alpha > 0) & (raw <= 0.99))
            grad_form = -0.5 * grad_raw * raw
            a, b, c = (splat[i][entry][..., None] for i in (2, 3, 4))
            parts = (-(grad_form * (2 * a * dx + 2 * b * dy)).sum(-1),
                     -(grad_form * (2 * b * dx + 2 * c * dy)).sum(-1),
                     (grad_form * dx * dx).sum(-1), (grad_form * 2 * dx * dy).sum(-1),
                     (grad_form * dy * dy).sum(-1),
                     (weight[..., None] * gi[:, None]).sum(-2), (grad_raw * fall).sum(-1))
            keep = valid.reshape(-1)
            at = entry.reshape(-1)[keep]
            for total, part in zip(grads, parts):
                total.index_add_(0, at, part.reshape(len(keep), *total.shape[1:])[keep])
    return image, grads


def _exact_ssim(image, target):
    """Mean SSIM over the pixels a whole 11 x 11 Gaussian window covers."""
    t = torch.arange(-5, 6, dtype=torch.float64)
    g = (-(t / 1.5) ** 2 / 2).exp()
    g = (g / g.sum()).tolist()

    def window(x):
        n = x.shape[1] - 10
        x = sum(k * x[:, i:i + n] for i, k in enumerate(g))
        n = x.shape[0] - 10
        return sum(k * x[i:i + n] for i, k in enumerate(g))

    mx, my = window(image), window(target)
    sxx = (window(image * image) - mx * mx).clamp_min(0)
    syy = (window(target * target) - my * my).clamp_min(0)
    sxy = window(image * target) - mx * my
    c1, c2 = 0.01 ** 2, 0.03 ** 2
    return (((2 * mx * my + c1) * (2 * sxy + c2))
            / ((mx * mx + my * my + c1) * (sxx + syy + c2))).mean()


def _exact_loss(case, image, target):
    if case["kind"] == "step":
        if case["scene"] == "slab":
            return image.square().mean()
        return (image - target).abs().mean()
    loss = (1 - LAMBDA_DSSIM) * (image.clamp(0, 1) - target).abs().mean()
    shown = image.clamp(0, 1) if case["kind"] == "train" else image
    return loss + LAMBDA_DSSIM * (1 - _exact_ssim(shown, target))


def exact(case, seed):
    g = _generator(seed)
    if case["kind"] == "loss":
        image, target = (t.double() for t in _loss_inputs(case, g))
        image.requires_grad_(True)
        loss = _exact_loss(case, image, target)
        (grad,) = torch.autograd.grad(loss, image)
        return {"loss": loss.detach(), "grad": grad}
    if case["n"] * case["views"] > 2_000_000:
        return None  # minutes of float64 work
    params = [p.double().requires_grad_(True) for p in _parameters(case, g)]
    indices = _draw_subset(case, g)
    used = params if indices is None else [p[indices] for p in params]
    backward = case["kind"] != "render"
    targets = _images(case, g).double() if backward else None
    images, losses = [], 0.0
    grads = [torch.zeros_like(p) for p in params]
    for view, camera in enumerate(_cameras(case, seed)):
        with torch.set_grad_enabled(backward):
            splat, depth, c00, c11 = _exact_project(used, camera, case["sh"])
        with torch.no_grad():
            lists = _exact_lists(splat, depth, c00, c11, case)
            if lists is None:
                return None
            if not backward:
                images.append(_exact_composite(splat, lists, case)[0])
                continue
        target = targets[view] if case["views"] > 1 else targets

        def grad_of(image):
            nonlocal losses
            with torch.enable_grad():
                image = image.detach().requires_grad_(True)
                loss = _exact_loss(case, image, target) / case["views"]
                losses = losses + loss.detach()
                return torch.autograd.grad(loss, image)[0]

        with torch.no_grad():
            image, projected = _exact_composite(splat, lists, case, grad_of)
        images.append(image)
        for total, part in zip(grads, torch.autograd.grad(splat, params, projected)):
            total += part
        del splat, projected
    image = torch.stack(images) if case["views"] > 1 else images[0]
    if not backward:
        return {"image": image}
    if case["kind"] == "step":
        return {"image": image, "loss": losses, **dict(zip(PARAMS, grads))}
    opacity, scale = params[3], params[2]
    regs = OPACITY_REG * opacity.sigmoid().mean() + SCALE_REG * scale.exp().mean()
    for i, part in zip((3, 2), torch.autograd.grad(regs, (opacity, scale))):
        grads[i] += part
    with torch.no_grad():
        # Adam's first step from zero moments: both bias corrections cancel.
        moved = {name: p - RATES[name] * grad / (grad.abs() + 1e-15)
                 for name, p, grad in zip(PARAMS, params, grads)}
    return {"image": image, "loss": losses + regs.detach(),
            **{"grad_" + name: grad for name, grad in zip(PARAMS, grads)}, **moved}
