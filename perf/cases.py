"""The workloads by which the matcher's speed is judged.

Each case is one call (or one short stream of calls) of the public Python
binding, as a dense-reconstruction program makes them: matching one rectified
pair, matching the pairs of a scene in one call, serving pairs as they arrive,
and the steps before and after the matcher (rectification, combining the pairs
of a view).  `listed()` gives fixed cases, `draw(rng)` more of the same ranges:

* pairs of 0.1 to 24 megapixels, right images 0.85 to 1.15 times as wide,
  disparity spans 32 to 512, the automatic hierarchy or one full-range level,
  16-bit images resident on the GPU or 8-bit images in host memory, with and
  without validity masks, every left-right check and sub-pixel fit;
* scenes of 2 to 10 pairs of 0.2 to 4 megapixels;
* rectification of 1 to 24 megapixel images of every element type, combining
  2 to 6 pairs on grids of 0.5 to 27 megapixels.

Inputs follow the repository's synthetic pairs (value noise of mean 128 and
sigma 40, a Voronoi partition with one disparity plane per cell, a forward
warp with fresh noise in the holes, N(0, 2) noise), made on the GPU from the
seed.  uint8 data enters as u8 * 257 where 16-bit images are given.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from regard3d_mvs_amd import (Camera, CameraModel, MultiStereoOptions, PairGeometry, StereoOptions, SubpixelMethod,
                              align16)
from regard3d_mvs_amd.multiview import Rig, kmat
from regard3d_mvs_amd.native import Matcher, automatic_levels


# ------------------------------------------------------------------ cases
def _match(w, h, nd, **more):
    case = {"kind": "match", "w": w, "h": h, "wr": w, "dmin": 0, "nd": nd, "levels": -1, "masks": False,
            "lr": "full", "subpixel": "equiangular", "uniqueness": 0.0, "flat": 0.0, "slope": 0.2, "place": "device"}
    case.update(more)
    return case


def listed():
    return [
        # A preview-size pair, one level over all its disparities: the smallest call, all launches and latency.
        {"name": "match_384x288_full", **_match(384, 288, 64, levels=0)},
        # The plain VGA pair, 64 disparities, one level.
        {"name": "match_vga_full", **_match(640, 480, 64, levels=0)},
        # The reference's own benchmark size: 1024 x 768, 128 disparities, one full-range level.
        {"name": "match_xga_full", **_match(1024, 768, 128, levels=0)},
        # A video frame with the automatic hierarchy.
        {"name": "match_1080p", **_match(1920, 1080, 256)},
        # What a rectifier really hands over: odd sizes, unequal widths, masks, a negative first disparity;
        # with the cheaper left-right check, the parabola fit and a uniqueness threshold.
        {"name": "match_ragged_masked", **_match(2737, 1811, 203, wr=2513, dmin=-41, masks=True, lr="diagonal",
                                                 subpixel="parabola", uniqueness=0.05)},
        # A camera picture read by a program that keeps 8-bit images and float maps in host memory.
        {"name": "match_12mp_host", **_match(4000, 3000, 320, place="host")},
        # The largest pair: 24 megapixels, 512 disparities, 30% low texture, resident on the GPU.
        {"name": "match_24mp", **_match(6048, 4032, 512, flat=0.3, slope=0.3)},
        # The pairs of a small scene in one call.
        {"name": "batch_scene", "kind": "batch", "count": 8, "mp0": 0.3, "mp1": 3.0, "nd0": 64, "nd1": 256,
         "shape_seed": 11},
        # Pairs served as they come, views kept on the device for their partners, host images in and maps out.
        {"name": "serve_stream", "kind": "serve", "count": 12, "per_view": 2, "mp0": 0.3, "mp1": 4.0, "nd0": 32,
         "nd1": 256, "shape_seed": 12},
        # The step before the matcher: a distorted 24 megapixel image into its rectified camera.
        {"name": "rectify_24mp", "kind": "rectify", "w": 6048, "h": 4032, "tw": 6200, "th": 4150, "dtype": "uint16",
         "model": "radial_k3"},
        # The step after the matcher: four pairs of a view on its grid.
        {"name": "combine_4_pairs", "kind": "combine", "w": 6048, "h": 4536, "pairs": 4, "min_pairs": 1},
    ]


def _log(rng, a, b):
    return math.exp(rng.uniform(math.log(a), math.log(b)))


def _size(rng, mp):
    """A size of about mp megapixels, 3:2, 4:3 or 16:9, neither side rounded to anything."""
    aspect = rng.choice((1.5, 4.0 / 3.0, 16.0 / 9.0))
    h = max(96, int(round(math.sqrt(mp * 1e6 / aspect))))
    return max(128, int(round(h * aspect * rng.uniform(0.97, 1.03)))), h


def draw(rng):
    kind = rng.choice(("match",) * 7 + ("batch", "serve", "rectify", "combine"))
    if kind == "match":
        full = rng.random() < 0.25
        w, h = _size(rng, _log(rng, 0.1, 1.2) if full else _log(rng, 0.25, 20.0))
        nd = int(round(_log(rng, 32, 128 if full else 448)))
        lr = rng.choice(("full", "full", "full", "diagonal", "off"))
        return _match(w, h, nd, wr=int(w * rng.choice((1.0, rng.uniform(0.85, 1.15)))),
                      dmin=rng.choice((0, 0, rng.randint(-60, 40))), levels=0 if full else -1,
                      masks=rng.random() < 0.3, lr=lr,
                      subpixel=rng.choice(("equiangular", "equiangular", "parabola", "none")),
                      uniqueness=rng.choice((0.0, 0.0, 0.05)), flat=rng.choice((0.0, 0.0, 0.3)),
                      slope=rng.uniform(0.1, 0.3), place=rng.choice(("device", "device", "host")))
    if kind in ("batch", "serve"):
        mp0 = _log(rng, 0.2, 0.6)
        case = {"kind": kind, "count": rng.randint(2, 10), "mp0": mp0, "mp1": mp0 * rng.uniform(1.5, 6.0),
                "nd0": rng.randint(32, 64), "nd1": rng.randint(96, 256), "shape_seed": rng.randrange(1 << 20)}
        if kind == "serve":
            case["per_view"] = rng.randint(1, 4)
        return case
    if kind == "rectify":
        w, h = _size(rng, _log(rng, 1.0, 22.0))
        s = rng.uniform(0.9, 1.05)
        return {"kind": "rectify", "w": w, "h": h, "tw": int(w * s), "th": int(h * s),
                "dtype": rng.choice(("uint8", "uint16", "float32")),
                "model": rng.choice(("pinhole", "radial_k1", "radial_k3", "brown_t2"))}
    w, h = _size(rng, _log(rng, 0.5, 24.0))
    return {"kind": "combine", "w": w, "h": h, "pairs": rng.randint(2, 6), "min_pairs": rng.randint(1, 2)}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)
    return g


def _uniform(g, n, a, b):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float32) * (b - a) + a


def _value_noise(h, w, g, mean=128.0, sigma=40.0):
    """Four octaves of bilinearly interpolated random lattices."""
    acc = torch.zeros((h, w), device="cuda")
    for cell in (2, 5, 13, 32):
        lat = torch.randn((h // cell + 2, w // cell + 2), generator=g, device="cuda")
        xs = torch.arange(w, device="cuda", dtype=torch.float32) / cell
        ys = torch.arange(h, device="cuda", dtype=torch.float32) / cell
        ix, iy = xs.long(), ys.long()
        fx, fy = xs - ix, (ys - iy)[:, None]
        rows = lat[:, ix] * (1.0 - fx) + lat[:, ix + 1] * fx
        acc += rows[iy] * (1.0 - fy) + rows[iy + 1] * fy
    acc -= acc.mean()
    return acc * (sigma / acc.std().clamp_min(1e-6)) + mean


def _voronoi(h, w, cell, g):
    """Nearest jittered-grid seed of every pixel: (labels, seed x, seed y)."""
    gh, gw = h // cell + 1, w // cell + 1
    sx = ((torch.arange(gw, device="cuda")[None, :] + torch.rand((gh, gw), generator=g, device="cuda")) * cell).ravel()
    sy = ((torch.arange(gh, device="cuda")[:, None] + torch.rand((gh, gw), generator=g, device="cuda")) * cell).ravel()
    xs, ys = torch.arange(w, device="cuda")[None, :], torch.arange(h, device="cuda")[:, None]
    cx, cy = (xs // cell).clamp_max(gw - 1), (ys // cell).clamp_max(gh - 1)
    best = torch.full((h, w), math.inf, device="cuda")
    lab = torch.zeros((h, w), dtype=torch.long, device="cuda")
    for dy in (-1, 0, 1):
        for dx in (-1, 0, 1):
            idx = (cy + dy).clamp(0, gh - 1) * gw + (cx + dx).clamp(0, gw - 1)
            d2 = (sx[idx] - xs) ** 2 + (sy[idx] - ys) ** 2
            closer = d2 < best
            best = torch.where(closer, d2, best)
            lab = torch.where(closer, idx, lab)
    return lab, sx, sy


def _u8(v):
    return v.round().clamp(0, 255).to(torch.uint8)


def _view(w, h, g, flat=0.0):
    """A left view (uint8) and its Voronoi partition; `flat` of its area is low-texture."""
    left = _value_noise(h, w, g)
    cell = max(32, int(round(math.sqrt(w * h / 40.0))))
    if flat > 0:
        lab, _, _ = _voronoi(h, w, max(64, cell // 2), g)
        n = int(lab.max()) + 1
        area = torch.bincount(lab.ravel(), minlength=n)
        order = torch.randperm(n, generator=g, device="cuda")
        before = torch.cumsum(area[order], 0) - area[order]
        chosen = torch.zeros(n, dtype=torch.bool, device="cuda")
        chosen[order[before < flat * w * h]] = True
        grey = 128.0 + torch.randn((h, w), generator=g, device="cuda")
        left = torch.where(chosen[lab], grey, left)
    return _u8(left), _voronoi(h, w, cell, g)


def _partner(left8, part, wr, dmin, span, slope, g):
    """The right image of a view: x_r = x_l - d for one disparity plane per Voronoi cell, the larger d wins."""
    h, w = left8.shape
    lab, sx, sy = part
    n = sx.numel()
    d0, a, b = _uniform(g, n, 0, span - 1), _uniform(g, n, -slope, slope), _uniform(g, n, -slope, slope)
    xs = torch.arange(w, device="cuda")[None, :]
    ys = torch.arange(h, device="cuda")[:, None]
    d = d0[lab] + a[lab] * (xs - sx[lab]) + b[lab] * (ys - sy[lab])
    disp = d.round().clamp(0, span - 1).long() + dmin
    xr = xs - disp
    ok = (xr >= 0) & (xr < wr)
    key = ((disp - dmin) << 40 | (ys * w + xs))[ok]
    win = torch.full((h * wr,), -1, dtype=torch.long, device="cuda")
    win.scatter_reduce_(0, (ys * wr + xr)[ok], key, "amax")
    src = (win & ((1 << 40) - 1)).clamp_max(h * w - 1)
    fresh = _u8(_value_noise(h, wr, g)).ravel()
    right = torch.where(win >= 0, left8.ravel()[src], fresh).reshape(h, wr).float()
    return _u8(right + 2.0 * torch.randn((h, wr), generator=g, device="cuda"))


def _mask(w, h, g):
    """Validity mask of a slightly turned and shifted picture inside its rectified frame."""
    t, l, r, b = (float(v) for v in _uniform(g, 4, 0.0, 0.04))
    s = [float(v) for v in _uniform(g, 4, -0.03, 0.03)]
    xs = torch.arange(w, device="cuda", dtype=torch.float32)[None, :] / w
    ys = torch.arange(h, device="cuda", dtype=torch.float32)[:, None] / h
    inside = (ys > t + s[0] * (xs - 0.5)) & (ys < 1 - b + s[1] * (xs - 0.5)) & (xs > l + s[2] * (ys - 0.5)) & (
        xs < 1 - r + s[3] * (ys - 0.5))
    return inside.to(torch.uint8) * 255


def _u16(img8):
    """8-bit values as the matcher's 16-bit images: u8 * 257."""
    return (img8.to(torch.int32) * 257).to(torch.uint16)


def _shapes(case):
    """Sizes and spans of a scene's pairs: part of the case, not of the seed."""
    rng = np.random.default_rng(case["shape_seed"])
    out = []
    while len(out) < case["count"]:
        mp = math.exp(rng.uniform(math.log(case["mp0"]), math.log(case["mp1"])))
        aspect = 1.5 if rng.random() < 0.5 else 4.0 / 3.0
        h = int(math.sqrt(mp * 1e6 / aspect))
        w = int(h * aspect)
        for _ in range(min(case.get("per_view", 1), case["count"] - len(out))):
            nd = int(round(math.exp(rng.uniform(math.log(case["nd0"]), math.log(case["nd1"])))))
            out.append((w, h, int(w * rng.uniform(0.85, 1.15)), nd))
    return out


def _options(case):
    return StereoOptions(levels=case["levels"], lr_max_diff=-1 if case["lr"] == "off" else 1,
                         lr_full_match=case["lr"] == "full", subpixel=SubpixelMethod[case["subpixel"]],
                         uniqueness=case["uniqueness"])


_PROGRAM = {}


def _matcher():
    """The program's one matcher: a context, like a device, lives as long as the program."""
    if "m" not in _PROGRAM:
        _PROGRAM["m"] = Matcher(0)
    return _PROGRAM["m"]


def _server():
    """A matcher whose request loop runs for the life of the program."""
    if "s" not in _PROGRAM:
        s = Matcher(0)
        s.serve_start(StereoOptions())
        _PROGRAM["s"] = s
    return _PROGRAM["s"]


def _match_images(case, seed):
    g = _gen(seed)
    w, h, wr = case["w"], case["h"], case["wr"]
    left, part = _view(w, h, g, case["flat"])
    right = _partner(left, part, wr, case["dmin"], case["nd"], case["slope"], g)
    ml = mr = None
    if case["masks"]:
        ml, mr = _mask(w, h, g), _mask(wr, h, g)
        left, right = left * (ml > 0), right * (mr > 0)  # the rectifier leaves 0 outside
    return left, right, ml, mr


def _combine_scene(case, seed):
    """A slanted plane seen by rectified pairs in varied directions: disparity
    maps with noise, holes and one pair that is off, as the matcher leaves them."""
    g = _gen(seed)
    around = ((0.8, 0.05, 0.1), (-0.7, 0.1, 0.0), (0.1, 0.75, -0.1), (-0.2, -0.7, 0.05), (0.55, 0.5, 0.0),
              (-0.5, 0.45, 0.08))
    rig = Rig(around[:case["pairs"]], scale=1.0)
    W, H = case["w"], case["h"]
    scale = W / 320.0
    rig.W, rig.H, rig.F, rig.CX, rig.CY = W, H, 280.0 * scale, 161.2 * scale, H / 2.0 - 1.3 * scale
    xs = torch.arange(W, device="cuda", dtype=torch.float64)[None, :]
    ys = torch.arange(H, device="cuda", dtype=torch.float64)[:, None]
    pairs = []
    for i, cp in enumerate(rig.partners):
        e1 = (cp - rig.cb) / np.linalg.norm(cp - rig.cb)
        e2 = np.cross(rig.rb[2], e1)
        e2 /= np.linalg.norm(e2)
        rr = np.stack([e1, e2, np.cross(e1, e2)])
        kl = kmat(rig.F, rig.CX, rig.CY)
        m = rr.T @ np.linalg.inv(kl)
        base = np.linalg.norm(cp - rig.cb)
        # Depth along the rectified axis of the plane through rig.point, then d = F * baseline / z + offset.
        n = rig.normal @ m
        axis = float((rig.point - rig.cb) @ rig.normal)
        z = axis / (n[0] * xs + n[1] * ys + n[2])
        d = (rig.F * base / z + 20.0 * scale).float()
        d += 0.15 * torch.randn((H, W), generator=g, device="cuda") + (6.0 if i == 2 else 0.0)
        lat = torch.rand((H // 40 + 1, W // 40 + 1), generator=g, device="cuda") < 0.12
        hole = lat[torch.arange(H, device="cuda")[:, None] // 40, torch.arange(W, device="cuda")[None, :] // 40]
        d = torch.where(hole | (torch.rand((H, W), generator=g, device="cuda") < 0.01), math.inf, d)
        conf = torch.rand((H, W), generator=g, device="cuda") * 0.9
        h2r = kl @ rr @ rig.rb.T @ np.linalg.inv(kmat(rig.F, rig.CX, rig.CY))
        pairs.append(PairGeometry(tuple(h2r.ravel()), rig.F * base, 20.0 * scale, tuple(cp), d, conf))
    return rig.grid(), pairs


def _rectify_cameras(case):
    w, h, tw, th = case["w"], case["h"], case["tw"], case["th"]
    f = 0.86 * w
    ax, ay, az = 0.0017, -0.0044, 0.0044
    rx = np.array([[1, 0, 0], [0, np.cos(ax), -np.sin(ax)], [0, np.sin(ax), np.cos(ax)]])
    ry = np.array([[np.cos(ay), 0, np.sin(ay)], [0, 1, 0], [-np.sin(ay), 0, np.cos(ay)]])
    rz = np.array([[np.cos(az), -np.sin(az), 0], [np.sin(az), np.cos(az), 0], [0, 0, 1]])
    params = {"pinhole": (), "radial_k1": (-0.05,), "radial_k3": (-0.06, 0.012, -0.001),
              "brown_t2": (-0.06, 0.012, -0.001, 3e-4, -2e-4)}[case["model"]]
    cam = Camera(w, h, f, f, w / 2 - 0.5, h / 2 - 0.5, CameraModel[case["model"]], params,
                 tuple((rz @ ry @ rx).ravel()))
    return cam, Camera(tw, th, 0.99 * f * tw / w, 0.99 * f * tw / w, tw / 2.0, th / 2.0)


def _rectify_source(case, seed):
    src8 = _u8(_value_noise(case["h"], case["w"], _gen(seed)))
    return {"uint8": lambda: src8, "uint16": lambda: _u16(src8), "float32": lambda: src8.float() / 255.0}[case["dtype"]]()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "match":
        left, right, ml, mr = _match_images(case, seed)
        if case["place"] == "host":
            images = [None if v is None else v.cpu().numpy() for v in (left, right, ml, mr)]
        else:
            images = [_u16(left), _u16(right), ml, mr]
        state = {"m": _matcher(), "images": images, "options": _options(case)}
    elif kind == "batch":
        g = _gen(seed)
        pairs = []
        for w, h, wr, nd in _shapes(case):
            left, part = _view(w, h, g)
            pairs.append({"left": _u16(left), "right": _u16(_partner(left, part, wr, 0, nd, 0.2, g)), "nd": nd})
        state = {"m": _matcher(), "pairs": pairs}
    elif kind == "serve":
        g = _gen(seed)
        views, pairs = [], []
        for k, (w, h, wr, nd) in enumerate(_shapes(case)):
            if k % case["per_view"] == 0:
                left, part = _view(w, h, g)
                views.append(left.cpu().numpy())
            pairs.append((len(views), (h, w), nd, _partner(left, part, wr, 0, nd, 0.2, g).cpu().numpy()))
        state = {"m": _server(), "views": views, "pairs": pairs}
    elif kind == "rectify":
        cam, target = _rectify_cameras(case)
        state = {"m": _matcher(), "src": _rectify_source(case, seed), "cam": cam, "target": target}
    else:
        grid, pairs = _combine_scene(case, seed)
        state = {"m": _matcher(), "grid": grid, "pairs": pairs,
                 "options": MultiStereoOptions(min_pairs=case["min_pairs"])}
    torch.cuda.synchronize()
    return {"kind": kind, "case": case, **state}


# ------------------------------------------------------------------ one pass
def run(state):
    m, kind, case = state["m"], state["kind"], state["case"]
    if kind == "match":
        left, right, ml, mr = state["images"]
        r = m.match(left, right, ml, mr, dmin=case["dmin"], nd=case["nd"], options=state["options"])
        return {"disparity": r.disparity, "confidence": r.confidence}
    if kind == "batch":
        return [{"disparity": r.disparity, "confidence": r.confidence} for r in m.match_batch(state["pairs"])]
    if kind == "serve":
        for k, img in enumerate(state["views"]):
            m.view_put(k + 1, img)
        tickets = [m.submit(shape, nd=nd, right=right, left_view=view) for view, shape, nd, right in state["pairs"]]
        done = [m.wait(t) for t in tickets]
        for k in range(len(state["views"])):
            m.view_evict(k + 1)
        return [{"disparity": r.disparity, "confidence": r.confidence} for r in done]
    if kind == "rectify":
        image, valid = m.rectify(state["src"], state["cam"], state["target"])
        return {"image": _plain(image), "valid": valid}
    depth, confidence, mask = m.combine_pairs(state["grid"], state["pairs"], state["options"])
    return {"depth": depth, "confidence": confidence, "mask": _plain(mask)}


def _plain(t):
    """uint16 results as int16 bits, the form in which torch indexes and compares them on the GPU."""
    return t.view(torch.int16) if t.dtype == torch.uint16 else t


# ------------------------------------------------------------------ work
def _match_work(w, h, wr, nd, levels, lr_full, in_bytes, masks=False):
    """Images in, two float maps out; integer operations of the cells that
    have to be looked at: per cell a cost (2), 8 path steps of 3 minima and 4
    additions, and the selection (1).  A hierarchy searches its coarsest level
    over all labels and at least 16 labels per pixel of the finer ones."""
    levels = levels if levels >= 0 else automatic_levels(w, h, nd)
    sides = 2 if lr_full else 1
    cells = sum((w >> k) * (h >> k) * (align16(max(nd >> k, 1)) if k == levels else 16) for k in range(levels + 1))
    return {"bytes": in_bytes * (w + wr) * h + (w + wr) * h * bool(masks) + 8 * w * h,
            "flops": sides * cells * (2 + 8 * 7 + 1)}


def work(case):
    kind = case["kind"]
    if kind == "match":
        return _match_work(case["w"], case["h"], case["wr"], case["nd"], case["levels"], case["lr"] == "full",
                           1 if case["place"] == "host" else 2, case["masks"])
    if kind in ("batch", "serve"):
        parts = [_match_work(w, h, wr, nd, -1, True, 2 if kind == "batch" else 1) for w, h, wr, nd in _shapes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    size = {"uint8": 1, "uint16": 2, "float32": 4}
    if kind == "rectify":
        s, target = size[case["dtype"]], case["tw"] * case["th"]
        return {"bytes": s * case["w"] * case["h"] + (s + 1) * target, "flops": target * (30 + 40)}
    n = case["w"] * case["h"]
    return {"bytes": n * (8 * case["pairs"] + 10), "flops": n * (40 * case["pairs"] + 80)}


# ------------------------------------------------------------------ 64-bit values
def _popcount(v):
    v = v - ((v >> 1) & 0x5555555555555555)
    v = (v & 0x3333333333333333) + ((v >> 2) & 0x3333333333333333)
    v = (v + (v >> 4)) & 0x0F0F0F0F0F0F0F0F
    return sum((v >> (8 * k)) & 0xFF for k in range(8))


def _exact_census(img):
    h, w = img.shape
    pad = torch.nn.functional.pad(img.double()[None, None], (4, 4, 3, 3), mode="replicate")[0, 0].long()
    bits = torch.zeros((h, w), dtype=torch.long, device=img.device)
    for dy in range(7):
        for dx in range(9):
            if (dy, dx) != (3, 4):
                bits = bits * 2 + (pad[dy:dy + h, dx:dx + w] < img).long()
    return bits


def _exact_paths(cost, img, o):
    """Sum of the 8 path costs of a full-range volume (h, w, labels), every path pixel by pixel."""
    h, w, n = cost.shape
    total = torch.zeros_like(cost)
    inf = 1 << 40

    def p2(a, b):
        return torch.clamp_min(o.p2 * o.p2_adapt // (o.p2_adapt + ((a - b).abs() >> 8)), o.p1 + 1)

    def step(prev, pen, c):
        low = prev.amin(-1, keepdim=True)
        side = torch.nn.functional.pad(prev, (1, 1), value=inf)
        near = torch.minimum(side[:, :-2], side[:, 2:]) + o.p1
        return c + torch.minimum(torch.minimum(prev, near), low + pen[:, None]) - low

    for dx, dy in ((1, 0), (-1, 0), (0, 1), (0, -1), (1, 1), (-1, -1), (-1, 1), (1, -1)):
        if dy == 0:
            cols = range(w) if dx > 0 else range(w - 1, -1, -1)
            prev = None
            for x in cols:
                prev = cost[:, x] if prev is None else step(prev, p2(img[:, x], img[:, x - dx]), cost[:, x])
                total[:, x] += prev
            continue
        prev = None
        for y in range(h) if dy > 0 else range(h - 1, -1, -1):
            new = cost[y].clone()
            if prev is not None:
                lo, hi = max(0, dx), w + min(0, dx)
                new[lo:hi] = step(prev[lo - dx:hi - dx], p2(img[y, lo:hi], img[y - dy, lo - dx:hi - dx]), cost[y, lo:hi])
            prev = new
            total[y] += new
    return total


def _exact_side(base, partner, dmin, n, o, subpixel, uniqueness):
    """Disparity and confidence of one matching direction, one tile, all labels."""
    h, w = base.shape
    wp = partner.shape[1]
    cb, cp = _exact_census(base), _exact_census(partner)
    xs = torch.arange(w, device=base.device)
    cost = torch.empty((h, w, n), dtype=torch.long, device=base.device)
    for k in range(n):
        xp = xs - dmin - k
        ok = (xp >= 0) & (xp < wp)
        cost[:, :, k] = torch.where(ok, _popcount(cb ^ cp[:, xp.clamp(0, wp - 1)]), o.invalid_cost)
    s = _exact_paths(cost, base, o)
    best_cost = s.amin(-1)
    labels = torch.arange(n, device=base.device)
    best = torch.where(s == best_cost[..., None], labels, n).amin(-1)
    second = torch.where((labels - best[..., None]).abs() <= 1, 0xFFFF, s).amin(-1)
    xp = xs - dmin - best
    ok = (xp >= 0) & (xp < wp)
    b, second = best_cost.double(), second.double()
    if uniqueness > 0:
        ok &= ~((second != 0xFFFF) & (b > (1.0 - uniqueness) * second))
    sm = s.gather(-1, (best - 1).clamp_min(0)[..., None])[..., 0].double()
    sp = s.gather(-1, (best + 1).clamp_max(n - 1)[..., None])[..., 0].double()
    if subpixel == "parabola":
        den = 2.0 * (sm - 2.0 * b + sp)
    else:
        den = 2.0 * torch.maximum(sm - b, sp - b)
    delta = torch.where(den > 0, (sm - sp) / torch.where(den > 0, den, 1.0), 0.0).clamp(-0.5, 0.5)
    delta = torch.where((best > 0) & (best < n - 1), delta, 0.0)
    if subpixel == "none":
        delta = torch.zeros_like(delta)
    d = torch.where(ok, dmin + best + delta, math.inf)
    conf = torch.where(ok & (second != 0xFFFF) & (second > 0), 1.0 - b / second.clamp_min(1.0), 0.0)
    return d, conf


def _exact_speckles(d, min_size, max_diff):
    """4-connected segments of close disparities by label propagation; the small ones become invalid."""
    h, w = d.shape
    lab = torch.arange(h * w, device=d.device).reshape(h, w)
    right, down = (d[:, 1:] - d[:, :-1]).abs() <= max_diff, (d[1:] - d[:-1]).abs() <= max_diff
    while True:
        new = lab.clone()
        new[:, 1:] = torch.where(right, torch.minimum(new[:, 1:], lab[:, :-1]), new[:, 1:])
        new[:, :-1] = torch.where(right, torch.minimum(new[:, :-1], lab[:, 1:]), new[:, :-1])
        new[1:] = torch.where(down, torch.minimum(new[1:], lab[:-1]), new[1:])
        new[:-1] = torch.where(down, torch.minimum(new[:-1], lab[1:]), new[:-1])
        new = new.ravel()[new.ravel()].reshape(h, w)
        if torch.equal(new, lab):
            break
        lab = new
    size = torch.bincount(lab.ravel(), minlength=h * w)
    return torch.where(size[lab] < min_size, math.inf, d)


def _exact_median(d):
    """Median of the valid values of the 3 x 3 window (the mean of the middle two for an even count)."""
    h, w = d.shape
    pad = torch.nn.functional.pad(d, (1, 1, 1, 1), value=math.inf)
    win = torch.stack([pad[y:y + h, x:x + w] for y in range(3) for x in range(3)], -1).sort(-1).values
    n = torch.isfinite(win).sum(-1, keepdim=True)
    hi = win.gather(-1, (n // 2).clamp_max(8))[..., 0]
    lo = win.gather(-1, ((n - 1) // 2).clamp_min(0))[..., 0]
    return torch.where(torch.isfinite(d), 0.5 * (lo + hi), d)


def _exact_match(case, seed):
    """The whole matcher for one full-range level in one tile (the blend is then the identity)."""
    o = _options(case)
    left8, right8, _, _ = _match_images(case, seed)
    left, right = left8.long() * 257, right8.long() * 257
    n = align16(case["nd"])
    (h, w), wr, dmin = left.shape, right.shape[1], case["dmin"]
    d, conf = _exact_side(left, right, dmin, n, o, case["subpixel"], case["uniqueness"])
    rd, _ = _exact_side(right.flip(1), left.flip(1), dmin + wr - w, n, o, case["subpixel"], case["uniqueness"])
    rd = rd.flip(1) - (wr - w)
    pos = torch.arange(w, device=d.device) - d
    xo = torch.where(torch.isfinite(d), torch.sign(pos) * torch.floor(pos.abs() + 0.5), -1.0).long()
    other = torch.where((xo >= 0) & (xo < wr), rd.gather(1, xo.clamp(0, wr - 1)), math.inf)
    good = torch.isfinite(d) & torch.isfinite(other) & ((d - other).abs() <= o.lr_max_diff)
    d = torch.where(good, d, math.inf)
    d = _exact_median(_exact_speckles(d, o.speckle_size, o.speckle_diff))
    return {"disparity": d, "confidence": conf}


def _exact_rectify(case, seed):
    """Bicubic resampling in 64 bits (the sizes drawn here sample the full resolution)."""
    cam, t = _rectify_cameras(case)
    src = _rectify_source(case, seed).double()
    h, w = src.shape
    r = torch.tensor(cam.rotation, dtype=torch.float64).reshape(3, 3)
    xs = (torch.arange(t.width, device="cuda", dtype=torch.float64)[None, :] - t.cx) / t.fx
    ys = (torch.arange(t.height, device="cuda", dtype=torch.float64)[:, None] - t.cy) / t.fy
    q = [float(r[i, 0]) * xs + float(r[i, 1]) * ys + float(r[i, 2]) for i in range(3)]
    ux, uy = q[0] / q[2], q[1] / q[2]
    k = tuple(cam.params) + (0.0,) * 5
    r2 = ux * ux + uy * uy
    radial = r2 * (k[0] + r2 * (k[1] + r2 * k[2])) if case["model"] != "radial_k1" else k[0] * r2
    t1, t2 = k[3], k[4]
    dx = ux + ux * radial + t2 * (r2 + 2 * ux * ux) + 2 * t1 * ux * uy
    dy = uy + uy * radial + t1 * (r2 + 2 * uy * uy) + 2 * t2 * ux * uy
    sx, sy = cam.fx * dx + cam.cx, cam.fy * dy + cam.cy
    inside = (q[2] > 1e-9) & (sx >= -0.5) & (sy >= -0.5) & (sx <= w - 0.5) & (sy <= h - 0.5)
    fx, fy = torch.floor(sx), torch.floor(sy)

    def weights(f):
        return (-0.5 * f ** 3 + f ** 2 - 0.5 * f, 1.5 * f ** 3 - 2.5 * f ** 2 + 1.0, -1.5 * f ** 3 + 2.0 * f ** 2 + 0.5 * f,
                0.5 * f ** 3 - 0.5 * f ** 2)

    wx, wy = weights(sx - fx), weights(sy - fy)
    x0, y0 = fx.long() - 1, fy.long() - 1
    out = torch.zeros_like(sx)
    for j in range(4):
        row = (y0 + j).clamp(0, h - 1) * w
        for i in range(4):
            out += wy[j] * wx[i] * src.ravel()[row + (x0 + i).clamp(0, w - 1)]
    return {"image": torch.where(inside, out, 0.0), "valid": None}


def _exact_combine(case, seed):
    """The vote and the weighted least squares over the pairs of a view, in 64 bits."""
    grid, pairs = _combine_scene(case, seed)
    o = MultiStereoOptions(min_pairs=case["min_pairs"])
    W, H, N = grid.width, grid.height, len(pairs)
    xs = torch.arange(W, device="cuda", dtype=torch.float64)[None, :].expand(H, W)
    ys = torch.arange(H, device="cuda", dtype=torch.float64)[:, None].expand(H, W)
    wi, ki, ci, have = [], [], [], []
    for p in pairs:
        g = p.grid_to_rect
        c = g[6] * xs + g[7] * ys + g[8]
        u, v = (g[0] * xs + g[1] * ys + g[2]) / c, (g[3] * xs + g[4] * ys + g[5]) / c
        d = p.disparity.double()
        h, w = d.shape
        inside = (c > 1e-9) & (u > -0.5) & (v > -0.5) & (u < w - 0.5) & (v < h - 0.5)
        x0, y0 = torch.floor(u).long().clamp(0, w - 1), torch.floor(v).long().clamp(0, h - 1)
        x1, y1 = (x0 + 1).clamp_max(w - 1), (y0 + 1).clamp_max(h - 1)
        q = torch.stack([d[y0, x0], d[y0, x1], d[y1, x0], d[y1, x1]])
        smooth = torch.isfinite(q).all(0) & (q.amax(0) - q.amin(0) <= 1.0)
        fx, fy = (u - x0).clamp(0, 1), (v - y0).clamp(0, 1)
        top, bottom = q[0] + fx * (q[1] - q[0]), q[2] + fx * (q[3] - q[2])
        xn = torch.floor(u + 0.5).long().clamp(0, w - 1)
        yn = torch.floor(v + 0.5).long().clamp(0, h - 1)
        s = torch.where(smooth, top + fy * (bottom - top), d[yn, xn])
        ok = inside & torch.isfinite(s) & (s > p.offset)
        k = p.fb / c
        have.append(ok)
        ki.append(torch.where(ok, k, 0.0))
        wi.append(torch.where(ok, (s - p.offset) / k, 0.0))
        ci.append(torch.where(ok, p.confidence.double()[yn, xn], 0.0))
    have, ki, wi, ci = (torch.stack(v) for v in (have, ki, wi, ci))
    n = have.sum(0)
    top_support = torch.zeros_like(n)
    top_conf = torch.full((H, W), -1.0, dtype=torch.float64, device="cuda")
    used = torch.zeros_like(have)
    for i in range(N):
        agree = have & have[i] & ((ki * (wi - wi[i])).abs() <= o.inlier_px)
        support, sc = agree.sum(0), (ci * agree).sum(0)
        better = have[i] & ((support > top_support) | ((support == top_support) & (sc > top_conf)))
        top_support, top_conf = torch.where(better, support, top_support), torch.where(better, sc, top_conf)
        used = torch.where(better, agree, used)
    for _ in range(N):
        sw = (ki * ki * used).sum(0)
        wopt = (ki * ki * wi * used).sum(0) / sw
        res = torch.where(used, (ki * (wi - wopt)).abs(), -1.0)
        worst, at = res.max(0)
        drop = worst > o.max_reprojection_px
        used = used & ~(drop & (torch.arange(N, device="cuda")[:, None, None] == at))
    m = used.sum(0)
    ok = (n >= o.min_pairs) & (m >= o.min_pairs) & ((m > n - m) | ((m >= 2) & (m >= n - m))) & (wopt > 0)
    z = 1.0 / wopt
    ik, rt = np.array(grid.inv_k).reshape(3, 3), np.array(grid.rot_t).reshape(3, 3)
    ray = rt @ ik
    point = torch.stack([grid.center[i] + z * (ray[i, 0] * xs + ray[i, 1] * ys + ray[i, 2]) for i in range(3)])

    def towards(centre):
        a = torch.tensor(centre, dtype=torch.float64, device="cuda")[:, None, None] - point
        return a / a.norm(dim=0)

    back = towards(grid.center)
    cos_min = math.cos(o.min_angle_deg * math.pi / 180.0)
    wide = torch.zeros_like(ok)
    for i, p in enumerate(pairs):
        wide |= used[i] & ((back * towards(p.partner_center)).sum(0) <= cos_min)
    ok &= wide
    return {"depth": torch.where(ok, z, 0.0),
            "confidence": torch.where(ok, (ci * used).sum(0) / m.clamp_min(1), 0.0), "mask": None}


def exact(case, seed):
    """Values in 64 bits, where plain torch reaches them in seconds: one-level
    matches of one tile, float rectification, combined depths of moderate
    grids.  A hierarchical match decides every level's search ranges by the
    level below; running it in plain torch takes minutes."""
    kind = case["kind"]
    if (kind == "match" and case["levels"] == 0 and max(case["w"], case["wr"], case["h"]) <= 512
            and case["lr"] == "full" and not case["masks"]):
        return _exact_match(case, seed)
    if kind == "rectify" and case["dtype"] == "float32":
        return _exact_rectify(case, seed)
    if kind == "combine" and case["w"] * case["h"] * case["pairs"] <= 120_000_000:
        return _exact_combine(case, seed)
    return None
