"""The work that users of nss_hip have it do, as timed cases.

Every case goes through the public Python entry points of
vapoursynth-nssfactory_amd/nss_hip.py on planes that are already on the device,
with the instance (BM3D, WNNM, NCSR or Server) a program keeps for a clip.
``exact`` restates the filters in float64 torch, from their definitions.
"""
from __future__ import annotations

import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "vapoursynth-nssfactory_amd"))
import nss_hip  # noqa: E402

# name: planes, sub-sampling of the planes after the first
FORMATS = {"GRAYS": (1, 0), "RGBS": (3, 0), "YUV444PS": (3, 0), "YUV420PS": (3, 1)}


def listed():
    bm3d = dict(kind="bm3d", final=True, sigma=10.0, step=8, group=8, group_basic=8, range=9, chroma=False,
                transform=0)
    return [
        # The smallest call: a preview or a cropped region through both
        # stages. Host work, launches and the tail of each kernel are all of it.
        dict(bm3d, name="yuv420-128x96-two-stage", fmt="YUV420PS", width=128, height=96),
        # A small frame with an overlapping grid and a wide window, one stage:
        # the usual way to judge settings on a test image.
        dict(bm3d, name="gray-256-dense", fmt="GRAYS", width=256, height=256, final=False, sigma=5.0, step=3,
             group=16, range=16),
        # CBM3D (groups from plane 0 for every plane) on odd, ragged planes:
        # cropped 4:4:4 material, grid and tiles that do not divide the plane.
        dict(bm3d, name="yuv444-1277x717-chroma", fmt="YUV444PS", width=1277, height=717, chroma=True, step=6),
        # The ordinary call: full-HD 4:2:0 video at the default shapes, both stages.
        dict(bm3d, name="yuv420-1080p-two-stage", fmt="YUV420PS", width=1920, height=1080),
        # The same frame's quality profile: overlapping grid, groups of 16 and
        # 32, windows of 39 x 39.
        dict(bm3d, name="yuv420-1080p-heavy", fmt="YUV420PS", width=1920, height=1080, sigma=3.0, step=3, group=32,
             group_basic=16, range=19),
        # The largest single plane: a 4K master, strong noise, in the bf16x3
        # form of the transforms (4K in FP32 is in the serving case).
        dict(bm3d, name="gray-4k-two-stage-bf16x3", fmt="GRAYS", width=3840, height=2160, sigma=20.0, transform=1),
        # Very wide search on a full-HD plane (repetitive textures), one stage.
        dict(bm3d, name="gray-1080p-range30", fmt="GRAYS", width=1920, height=1080, final=False, group=16, range=30),
        # Video in time: both stages with radius 1 over a clip that pans, from
        # the first push to the last pop.
        dict(kind="temporal", name="yuv420-1080p-radius1", fmt="YUV420PS", width=1920, height=1080, frames=8,
             radius=1, final=True, sigma=5.0, step=8, group=8, range=9),
        # Several clips at once through the serving loop: a burst of full-HD
        # 4:2:0 and 4K RGB frames, queued together and drained.
        dict(kind="server", name="serving-1080p-4k", width=1920, height=1080, frames=3, width2=3840, height2=2160,
             frames2=1, sigma=10.0),
        # WNNM at its defaults on a full-HD plane.
        dict(kind="wnnm", name="wnnm-1080p", fmt="GRAYS", width=1920, height=1080, sigma=10.0, step=8, group=8,
             range=7, residual=False),
        # WNNM's quality setting: four times the groups, each of 16, centred.
        dict(kind="wnnm", name="wnnm-1080p-dense", fmt="GRAYS", width=1920, height=1080, sigma=10.0, step=4,
             group=16, range=9, residual=True),
        # NCSR at its defaults (two rounds of matching and filtering).
        dict(kind="ncsr", name="ncsr-1080p", fmt="GRAYS", width=1920, height=1080, sigma=10.0, step=8, group=8,
             range=7),
    ]


def _size(rng, low, high, even):
    w = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    h = max(64, int(w * rng.choice([9 / 16, 9 / 16, 3 / 4, 1.0, 16 / 9 if w < 1400 else 9 / 16])))
    return (w & ~1, h & ~1) if even else (w, h)


def _references(case, width, height):
    return ((width - 8 + case["step"] - 1) // case["step"] + 1) * ((height - 8 + case["step"] - 1) // case["step"] + 1)


def _cost_ms(case):
    """A rough time, to keep drawn cases below the largest listed one."""
    refs = sum(_references(case, w, h) for h, w in _dims(case["fmt"], case["width"], case["height"]))
    window = (2 * case["range"] + 1) ** 2
    if case["kind"] in ("wnnm", "ncsr"):
        per = {8: 1e-5, 16: 4e-5}[case["group"]]
        return refs * (per + window * 5e-9) * (2 if case["kind"] == "ncsr" else 1)
    each = refs * (window * 4.3e-9 + case["group"] * 2.5e-7) * (2 if case["final"] else 1)
    if case["kind"] == "temporal":
        return 5 * each * case["radius"] * case["frames"]
    return each


def draw(rng):
    """One more case of the same ranges, below the cost of the largest listed one."""
    while True:
        kind = rng.choice(["bm3d"] * 6 + ["temporal"] * 2 + ["wnnm", "ncsr", "server"])
        if kind == "server":
            w, h = _size(rng, 320, 1920, True)
            w2, h2 = _size(rng, 320, 2560, False)
            return dict(kind=kind, width=w, height=h, frames=rng.randint(1, 4), width2=w2, height2=h2,
                        frames2=rng.randint(1, 2), sigma=rng.choice([3.0, 5.0, 10.0, 20.0]))
        fmt = rng.choice(["GRAYS", "GRAYS", "YUV420PS", "YUV420PS", "YUV444PS", "RGBS"])
        sigma = rng.choice([3.0, 5.0, 10.0, 20.0])
        if kind == "bm3d":
            w, h = _size(rng, 128, 3840, fmt == "YUV420PS")
            case = dict(kind=kind, fmt=fmt, width=w, height=h, final=rng.random() < 0.7, sigma=sigma,
                        step=rng.choice([3, 4, 6, 7, 8, 8, 8]), group=rng.choice([8, 8, 16, 32]),
                        group_basic=rng.choice([8, 8, 16]), range=rng.choice([7, 9, 9, 12, 16, 19, 24, 30]),
                        chroma=fmt == "YUV444PS" and rng.random() < 0.5, transform=rng.choice([0, 0, 0, 0, 1, 2]))
        elif kind == "temporal":
            w, h = _size(rng, 240, 1920, fmt == "YUV420PS")
            case = dict(kind=kind, fmt=fmt, width=w, height=h, frames=rng.randint(4, 8), radius=rng.choice([1, 1, 2]),
                        final=rng.random() < 0.7, sigma=sigma, step=rng.choice([6, 8, 8]),
                        group=rng.choice([8, 8, 16]), range=rng.choice([7, 9, 9, 12]))
        else:
            w, h = _size(rng, 192, 1920, fmt == "YUV420PS")
            case = dict(kind=kind, fmt=fmt, width=w, height=h, sigma=sigma, step=rng.choice([4, 6, 8, 8]),
                        group=rng.choice([8, 8, 16]), range=rng.choice([7, 7, 9, 12]))
            if kind == "wnnm":
                case["residual"] = rng.random() < 0.5
        if _cost_ms(case) < 5.0:
            return case


# ---------------------------------------------------------------------------
# Inputs: sinusoids and flat rectangles (luma, gray, RGB) or a smooth field
# (chroma), with white noise of the filter's sigma.
# ---------------------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _dims(fmt, width, height):
    n, sub = FORMATS[fmt]
    return [(height >> (sub if i else 0), width >> (sub if i else 0)) for i in range(n)]


def _clean(h, w, rng, chroma):
    dev = _device()
    y = torch.arange(h, device=dev, dtype=torch.float32)[:, None]
    x = torch.arange(w, device=dev, dtype=torch.float32)[None, :]
    img = torch.zeros(h, w, device=dev)
    for _ in range(3 if chroma else 6):
        a = 1 / 6 if chroma else rng.uniform(0.04, 0.12)
        f = rng.uniform(0.002, 0.02) if chroma else rng.uniform(0.01, 0.2)
        ang, phi = rng.uniform(0, 2 * math.pi), rng.uniform(0, 2 * math.pi)
        img += a * torch.sin(2 * math.pi * (f * math.cos(ang) * x + f * math.sin(ang) * y) + phi)
    if chroma:
        return img
    img += 0.5
    low, high = max(1, min(w, h) // 32), max(2, min(w, h) // 4)
    for _ in range(20):
        rw, rh = rng.randint(low, high), rng.randint(low, high)
        x0, y0 = rng.randint(0, w - rw), rng.randint(0, h - rh)
        img[y0:y0 + rh, x0:x0 + rw] = rng.uniform(0, 1)
    return img.clamp_(0, 1)


def _clip(fmt, width, height, frames, sigma, seed):
    """A noisy clip: the first frame, shifted by a few pixels from frame to frame."""
    rng = random.Random(seed)
    gen = torch.Generator(device=_device()).manual_seed(seed)
    sub = FORMATS[fmt][1]
    base = [_clean(h, w, rng, i > 0 and fmt.startswith("YUV")) for i, (h, w) in
            enumerate(_dims(fmt, width, height))]
    out, dx, dy = [], 0, 0
    for n in range(frames):
        if n:
            dx, dy = dx + rng.randint(-4, 4), dy + rng.randint(-4, 4)
        planes = []
        for i, p in enumerate(base):
            s = sub if i else 0
            yi = (torch.arange(p.shape[0], device=p.device) - (dy >> s)).clamp_(0, p.shape[0] - 1)
            xi = (torch.arange(p.shape[1], device=p.device) - (dx >> s)).clamp_(0, p.shape[1] - 1)
            noise = torch.randn(p.shape, generator=gen, device=p.device)
            planes.append((p[yi][:, xi] + noise * (sigma / 255)).contiguous())
        out.append(planes)
    return out


def _server_frames(case, seed):
    first = _clip("YUV420PS", case["width"], case["height"], case["frames"], case["sigma"], seed)
    second = _clip("RGBS", case["width2"], case["height2"], case["frames2"], case["sigma"], seed + 500009)
    return first, second


# ---------------------------------------------------------------------------
# The cases.
# ---------------------------------------------------------------------------

def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "server":
        first, second = _server_frames(c, seed)
        srv = nss_hip.Server(max_batch_frames=8, max_inflight=2)
        a = srv.open_stream("YUV420PS", c["width"], c["height"], sigma=c["sigma"], final=1)
        b = srv.open_stream("RGBS", c["width2"], c["height2"], sigma=c["sigma"], final=1)
        queue = [(a, f, [torch.empty_like(p) for p in f]) for f in first]
        queue += [(b, f, [torch.empty_like(p) for p in f]) for f in second]
        return dict(kind=kind, server=srv, queue=queue)
    clip = _clip(c["fmt"], c["width"], c["height"], c.get("frames", 1), c["sigma"], seed)
    shape = (c["fmt"], c["width"], c["height"])
    if kind == "bm3d":
        inst = nss_hip.BM3D(*shape, sigma=c["sigma"], block_step=c["step"], group_size=c["group"],
                            group_size_basic=c["group_basic"] if c["final"] else None, bm_range=c["range"],
                            chroma=int(c["chroma"]), final=int(c["final"]), transform=c["transform"])
    elif kind == "temporal":
        inst = nss_hip.BM3D(*shape, frames=c["frames"], sigma=c["sigma"], radius=c["radius"], block_step=c["step"],
                            group_size=c["group"], bm_range=c["range"], final=int(c["final"]))
        return dict(kind=kind, inst=inst, clip=clip)
    elif kind == "wnnm":
        inst = nss_hip.WNNM(*shape, sigma=c["sigma"], block_step=c["step"], group_size=c["group"],
                            bm_range=c["range"], residual=int(c["residual"]))
    else:
        inst = nss_hip.NCSR(*shape, sigma=c["sigma"], block_step=c["step"], group_size=c["group"],
                            bm_range=c["range"])
    return dict(kind=kind, inst=inst, planes=clip[0])


def run(state):
    if state["kind"] == "server":
        for stream, planes, out in state["queue"]:
            state["server"].submit(stream, planes, out)
        state["server"].drain()
        return [out for _, _, out in state["queue"]]
    if state["kind"] == "temporal":
        state["inst"].seek(0)
        return state["inst"].filter_clip(state["clip"])
    return state["inst"](state["planes"])


def _plane_flops(case, h, w, group, directions):
    """Matching (3 operations per pixel of each candidate patch) and the fast
    transforms of the groups: 36 operations per 8-point DCT line, 2 per sample
    and level of the Haar axis."""
    r, s = case["range"], case["step"]
    xs = [min(i * s, w - 8) for i in range((w - 8 + s - 1) // s + 1)]
    ys = [min(i * s, h - 8) for i in range((h - 8 + s - 1) // s + 1)]
    wx = sum(min(x + r, w - 8) - max(x - r, 0) + 1 for x in xs)
    wy = sum(min(y + r, h - 8) - max(y - r, 0) + 1 for y in ys)
    match, refs = 192 * (wx * wy - len(xs) * len(ys)), len(xs) * len(ys)
    return match, refs * directions * (group * 16 * 36 + 64 * 2 * (group - 1)), refs


def work(case):
    c, kind = case, case["kind"]
    if kind == "server":
        total = {"bytes": 0, "flops": 0}
        for fmt, w, h, n in (("YUV420PS", c["width"], c["height"], c["frames"]),
                             ("RGBS", c["width2"], c["height2"], c["frames2"])):
            one = work(dict(kind="bm3d", fmt=fmt, width=w, height=h, final=True, step=8, group=8, group_basic=8,
                            range=9, chroma=False))
            total = {k: total[k] + n * one[k] for k in total}
        return total
    dims = _dims(c["fmt"], c["width"], c["height"])
    frames = c.get("frames", 1)
    flops = 0
    for i, (h, w) in enumerate(dims):
        g = c["group"]
        if kind in ("wnnm", "ncsr"):
            match, _, refs = _plane_flops(c, h, w, g, 0)
            # Gram matrix and the product back (2 * 64 g^2 each), a symmetric
            # eigenproblem of size g (about 9 g^3)
            flops += (match + refs * (256 * g * g + 9 * g ** 3)) * (2 if kind == "ncsr" else 1)
            continue
        stages = [(c.get("group_basic", g), 2), (g, 3)] if c["final"] else [(g, 2)]
        for group, directions in stages:
            match, transform, refs = _plane_flops(c, h, w, group, directions)
            if c.get("chroma") and i:
                match = 0
            if kind == "temporal":
                match += refs * 192 * 2 * c["radius"] * 81  # one seed's window per layer and direction
            flops += match + transform
    return {"bytes": 8 * frames * sum(h * w for h, w in dims), "flops": frames * flops}


# ---------------------------------------------------------------------------
# The filters in float64.
# ---------------------------------------------------------------------------

BLOCK = 8


def _positions(n, step, device):
    return (torch.arange((n - BLOCK + step - 1) // step + 1, device=device) * step).clamp_(max=n - BLOCK)


def _spatial(plane, step, rng, group):
    """Matches of every reference: x, y, distance [references, group] in the
    order reference, then (distance, y, x); count of real entries."""
    h, w = plane.shape
    ys, xs = _positions(h, step, plane.device), _positions(w, step, plane.device)
    patches = plane.unfold(0, BLOCK, 1).unfold(1, BLOCK, 1)
    ref = patches[ys][:, xs]
    side = 2 * rng + 1
    dist = torch.full((len(ys), len(xs), side * side), math.inf, dtype=plane.dtype, device=plane.device)
    for dy in range(-rng, rng + 1):
        yy = ys + dy
        vy = (yy >= 0) & (yy <= h - BLOCK)
        rows = patches[yy.clamp(0, h - BLOCK)]
        for dx in range(-rng, rng + 1):
            xx = xs + dx
            v = vy[:, None] & ((xx >= 0) & (xx <= w - BLOCK))[None, :]
            d = (ref - rows[:, xx.clamp(0, w - BLOCK)]).square_().sum((2, 3))
            dist[:, :, (dy + rng) * side + dx + rng] = torch.where(v, d, math.inf)
    dist[:, :, rng * side + rng] = -1.0  # the reference comes first
    dist = dist.reshape(-1, side * side)
    count = torch.isfinite(dist).sum(1).clamp_(max=group)
    parts = []
    for d in dist.split(32768):
        s = torch.sort(d, dim=1, stable=True)
        parts.append((s.values[:, :group], s.indices[:, :group]))
    d, o = (torch.cat(p) for p in zip(*parts))
    cy, cx = ys.repeat_interleave(len(xs))[:, None], xs.repeat(len(ys))[:, None]
    real = torch.arange(group, device=d.device)[None, :] < count[:, None]
    y, x = cy + o // side - rng, cx + o % side - rng
    return torch.where(real, x, cx), torch.where(real, y, cy), torch.where(real, d.clamp_min(0), 0), count


def _predictive(frames, center, radius, step, rng, group, ps_num=2, ps_range=4):
    """The temporal search: the spatial matches of the centre frame, then per
    direction a chain of windows around each layer's best ps_num."""
    x, y, d, count = _spatial(frames[center], step, rng, group)
    n, (h, w) = len(x), frames[0].shape
    ref = frames[center].unfold(0, BLOCK, 1).unfold(1, BLOCK, 1)[y[:, 0], x[:, 0]]
    far = torch.arange(group, device=x.device)[None, :] >= count[:, None]
    layers = {center: (x[:, 1:], y[:, 1:], d[:, 1:].masked_fill(far[:, 1:], math.inf))}
    off = torch.arange(-ps_range, ps_range + 1, device=x.device)
    for sign in (-1, 1):
        cx, cy = x[:, :ps_num], y[:, :ps_num]
        for k in range(1, radius + 1):
            f = center + sign * k
            if not 0 <= f < len(frames):
                break
            px = (cx[:, :, None, None] + off[None, None, None, :]).expand(-1, -1, len(off), -1).reshape(n, -1)
            py = (cy[:, :, None, None] + off[None, None, :, None]).expand(-1, -1, -1, len(off)).reshape(n, -1)
            ok = (px >= 0) & (px <= w - BLOCK) & (py >= 0) & (py <= h - BLOCK)
            key = torch.where(ok, py * w + px, h * w).sort(dim=1).values  # raster order, each position once
            ok = key < h * w
            ok[:, 1:] &= key[:, 1:] != key[:, :-1]
            py, px = (key // w).clamp_(max=h - BLOCK), (key % w).clamp_(max=w - BLOCK)
            patches = frames[f].unfold(0, BLOCK, 1).unfold(1, BLOCK, 1)
            dd = torch.cat([(patches[b, a] - c[:, None]).square_().sum((2, 3))
                            for a, b, c in zip(px.split(8192), py.split(8192), ref.split(8192))])
            s = torch.sort(dd.masked_fill_(~ok, math.inf), dim=1, stable=True)
            o = s.indices[:, :min(ps_num, group)]
            cx, cy = px.gather(1, o), py.gather(1, o)
            layers[f] = (cx, cy, s.values[:, :o.shape[1]])
    order = sorted(layers)
    ax, ay, ad = (torch.cat([layers[f][q] for f in order], 1) for q in range(3))
    at = torch.cat([torch.full_like(layers[f][0], f) for f in order], 1)
    s = torch.sort(ad, dim=1, stable=True)
    o = s.indices[:, :group - 1]
    first = torch.full_like(x[:, :1], center)
    count = 1 + torch.isfinite(s.values[:, :group - 1]).sum(1)
    return (torch.cat([x[:, :1], ax.gather(1, o)], 1), torch.cat([y[:, :1], ay.gather(1, o)], 1),
            torch.cat([first, at.gather(1, o)], 1), count)


def _dct():
    k = torch.arange(BLOCK, dtype=torch.float64)
    m = torch.cos(math.pi * (k[None, :] + 0.5) * k[:, None] / BLOCK) * math.sqrt(2 / BLOCK)
    m[0] *= math.sqrt(0.5)
    return m.to(_device())


def _haar(n):
    """Orthonormal Haar matrix, the mean in row 0."""
    m = torch.ones(1, 1, dtype=torch.float64)
    while m.shape[0] < n:
        k = m.shape[0]
        m = torch.cat([torch.kron(m, torch.tensor([[1.0, 1.0]], dtype=torch.float64)),
                       torch.kron(torch.eye(k, dtype=torch.float64),
                                  torch.tensor([[1.0, -1.0]], dtype=torch.float64))]) / math.sqrt(2)
    return m.to(_device())


def _forward(cube):
    dct = _dct()
    n, g = cube.shape[:2]
    return torch.matmul(_haar(g), torch.matmul(torch.matmul(dct, cube), dct.t()).reshape(n, g, -1))


def _shrink(cube, ref, sigma):
    """Filtered groups [references, group, 8, 8] and their weights."""
    c = _forward(cube)
    if ref is None:
        keep = c.abs() >= 2.7 * sigma
        keep[:, 0, 0] = True
        c *= keep
        weight = 1.0 / keep.sum((1, 2)).clamp(min=1).double()
    else:
        r2 = _forward(ref).square_()
        gain = r2 / (r2 + sigma * sigma)
        gain[:, 0, 0] = 1.0
        c *= gain
        weight = 1.0 / gain.square_().sum((1, 2)).clamp(min=1e-12)
    n, g = cube.shape[:2]
    dct = _dct()
    c = torch.matmul(_haar(g).t(), c).reshape(n, g, BLOCK, BLOCK)
    return torch.matmul(torch.matmul(dct.t(), c), dct), weight


def _gather(frames, x, y, t, count):
    patches = frames.unfold(1, BLOCK, 1).unfold(2, BLOCK, 1)[t, y, x]
    real = torch.arange(x.shape[1], device=x.device)[None, :] < count[:, None]
    return patches * real[:, :, None, None]


def _add(num, den, values, weight, x, y, t, count):
    """Weighted patches into the frames' sums num, den [frames, h, w]."""
    _, h, w = num.shape
    k = torch.arange(BLOCK, device=x.device)
    real = (torch.arange(x.shape[1], device=x.device)[None, :] < count[:, None])[:, :, None, None]
    for v, a, b, c, q, wt in zip(*(s.split(16384) for s in (values, x, y, t, real, weight))):
        at = (c * h + b)[:, :, None, None] * w + k[:, None] * w + a[:, :, None, None] + k
        wt = (wt[:, None, None, None] * q).expand(v.shape)
        num.view(-1).index_add_(0, at.reshape(-1), (v * wt).reshape(-1))
        den.view(-1).index_add_(0, at.reshape(-1), wt.reshape(-1))


def _divide(num, den, source):
    return torch.where(den > 1e-12, num / den.clamp(min=1e-300), source)


def _bm3d_frame(planes, c):
    """Both stages (or the one) of a spatial frame."""
    planes = [p.double() for p in planes]
    sigma = float(torch.tensor(c["sigma"] / 255 * 0.75, dtype=torch.float32))
    ref = None
    for group in ([c["group_basic"], c["group"]] if c["final"] else [c["group"]]):
        out, found = [], None
        for i, p in enumerate(planes):
            if found is None or not c["chroma"]:
                found = _spatial(p if ref is None else ref[i], c["step"], c["range"], group)
            x, y, _, count = found
            t = torch.zeros_like(x)
            num, den = torch.zeros_like(p)[None], torch.zeros_like(p)[None]
            for xs, ys, ts, ks in zip(*(s.split(65536) for s in (x, y, t, count))):
                cube = _gather(p[None], xs, ys, ts, ks)
                v, weight = _shrink(cube, None if ref is None else _gather(ref[i][None], xs, ys, ts, ks), sigma)
                _add(num, den, v, weight, xs, ys, ts, ks)
            out.append(_divide(num[0], den[0], p))
        ref = out
    return ref


def _bm3d_clip(clip, c):
    planes = [torch.stack([f[i] for f in clip]).double() for i in range(len(clip[0]))]
    sigma = float(torch.tensor(c["sigma"] / 255 * 0.75, dtype=torch.float32))
    out = []
    for p in planes:
        ref = None
        for _ in range(2 if c["final"] else 1):
            num, den = torch.zeros_like(p), torch.zeros_like(p)
            for center in range(len(p)):
                x, y, t, count = _predictive(p if ref is None else ref, center, c["radius"], c["step"], c["range"],
                                             c["group"])
                v, weight = _shrink(_gather(p, x, y, t, count),
                                    None if ref is None else _gather(ref, x, y, t, count), sigma)
                _add(num, den, v, weight, x, y, t, count)
            ref = _divide(num, den, p)
        out.append(ref)
    return [[p[n] for p in out] for n in range(len(clip))]


def _svd(a):
    """Singular values (descending) and right vectors of the columns of a
    [references, 64, n], from the eigenvectors of the Gram matrix (on the CPU:
    many small problems)."""
    gram = torch.matmul(a.transpose(1, 2), a)
    vals, vecs = torch.linalg.eigh(gram.cpu())
    vals, vecs = vals.flip(1).to(a.device), vecs.flip(2).to(a.device)
    return vals.clamp_min(0).sqrt(), vecs


def _group_filter(plane, match, c):
    """One round of WNNM or NCSR over a plane."""
    sigma = float(torch.tensor(c["sigma"], dtype=torch.float32) / 255)
    x, y, d, count = _spatial(match, c["step"], c["range"], c["group"])
    t = torch.zeros_like(x)
    n = c["group"]  # the windows of these cases always fill the group
    a = _gather(plane[None], x, y, t, count).reshape(len(x), n, 64).transpose(1, 2)
    centred = c["kind"] == "ncsr" or c["residual"]
    mean = a.mean(2, keepdim=True) if centred else torch.zeros_like(a[:, :, :1])
    a = a - mean
    s, v = _svd(a)
    if c["kind"] == "wnnm":
        left = s * s - 8.0 * math.sqrt(2.0 * n) * sigma * sigma
        keep = left > 0
        if not c["residual"]:
            keep[:, 0] = False
            keep[:, 1:] = keep[:, 1:].cumprod(1).bool()
        else:
            keep = keep.cumprod(1).bool()
        new = torch.where(keep, (s + left.clamp_min(0).sqrt()) * 0.5, 0)
        if not c["residual"]:
            new[:, 0], keep[:, 0] = s[:, 0], True
        gain = new / s.clamp_min(1e-30)
        out = torch.matmul(a, torch.matmul(v * gain[:, None, :], v.transpose(1, 2))) + mean
        kept = keep.sum(1).double()
        weight = torch.where(kept > 0, 1.0 / kept.clamp_min(1), 1.0)
    else:
        code = s[:, :, None] * v.transpose(1, 2)  # rows: codes of the directions
        wt = torch.exp(-d / max(2.0 * 64 * sigma * sigma, 1e-12))
        beta = (code * wt[:, None, :]).sum(2, keepdim=True) / wt.sum(1)[:, None, None]
        e = code - beta
        moment = e.square().sum(2, keepdim=True)
        tau = 2.0 * math.sqrt(2.0) * sigma * sigma / ((moment / n).sqrt() + 1e-12)
        new = e.sign() * (e.abs() - tau).clamp_min(0) + beta
        # directions of no energy carry no code
        inv = torch.where(s > 1e-12 * s[:, :1], 1.0 / s.clamp_min(1e-300), 0)
        out = torch.matmul(torch.matmul(a, v) * inv[:, None, :], new) + mean
        weight = torch.ones(len(x), dtype=a.dtype, device=a.device)
    num, den = torch.zeros_like(plane)[None], torch.zeros_like(plane)[None]
    _add(num, den, out.transpose(1, 2).reshape(len(x), n, BLOCK, BLOCK), weight, x, y, t, count)
    return _divide(num[0], den[0], plane)


def exact(case, seed):
    c, kind = case, case["kind"]
    with torch.no_grad():
        if kind == "server":
            spatial = dict(c, final=True, step=8, group=8, group_basic=8, range=9, chroma=False)
            return [_bm3d_frame(f, spatial) for f in sum(_server_frames(c, seed), [])]
        clip = _clip(c["fmt"], c["width"], c["height"], c.get("frames", 1), c["sigma"], seed)
        if kind == "bm3d":
            return _bm3d_frame(clip[0], c)
        if kind == "temporal":
            return _bm3d_clip(clip, c)
        planes = [p.double() for p in clip[0]]
        if kind == "wnnm":
            return [_group_filter(p, p, c) for p in planes]
        out = []
        for p in planes:
            est = _group_filter(p, p, c)
            est = est + 0.1 * (p - est)
            out.append(_group_filter(est, est, c))
        return out
