"""The work that programs give this library, as cases that can be timed and compared.

Each case is one call sequence of a stacking program through the public Python interface, on
synthetic frames made from a seed.  The sizes come from the library's configurations, tests and
benchmark workloads (640x480 plain stacks, 1920x1080 affine batches, 1024x1024 turbulence, 4096x3000
raw Bayer frames, mixed-size focus stacks) or are generic.  `exact` restates the small arithmetic
definitions in 64-bit torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import serstacker_amd as S
from serstacker_amd import _lib

DEV = "cuda:0"
F64 = torch.float64


# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------
def listed():
    return [
        # one frame of a live 320x240 region of interest, aligned as it arrives: launches and latency
        dict(name="frame_320x240", family="frame", w=320, h=240, motion=3, levels=3, scale=1.0, eps=0.02, method=0),
        # the plain method's stack: 64 mono frames, euclidean, three levels, weights, stack
        dict(name="stack_640x480_euclidean", family="stack", n=64, w=640, h=480, motion=1, levels=3, scale=1.0,
             eps=1e-4, method=0),
        # the batched affine workload: 1080p planetary frames through the device-driven batch
        dict(name="stack_1080p_affine", family="stack_batch", n=192, w=1920, h=1080, motion=3, levels=4, scale=1.0,
             eps=0.02),
        # alignment of an RGB focus sequence by translation, at the half size the options default to
        dict(name="align_rgb_translation", family="align", n=24, w=2048, h=1536, levels=3, scale=0.5, eps=0.02),
        # turbulence: phase correlation, dense flow, bicubic warp and average
        dict(name="turbulence_1024", family="turbulence", n=48, w=1024, h=1024, levels=5, support=3),
        # pre-alignment of raw Bayer frames on their 2x2-binned luminance
        dict(name="phasecorr_raw_4096x3000", family="phasecorr", n=16, w=4096, h=3000, binning=2, u16=True),
        # Bayer-aware average of the same frames by their translations
        dict(name="bayer_4096x3000", family="bayer", n=32, w=4096, h=3000, u16=True, colorid=8),
        # focus stacking of mixed-size sequences in one batch (odd size and mono among them)
        dict(name="focus_mixed", family="focus", sizes="1024x768x3x16,1537x1021x1x9,2048x1536x3x12", sigma=5.0,
             levels=6),
        # the best-frame scan over raw frames before a stack
        dict(name="master_scan_4096x3000", family="master", n=24, w=4096, h=3000, colorid=8, kradius=1, dscale=1),
        # raw frames to f32 BGR, the conversion in front of a colour stack
        dict(name="input_2048x1536_bgr", family="input", n=24, w=2048, h=1536, colorid=8, bpp=12, algorithm=-1,
             dark=False),
        # a colour stack of already aligned frames with per-pixel weight maps, odd size
        dict(name="accumulate_rgb_1501x1003", family="accumulate", n=24, w=1501, h=1003, cn=3, motion=3, wmaps=True,
             interp=1),
        # the finished colour stack: holes filled, then sharpened
        dict(name="finish_2880x1620_rgb", family="finish", w=2880, h=1620, cn=3, sigma=3.0, alpha=0.6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["frame", "stack", "stack", "stack_batch", "stack_batch", "align", "turbulence", "phasecorr",
                         "bayer", "focus", "master", "input", "accumulate", "finish"])
    c = dict(family=family)
    if family == "frame":
        w = _log(rng, 160, 1280)
        c.update(w=w, h=max(120, int(w * rng.uniform(0.5, 1.0))), motion=rng.choice([0, 1, 2, 3]),
                 levels=rng.choice([2, 3]), scale=rng.choice([1.0, 0.5]), eps=0.02, method=rng.choice([0, 0, 1, 2, 3]))
    elif family == "stack":
        w = _log(rng, 240, 1280)
        c.update(n=_log(rng, 4, 64), w=w, h=max(160, int(w * rng.uniform(0.5, 1.0))), motion=rng.choice([0, 1, 2, 3]),
                 levels=rng.choice([2, 3, 4]), scale=1.0, eps=rng.choice([1e-4, 0.02]), method=rng.choice([0, 0, 2, 3]))
    elif family == "stack_batch":
        w = _log(rng, 320, 1920)
        h = max(240, int(w * rng.uniform(0.5, 1.0)))
        c.update(n=max(4, min(_log(rng, 8, 512), 192 * 1920 * 1080 // (w * h))), w=w, h=h,
                 motion=rng.choice([0, 1, 3, 3]), levels=rng.choice([3, 4]), scale=1.0, eps=0.02)
    elif family == "align":
        w = _log(rng, 512, 3072)
        h = max(384, int(w * rng.uniform(0.5, 0.9)))
        c.update(n=max(2, min(_log(rng, 4, 48), 24 * 2048 * 1536 // (w * h))), w=w, h=h, levels=rng.choice([2, 3]),
                 scale=rng.choice([1.0, 0.5]), eps=0.02)
    elif family == "turbulence":
        w = rng.choice([256, 512, 512, 1024])
        h = w if rng.random() < 0.5 else int(w * rng.uniform(0.6, 1.0))
        c.update(n=_log(rng, 2, 48), w=w, h=h, levels=rng.choice([4, 5]), support=rng.choice([3, 4]))
    elif family == "phasecorr":
        w = _log(rng, 200, 4096)
        h = int(w * rng.uniform(0.5, 1.0))
        b = rng.choice([1, 2]) if w <= 2048 else 2
        c.update(n=max(1, min(_log(rng, 1, 64), 16 * 4096 * 3000 // (w * h))), w=w, h=h, binning=b,
                 u16=rng.random() < 0.6)
    elif family == "bayer":
        w = _log(rng, 400, 4096) // 2 * 2
        h = int(w * rng.uniform(0.5, 1.0)) // 2 * 2
        c.update(n=max(1, min(_log(rng, 2, 64), 32 * 4096 * 3000 // (w * h))), w=w, h=h, u16=rng.random() < 0.7,
                 colorid=rng.choice([8, 9, 10, 11]))
    elif family == "focus":
        sizes = []
        for _ in range(rng.choice([1, 2, 3])):
            w = _log(rng, 256, 2048)
            sizes.append("%dx%dx%dx%d" % (w, max(200, int(w * rng.uniform(0.5, 0.9))), rng.choice([1, 3, 3]),
                                          rng.randint(2, 14)))
        c.update(sizes=",".join(sizes), sigma=rng.choice([1.5, 3.0, 5.0]), levels=rng.choice([0, 4, 6]))
    elif family == "master":
        w = _log(rng, 320, 4096) // 2 * 2
        h = int(w * rng.uniform(0.5, 1.0)) // 2 * 2
        c.update(n=max(1, min(_log(rng, 1, 100), 24 * 4096 * 3000 // (w * h))), w=w, h=h, colorid=rng.choice([0, 8, 11]),
                 kradius=rng.choice([1, 1, 2]), dscale=rng.choice([1, 1, 2]))
    elif family == "input":
        w = _log(rng, 321, 3072)
        h = int(w * rng.uniform(0.5, 1.0))
        c.update(n=max(1, min(_log(rng, 1, 64), 24 * 2048 * 1536 // (w * h))), w=w // 2 * 2, h=h // 2 * 2,
                 colorid=rng.choice([8, 9, 10, 11]), bpp=rng.choice([10, 12, 16]), algorithm=rng.choice([-1, 2, 4, 5]),
                 dark=rng.random() < 0.4)
    elif family == "accumulate":
        w = _log(rng, 301, 1920)
        h = int(w * rng.uniform(0.5, 1.0))
        cn = rng.choice([1, 3])
        c.update(n=max(2, min(_log(rng, 2, 64), 24 * 1501 * 1003 * 3 // (w * h * cn))), w=w, h=h, cn=cn,
                 motion=rng.choice([0, 1, 3]), wmaps=rng.random() < 0.5, interp=rng.choice([1, 1, 2]))
    else:
        w = _log(rng, 320, 2880)
        c.update(w=w, h=int(w * rng.uniform(0.5, 1.0)), cn=rng.choice([1, 3]), sigma=round(rng.uniform(0.8, 6.0), 2),
                 alpha=round(rng.uniform(0.2, 0.8), 2))
    return c


# ---------------------------------------------------------------------------------------------
# synthetic inputs (torch only)
# ---------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 2654435761 % (1 << 31) + 17)
    return g


def _rand(g, *shape):
    return torch.rand(shape, generator=g, device=DEV)


def _gauss(img, sigma):
    """Separable gaussian of (b, 1, h, w), replicated borders."""
    if sigma <= 0:
        return img
    r = int(3 * sigma + 0.5)
    t = torch.arange(-r, r + 1, device=DEV, dtype=img.dtype)
    k = torch.exp(-t * t / (2 * sigma * sigma))
    k = k / k.sum()
    img = torch.nn.functional.pad(img, (r, r, r, r), mode="replicate")
    img = torch.nn.functional.conv2d(img, k.view(1, 1, 1, -1))
    return torch.nn.functional.conv2d(img, k.view(1, 1, -1, 1))


def _grid(w, h, dtype=torch.float32):
    ys, xs = torch.meshgrid(torch.arange(h, device=DEV, dtype=dtype), torch.arange(w, device=DEV, dtype=dtype),
                            indexing="ij")
    return xs, ys


def _sample(img, xs, ys):
    """img (1, c, h, w) at the positions (h', w'), bicubic, borders replicated."""
    h, w = img.shape[-2:]
    grid = torch.stack([xs / (w - 1) * 2 - 1, ys / (h - 1) * 2 - 1], -1)[None]
    return torch.nn.functional.grid_sample(img, grid, mode="bicubic", padding_mode="border", align_corners=True)


def _disk(g, w, h):
    """A textured limb-darkened disk (1, 1, h, w) on a dark background, peak 1."""
    xs, ys = _grid(w, h)
    r = 0.39 * min(w, h)
    d2 = ((xs - w / 2) ** 2 + (ys - h / 2) ** 2) / (r * r)
    mu = torch.sqrt((1 - d2).clamp(min=0))
    tex = _gauss(_rand(g, 1, 1, h, w) - 0.5, 3.0)[0, 0]
    tex = tex / tex.std() * 0.06
    body = (1 - 0.6 * (1 - mu)) * (1 + tex)
    return _gauss(torch.where(d2 < 1, body, torch.zeros_like(body))[None, None], 0.8)


def _noisy(g, img, scale=2000.0 / 65536.0):
    """Photon noise of a 2000 e- peak and 4 e- of read noise, in units of `scale` at the peak."""
    e = img * 2000.0
    e = e + torch.sqrt(e.clamp(min=0)) * torch.randn(img.shape, generator=g, device=DEV)
    return (e + 4.0 * torch.randn(img.shape, generator=g, device=DEV)) * (scale / 2000.0)


def _planet_frames(g, n, w, h, motion, cn=1):
    """(reference, frames): the disk moved by a random transform of the motion per frame, blurred by seeing."""
    scene = _disk(g, w, h)
    blurred = [_gauss(scene, s) for s in (0.0, 0.9, 1.5, 2.1)]
    u = lambda: float(torch.rand((), generator=g, device=DEV)) * 2 - 1
    xs, ys = _grid(w, h)
    cx, cy = w / 2, h / 2
    span = min(20.0, 0.02 * min(w, h) + 2)
    frames = torch.empty((n, h, w) if cn == 1 else (n, h, w, cn), device=DEV)
    for i in range(n):
        a = math.radians(u() * (1.0 if motion == 3 else 0.5)) if motion else 0.0
        s = 1 + 0.005 * u() if motion >= 2 else 1.0
        sh = 0.002 * u() if motion == 3 else 0.0
        tx, ty = span * u(), span * u()
        px = s * (math.cos(a) * (xs - cx) - math.sin(a) * (ys - cy)) + sh * (ys - cy) + cx + tx
        py = s * (math.sin(a) * (xs - cx) + math.cos(a) * (ys - cy)) + cy + ty
        img = _sample(blurred[i % 4], px, py)[0, 0]
        if cn == 1:
            frames[i] = _noisy(g, img)
        else:
            for k in range(cn):
                frames[i, ..., k] = _noisy(g, img * (1.0 - 0.2 * k))
    return (scene[0, 0] * (2000.0 / 65536.0)).contiguous(), frames


def _field(g, w, h, octaves=5, base=128):
    """Sum of octaves of value noise (1, 1, h, w) in [0, 1]."""
    acc = torch.zeros((1, 1, h, w), device=DEV)
    amp, tot = 1.0, 0.0
    for o in range(octaves):
        gw, gh = max(2, w // max(base >> o, 2) + 2), max(2, h // max(base >> o, 2) + 2)
        acc += amp * torch.nn.functional.interpolate(_rand(g, 1, 1, gh, gw), size=(h, w), mode="bicubic",
                                                     align_corners=False)
        tot += amp
        amp *= 0.6
    return (acc / tot).clamp(0, 1)


def _star_frames(g, n, w, h):
    """12-bit raw frames (int16 storage) of a star field over sky, with their translations (even steps + sub-pixel)."""
    m = 32
    xs, ys = _grid(w + 2 * m, h + 2 * m)
    r = torch.sqrt((xs - w / 2 - m) ** 2 + ((ys - h / 2 - m) * 1.3) ** 2) / (0.1 * w)
    sky = 200 + 900 * torch.exp(-2.0 * r ** 0.66)
    stars = torch.zeros((1, 1) + sky.shape, device=DEV)
    k = 400
    px = (_rand(g, k) * (w - 8) + m + 4).long()
    py = (_rand(g, k) * (h - 8) + m + 4).long()
    stars[0, 0, py, px] = torch.exp(_rand(g, k) * 4.0) * 600.0
    scene = sky[None, None] + _gauss(stars, 1.8)
    shifts = torch.round(_rand(g, n, 2) * 14 - 7) * 2 + (_rand(g, n, 2) - 0.5)
    out = torch.empty((n, h, w), dtype=torch.int16, device=DEV)
    sh = shifts.cpu().numpy()
    for i in range(n):
        fx, fy = sh[i]
        ix, iy = int(math.floor(fx)), int(math.floor(fy))
        ax, ay = float(fx - ix), float(fy - iy)
        v = scene[0, 0]
        c = lambda dy, dx: v[m - iy - dy:m - iy - dy + h, m - ix - dx:m - ix - dx + w]
        img = (1 - ay) * ((1 - ax) * c(0, 0) + ax * c(0, 1)) + ay * ((1 - ax) * c(1, 0) + ax * c(1, 1))
        img = img + torch.sqrt(img) * torch.randn(img.shape, generator=g, device=DEV)
        out[i] = img.clamp(0, 4095).to(torch.int16)
    return out, sh.astype(np.float32)


def _statuses(params, nparams):
    st = (_lib.RegistrationStatus * len(params))()
    for i, p in enumerate(params):
        st[i].ok, st[i].nparams = 1, nparams
        for k in range(nparams):
            st[i].params[k] = float(p[k])
    return st


def _views(frames):
    return _lib.images([S.image_view(f) for f in frames])


def _params(st):
    return np.array([s.params[:] for s in st], np.float32)


def _reg(case, w, h, **kw):
    o = S.c_image_registration_options(motion_type=case.get("motion", 0), scale=case["scale"], eps=case["eps"],
                                       ecch_max_level=case["levels"], max_iterations=50,
                                       ecc_method=case.get("method", 0), **kw)
    return S.c_frame_registration(o)


def _compute_device(acc, avg, mask):
    """The stack into device images, where the finish of a colour stack takes it from."""
    a, m = S.image_view(avg, out=True), S.image_view(mask, out=True)
    _lib.check(_lib.load().ssg_accumulation_compute(acc._h, a, m, 1.0), "compute")
    return dict(avg=avg, mask=mask)


# ---------------------------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------------------------
def _inputs(case, seed):
    """The seeded tensors and arrays of a case; `exact` starts from the same."""
    g, f = _gen(seed), case["family"]
    if f in ("frame", "stack", "stack_batch"):
        ref, frames = _planet_frames(g, case.get("n", 1), case["w"], case["h"], case["motion"])
        return dict(ref=ref, frames=frames)
    if f == "align":
        n, w, h = case["n"], case["w"], case["h"]
        scene = torch.cat([_field(g, w, h) for _ in range(3)], 1)
        xs, ys = _grid(w, h)
        sh = (_rand(g, n, 2) * 12 - 6).cpu().numpy()
        sh[0] = 0
        frames = torch.empty((n, h, w, 3), device=DEV)
        for i in range(n):
            frames[i] = _sample(scene, xs + float(sh[i, 0]), ys + float(sh[i, 1]))[0].permute(1, 2, 0)
        frames += 0.004 * torch.randn(frames.shape, generator=g, device=DEV)
        return dict(frames=frames)
    if f == "turbulence":
        n, w, h = case["n"], case["w"], case["h"]
        scene = _disk(g, w, h)
        xs, ys = _grid(w, h)
        frames = torch.empty((n, h, w), device=DEV)
        for i in range(n):
            d = torch.nn.functional.interpolate(torch.randn((1, 2, 8, 8), generator=g, device=DEV) * 1.5, size=(h, w),
                                                mode="bicubic", align_corners=True)[0]
            t = (_rand(g, 2) * 20 - 10).cpu()
            frames[i] = _sample(scene, xs - d[0] - float(t[0]), ys - d[1] - float(t[1]))[0, 0]
        frames += 0.005 * torch.randn(frames.shape, generator=g, device=DEV)
        return dict(ref=scene[0, 0].contiguous(), frames=frames)
    if f in ("phasecorr", "bayer"):
        raw, shifts = _star_frames(g, case["n"] + 1, case["w"], case["h"])
        if not case["u16"]:
            raw = raw.to(torch.float32) / 4096.0
        return dict(ref=raw[0], frames=raw[1:], shifts=shifts[1:])
    if f == "focus":
        seqs = []
        for spec in case["sizes"].split(","):
            w, h, cn, n = (int(v) for v in spec.split("x"))
            scene = torch.cat([_field(g, w, h, 6) for _ in range(cn)], 1)
            soft = torch.cat([_gauss(scene[:, c:c + 1], 2.4) for c in range(cn)], 1)
            z = _field(g, w, h, 2, 512)[0, 0]
            z = (z - z.min()) / (z.max() - z.min())
            sh = (_rand(g, n, 2) * 12 - 6).cpu().numpy().astype(np.float32)
            xs, ys = _grid(w, h)
            fr = torch.empty((n, h, w) if cn == 1 else (n, h, w, cn), device=DEV)
            for i in range(n):
                t = ((z - i / max(n - 1, 1)).abs() * 2).clamp(0, 1)
                img = _sample(scene * (1 - t) + soft * t, xs - float(sh[i, 0]), ys - float(sh[i, 1]))[0]
                fr[i] = img[0] if cn == 1 else img.permute(1, 2, 0)
            seqs.append((fr, sh))
        return dict(seqs=seqs)
    if f == "master":
        n, w, h = case["n"], case["w"], case["h"]
        scene = _field(g, w, h)[0, 0] * 3000 + 300
        out = torch.empty((n, h, w), dtype=torch.int16, device=DEV)
        for i in range(n):
            out[i] = (scene + torch.sqrt(scene) * torch.randn(scene.shape, generator=g, device=DEV)).clamp(0, 4095).to(
                torch.int16)
        return dict(frames=out)
    if f == "input":
        n, w, h = case["n"], case["w"], case["h"]
        scene = _field(g, w, h)[0, 0]
        top = float(2 ** case["bpp"] - 1) if case["bpp"] < 16 else 65535.0
        raw = torch.empty((n, h, w), dtype=torch.int32, device=DEV)
        for i in range(n):
            raw[i] = ((scene + 0.02 * torch.randn(scene.shape, generator=g, device=DEV)).clamp(0, 1) * top).to(torch.int32)
        raw = raw.to(torch.int16) if case["bpp"] < 16 else ((raw + 32768) % 65536 - 32768).to(torch.int16)
        d = dict(frames=raw)
        if case["dark"]:
            d["dark"] = 0.01 * _rand(g, h, w)
            d["flat"] = 0.8 + 0.4 * _rand(g, h, w)
        return d
    if f == "accumulate":
        n, w, h, cn = case["n"], case["w"], case["h"], case["cn"]
        scene = torch.cat([_field(g, w, h) for _ in range(cn)], 1)[0]
        frames = torch.empty((n, h, w) if cn == 1 else (n, h, w, cn), device=DEV)
        for i in range(n):
            img = scene + 0.01 * torch.randn(scene.shape, generator=g, device=DEV)
            frames[i] = img[0] if cn == 1 else img.permute(1, 2, 0)
        u = (_rand(g, n, 6) * 2 - 1).cpu().numpy().astype(np.float64)
        if case["motion"] == 0:
            p = u[:, :2] * 12
        elif case["motion"] == 1:
            p = np.stack([u[:, 0] * 12, u[:, 1] * 12, u[:, 2] * 0.01], 1)
        else:
            p = np.stack([1 + 0.005 * u[:, 0], 0.01 * u[:, 1], 12 * u[:, 2], 0.01 * u[:, 3], 1 + 0.005 * u[:, 4],
                          12 * u[:, 5]], 1)
        d = dict(frames=frames, params=p.astype(np.float32))
        if case["wmaps"]:
            d["wmaps"] = torch.cat([_field(g, w, h, 3) for _ in range(n)], 1)[0] + 0.05
        else:
            d["weights"] = (0.2 + _rand(g, n)).cpu().numpy()
        return d
    n, w, h, cn = 1, case["w"], case["h"], case["cn"]
    img = torch.cat([_field(g, w, h, 7) for _ in range(cn)], 1)[0]
    img = (img[0] if cn == 1 else img.permute(1, 2, 0)).contiguous()
    hole = _rand(g, h, w) < 0.01
    hole[: max(1, h // 40)] = True  # the rows that no frame covered
    mask = torch.where(hole, 0, 255).to(torch.uint8)
    return dict(img=img, mask=mask)


def prepare(case, seed):
    s, f = _inputs(case, seed), case["family"]
    s["case"] = case
    w, h = case.get("w"), case.get("h")
    if f in ("frame", "stack", "stack_batch", "align"):
        s["reg"] = _reg(case, w, h)
        assert s["reg"].setup_reference_frame(s["ref"] if "ref" in s else s["frames"][0])
        s["views"] = _views(s["frames"])
        if f in ("stack", "stack_batch"):
            s["acc"] = S.c_weigthed_average(w, h, 1)
    elif f == "turbulence":
        s["pc"] = S.phase_correlation(w, h, 1)
        s["pc"].set_reference(s["ref"])
        s["flow"] = S.c_eccflow(max_iterations=3, support_scale=case["support"], max_pyramid_level=case["levels"] - 1,
                                downscale=_lib.ECCFLOW_DOWNSCALE_PYRAMID)
        s["flow"].set_reference_image(s["ref"])
        s["acc"] = S.c_weigthed_average(w, h, 1)
        s["ident"] = torch.stack(_grid(w, h), -1)
        s["maps"] = torch.empty((case["n"], h, w, 2), device=DEV)
        s["views"], s["mviews"] = _views(s["frames"]), _views(s["maps"])
    elif f == "phasecorr":
        s["pc"] = S.phase_correlation(w, h, case["binning"])
        s["pc"].set_reference(s["ref"])
        s["views"] = _views(s["frames"])
    elif f == "bayer":
        s["acc"] = S.c_bayer_average(w, h, case["colorid"], 12)
        s["out"] = torch.empty((h, w, 3), device=DEV), torch.empty((h, w), dtype=torch.uint8, device=DEV)
        s["views"] = _views(s["frames"])
        s["st"] = _statuses(s["shifts"], 2)
    elif f == "focus":
        s["stacks"], s["views"], s["outs"], s["shifts"] = [], [], [], []
        for fr, sh in s["seqs"]:
            cn = 1 if fr.dim() == 3 else fr.shape[3]
            s["stacks"].append(S.c_laplacian_pyramid_focus_stacking(
                fr.shape[2], fr.shape[1], cn, fusing_policy=_lib.FOCUS_LPG_WEIGHTS, lpg_k=6.0, lpg_p=2.0,
                lpg_sigma=case["sigma"], max_levels=case["levels"]))
            s["views"].append(_views(fr))
            s["outs"].append(torch.empty(fr.shape[1:], device=DEV))
            s["shifts"].append(sh)
    elif f == "master":
        s["views"] = _views(s["frames"])
    elif f == "input":
        half = case["algorithm"] == _lib.DEBAYER_SP
        s["out"] = torch.empty((case["n"], h // 2, w // 2, 3) if half else (case["n"], h, w, 3), device=DEV)
        s["views"], s["oviews"] = _views(s["frames"]), _views(s["out"])
    elif f == "accumulate":
        s["acc"] = S.c_weigthed_average(w, h, case["cn"])
        s["out"] = (torch.empty((h, w) if case["cn"] == 1 else (h, w, case["cn"]), device=DEV),
                    torch.empty((h, w), dtype=torch.uint8, device=DEV))
        s["views"] = _views(s["frames"])
        s["st"] = _statuses(s["params"], s["params"].shape[1])
        if "wmaps" in s:
            s["wviews"] = _views(s["wmaps"])
    else:
        s["full"], s["fmask"] = torch.empty_like(s["img"]), torch.empty_like(s["mask"])
        s["out"] = torch.empty_like(s["img"])
    torch.cuda.synchronize()  # the library's streams do not wait for torch's
    return s


def run(s):
    case = s["case"]
    f = case["family"]
    # of a registration: the parameters and the correlation (iteration counts describe the path to them)
    if f == "frame":
        ok = s["reg"].register_frame(s["frames"][0])
        st = s["reg"].status()
        return dict(ok=int(ok), params=np.array(st.params[:], np.float32), rho=float(st.rho))
    if f == "stack":
        st = s["reg"].register_batch(s["views"])
        wts = S.frame_sharpness(s["views"])
        s["acc"].clear()
        s["acc"].add_registered_batch(s["views"], st, case["motion"], frame_weights=wts)
        avg, mask = s["acc"].compute()
        return dict(params=_params(st), rho=np.array([x.rho for x in st]), weights=wts, avg=avg, mask=mask)
    if f == "stack_batch":
        s["acc"].clear()
        st = s["reg"].stack_batch(s["acc"], s["views"])
        avg, mask = s["acc"].compute()
        return dict(params=_params(st), rho=np.array([x.rho for x in st]), avg=avg, mask=mask)
    if f == "align":
        st = s["reg"].register_batch(s["views"])
        return dict(params=_params(st)[:, :2].copy(), rho=np.array([x.rho for x in st]))
    if f == "turbulence":
        est = s["pc"].estimate(s["views"])
        t = torch.from_numpy(est[:, :2].astype(np.float32)).to(DEV)
        torch.add(s["ident"].unsqueeze(0), t[:, None, None, :], out=s["maps"])
        torch.cuda.synchronize()  # the library's streams do not wait for torch's
        s["flow"].compute_batch(s["views"], s["mviews"], rmaps=s["mviews"])
        s["acc"].clear()
        s["acc"].add_remapped_batch(s["views"], s["mviews"], interpolation=_lib.INTER_CUBIC)
        avg, mask = s["acc"].compute()
        return dict(shifts=est, maps=s["maps"], avg=avg, mask=mask)
    if f == "phasecorr":
        return s["pc"].estimate(s["views"])
    if f == "bayer":
        s["acc"].clear()
        s["acc"].add_registered_batch(s["views"], s["st"], _lib.MOTION_TRANSLATION)
        return _compute_device(s["acc"], *s["out"])
    if f == "focus":
        for st in s["stacks"]:
            st.clear()
        S.focus_stack_batch(s["stacks"], s["views"], s["shifts"])
        return [st.compute(o) for st, o in zip(s["stacks"], s["outs"])]
    if f == "master":
        return S.master_frame_quality(s["views"], case["colorid"], case["kradius"], case["dscale"])
    if f == "input":
        S.read_input_frames(s["views"], case["colorid"], case["bpp"], case["algorithm"], dark=s.get("dark"),
                            flat=s.get("flat"), outs=s["oviews"])
        return s["out"]
    if f == "accumulate":
        s["acc"].clear()
        s["acc"].add_registered_batch(s["views"], s["st"], case["motion"], frame_weights=s.get("weights"),
                                      interpolation=case["interp"], weight_maps=s.get("wviews"))
        return _compute_device(s["acc"], *s["out"])
    S.average_pyramid_inpaint(s["img"], s["mask"], out=s["full"], out_mask=s["fmask"])
    S.unsharp_mask(s["full"], case["sigma"], case["alpha"], out=s["out"])
    return dict(full=s["full"], mask=s["fmask"], out=s["out"])


def work(case):
    f = case["family"]
    w, h, n = case.get("w", 0), case.get("h", 0), case.get("n", 1)
    px = w * h
    if f in ("frame", "align"):
        # the frames and the reference read; a few operations per pixel and level at the least
        return dict(bytes=4 * px * ((3 if f == "align" else 1) * n + 1), flops=60 * px * n)
    if f in ("stack", "stack_batch"):
        return dict(bytes=4 * px * (n + 1) + 5 * px, flops=100 * px * n)
    if f == "turbulence":
        return dict(bytes=px * (4 * n + 4 + 8 * n + 5), flops=px * n * (5 * 2 * math.log2(max(px, 2)) + 250))
    if f == "phasecorr":
        b = case["binning"]
        return dict(bytes=(2 if case["u16"] else 4) * px * n, flops=n * (px / b / b) * 10 * math.log2(max(px, 2)))
    if f == "bayer":
        return dict(bytes=(2 if case["u16"] else 4) * px * n + 13 * px, flops=24 * px * n)
    if f == "focus":
        t = dict(bytes=0, flops=0)
        for spec in case["sizes"].split(","):
            w, h, cn, n = (int(v) for v in spec.split("x"))
            t["bytes"] += 4 * w * h * cn * (n + 1)
            t["flops"] += w * h * n * (4 * int(8 * case["sigma"] + 1) + 60 + 50 * cn)
        return t
    if f == "master":
        return dict(bytes=2 * px * n + 8 * n, flops=10 * px * n)
    if f == "input":
        o = px // 4 if case["algorithm"] == _lib.DEBAYER_SP else px
        return dict(bytes=n * (2 * px + 12 * o), flops=12 * px * n)
    if f == "accumulate":
        cn = case["cn"]
        return dict(bytes=px * (n * (4 * cn + (4 if case["wmaps"] else 0)) + 4 * cn + 1), flops=px * n * 12 * (cn + 1))
    cn = case["cn"]
    return dict(bytes=px * (4 * cn + 1 + 2 * 4 * cn + 1), flops=60 * px * cn)


def tolerance(case):
    """About four times what the 64-bit restatement below differs by over the drawn sizes."""
    f = case["family"]
    if f in ("frame", "stack", "stack_batch", "align"):
        # an iteration on positions quantised to 1/32 px that stops on a threshold: 32-bit sums in another
        # order end on another side of the threshold for some frames, within the library's bar of 0.01 px
        # (0.1 px for the damped and inverse-compositional rules, which compare two nearly equal errors)
        loose = case.get("method", 0) != 0
        return {"rel": 1e-2 if loose else 3e-3, "max": 0.1 if loose else 0.04, "differ": 1e-3}
    if f == "turbulence":
        # shifts 1e-6; a flow that differs in its last digits moves samples across 1/32 px steps
        return {"rel": 5e-5, "max": 5e-2, "differ": 1e-4}
    if f == "phasecorr":
        return {"rel": 1e-6, "max": 4e-6}  # the fitted position of the peak of a 32-bit transform
    if f == "bayer":
        return {"rel": 1.2e-5, "max": 1e-3}  # tap weights from 32-bit positions
    if f == "accumulate":
        return {"rel": 4e-5, "max": 1e-2}  # samples at 32-bit positions quantised to 1/32 px
    if f == "focus":
        return {"rel": 5e-7, "max": 1e-5}
    if f == "master":
        return {"rel": 1e-12, "max": 1e-12}  # 64-bit sums of the same whole values
    if f == "input":
        return {"rel": 5e-7, "max": 5e-6} if case["dark"] else "exact"
    return {"rel": 1e-6, "max": 1e-5}


# ---------------------------------------------------------------------------------------------
# the same results in 64-bit torch
# ---------------------------------------------------------------------------------------------
def _reflect101(i, n):
    if n == 1:
        return torch.zeros_like(i)
    i = i.abs() % (2 * (n - 1))
    return torch.where(i >= n, 2 * (n - 1) - i, i)


def _edge(img, l, r, t, b, mode):
    """(b, h, w) padded: "clamp", "r101" (mirror without the edge) or "mirror" (with it)."""
    h, w = img.shape[-2:]
    ys, xs = torch.arange(-t, h + b, device=img.device), torch.arange(-l, w + r, device=img.device)
    if mode == "clamp":
        ys, xs = ys.clamp(0, h - 1), xs.clamp(0, w - 1)
    elif mode == "r101":
        ys, xs = _reflect101(ys, h), _reflect101(xs, w)
    else:
        ys, xs = ys % (2 * h), xs % (2 * w)
        ys, xs = torch.minimum(ys, 2 * h - 1 - ys), torch.minimum(xs, 2 * w - 1 - xs)
    return img[..., ys, :][..., xs]


def _sep64(img, kx, ky, mode):
    rx, ry = len(kx) // 2, len(ky) // 2
    h, w = img.shape[-2:]
    p = _edge(img, rx, rx, ry, ry, mode)
    a = sum(k * p[..., i:i + w] for i, k in enumerate(kx) if k)
    return sum(k * a[..., i:i + h, :] for i, k in enumerate(ky) if k)


def _gk(n, sigma):
    v = [math.exp(-0.5 * ((i - (n - 1) / 2) / sigma) ** 2) for i in range(n)]
    return [x / sum(v) for x in v]


def _down64(img, dw, dh, mode="r101"):
    k = [1 / 16, 4 / 16, 6 / 16, 4 / 16, 1 / 16]
    h, w = img.shape[-2:]
    p = _edge(img, 2, max(2, 2 * dw + 1 - w), 2, max(2, 2 * dh + 1 - h), mode)
    a = sum(c * p[..., i:i + 2 * dw - 1:2] for i, c in enumerate(k))
    return sum(c * a[..., i:i + 2 * dh - 1:2, :] for i, c in enumerate(k))


def _up64(img, dw, dh):
    def axis(a, n):  # along the last axis: mirrored on the left, replicated on the right
        s = a.shape[-1]
        left = a[..., 1:2] if s > 1 else a[..., :1]
        p = torch.cat([left, a, a[..., -1:]], -1)
        out = torch.empty(a.shape[:-1] + (2 * s,), dtype=a.dtype, device=a.device)
        out[..., 0::2] = (p[..., :-2] + 6 * p[..., 1:-1] + p[..., 2:]) / 8
        out[..., 1::2] = (p[..., 1:-1] + p[..., 2:]) / 2
        if n > 2 * s:
            out = torch.cat([out, out[..., -2:-1]], -1)
        return out[..., :n]
    return axis(axis(img, dw).transpose(-1, -2), dh).transpose(-1, -2)


def _taps(sx, sy):
    X, Y = torch.round(sx * 32).long(), torch.round(sy * 32).long()
    return X >> 5, Y >> 5, X & 31, Y & 31


def _fetch(img, ix, iy, border):
    """img (b, h, w) at (b, h', w') integer positions; 0 outside for "zero"."""
    h, w = img.shape[-2:]
    inside = (ix >= 0) & (ix < w) & (iy >= 0) & (iy < h)
    if border == "r101":
        xx, yy = _reflect101(ix, w), _reflect101(iy, h)
    else:
        xx, yy = ix.clamp(0, w - 1), iy.clamp(0, h - 1)
    v = torch.gather(img.reshape(img.shape[0], -1), 1, (yy * w + xx).reshape(img.shape[0], -1)).reshape(ix.shape)
    return torch.where(inside, v, torch.zeros_like(v)) if border == "zero" else v


def _remap64(img, sx, sy, border, cubic=False):
    ix, iy, fx, fy = _taps(sx, sy)
    if not cubic:
        tx, ty = fx.to(F64) / 32, fy.to(F64) / 32
        return ((1 - ty) * ((1 - tx) * _fetch(img, ix, iy, border) + tx * _fetch(img, ix + 1, iy, border)) +
                ty * ((1 - tx) * _fetch(img, ix, iy + 1, border) + tx * _fetch(img, ix + 1, iy + 1, border)))

    def coef(f):
        x, A = f.to(F64) / 32, -0.75
        c0 = ((A * (x + 1) - 5 * A) * (x + 1) + 8 * A) * (x + 1) - 4 * A
        c1 = ((A + 2) * x - (A + 3)) * x * x + 1
        c2 = ((A + 2) * (1 - x) - (A + 3)) * (1 - x) * (1 - x) + 1
        return [c0, c1, c2, 1 - c0 - c1 - c2]
    cx, cy = coef(fx), coef(fy)
    return sum(cy[j] * sum(cx[i] * _fetch(img, ix + i - 1, iy + j - 1, border) for i in range(4)) for j in range(4))


def _mask64(sx, sy, w, h, least):
    """remap of an all-255 8-bit mask with 15-bit weights, constant 0 outside, compared with `least`."""
    ix, iy, fx, fy = _taps(sx, sy)
    unit = (fx == 0) & (fy == 0)
    tot = torch.zeros_like(ix)
    for dy in (0, 1):
        for dx in (0, 1):
            wt = (fx if dx else 32 - fx) * (fy if dy else 32 - fy) * 32
            if dx == dy:
                wt = torch.where(unit, torch.full_like(wt, 1 if dx else 32767), wt)
            ins = (ix + dx >= 0) & (ix + dx < w) & (iy + dy >= 0) & (iy + dy < h)
            tot += torch.where(ins, wt, torch.zeros_like(wt))
    return ((255 * tot + 16384) >> 15) >= least


def _erode5(m):
    return torch.nn.functional.max_pool2d((~m).to(torch.float32)[:, None], 5, 1, 2)[:, 0] == 0


def _map64(motion, p, w, h):
    """Positions (b, h, w) of the parameters (b, np)."""
    xs, ys = _grid(w, h, F64)
    q = [p[:, i, None, None] for i in range(p.shape[1])]
    if motion == 0:
        return xs + q[0], ys + q[1]
    if motion == 3:
        return q[0] * xs + q[1] * ys + q[2], q[3] * xs + q[4] * ys + q[5]
    s = q[3] if motion == 2 else 1.0
    c, n = torch.cos(q[2]), torch.sin(q[2])
    return s * (c * xs - n * ys) + q[0], s * (n * xs + c * ys) + q[1]


def _ecc64(ref, frames, motion, nlev, eps0, max_it=50, step=1.5):
    """Forward-additive ECC over the pyramid, translation first (no masks): (parameters, rho)."""
    h, w = ref.shape
    k = _gk(7, 1.0)
    R, Cu = [_sep64(ref.to(F64)[None], k, k, "clamp")], [_sep64(frames.to(F64), k, k, "clamp")]
    while len(R) < nlev:
        nh, nw = (((v + 1) >> 1) & ~1 for v in R[-1].shape[-2:])
        if min(nw, nh) < 16:
            break
        R.append(_down64(R[-1], nw, nh))
        Cu.append(_down64(Cu[-1], nw, nh))
    n, L = len(frames), len(R)
    d5, s3 = [1 / 12, -2 / 3, 0, 2 / 3, -1 / 12], [0.25, 0.5, 0.25]

    def align(mot, p):
        tr = [2, 5] if mot == 3 else [0, 1]
        if L > 1:
            p[:, tr] *= R[-1].shape[-1] / R[0].shape[-1]
        for l in range(L - 1, -1, -1):
            r, c = R[l], Cu[l]
            lh, lw = r.shape[-2:]
            act = torch.arange(n, device=DEV)
            xs, ys = _grid(lw, lh, F64)
            for _ in range(max_it):
                if not len(act):
                    break
                sx, sy = _map64(mot, p[act], lw, lh)
                g = _remap64(c[act], sx, sy, "clamp")
                m = _mask64(sx, sy, lw, lh, 255).to(F64)
                gx, gy = _sep64(g, d5, s3, "clamp") * m, _sep64(g, s3, d5, "clamp") * m
                cnt = m.sum((1, 2))
                mf, mg = (r * m).sum((1, 2)) / cnt, (g * m).sum((1, 2)) / cnt
                sf = ((r - mf[:, None, None]) ** 2 * m).sum((1, 2)).sqrt()
                sg = ((g - mg[:, None, None]) ** 2 * m).sum((1, 2)).sqrt()
                rhs = ((g - mg[:, None, None]) - (sg / sf)[:, None, None] * (r - mf[:, None, None])) * m
                if mot == 0:
                    J = [gx, gy]
                elif mot == 3:
                    J = [gx * xs, gx * ys, gx, gy * xs, gy * ys, gy]
                else:
                    q = p[act]
                    sc = q[:, 3, None, None] if mot == 2 else 1.0
                    ca, sa = torch.cos(q[:, 2, None, None]), torch.sin(q[:, 2, None, None])
                    A, B = sa * xs + ca * ys, ca * xs - sa * ys
                    J = [gx, gy, sc * (gy * B - gx * A)] + ([gx * B + gy * A] if mot == 2 else [])
                H = torch.stack([torch.stack([(a * b).sum((1, 2)) for b in J], -1) for a in J], -2)
                e = torch.stack([(a * rhs).sum((1, 2)) for a in J], -1)
                dp = -step * torch.linalg.solve(H, e[..., None])[..., 0]
                p[act] += dp
                if mot == 0:
                    ep = dp.norm(dim=1)
                elif mot == 3:
                    s_ = torch.tensor([lw, lh, 1.0, lw, lh, 1.0], device=DEV, dtype=F64)
                    ep = (dp * s_).norm(dim=1)
                else:
                    ds = dp[:, 3] if mot == 2 else torch.ones(len(act), device=DEV, dtype=F64)
                    sn = torch.sin(dp[:, 2])
                    ep = (dp[:, 0] ** 2 + dp[:, 1] ** 2 + (lw * sn) ** 2 + (lh * sn) ** 2 + (max(lw, lh) * ds) ** 2).sqrt()
                act = act[~(ep < eps0 * (1 << l))]
            if l > 0:
                p[:, tr] *= R[l - 1].shape[-1] / lw
        return p

    npar = {0: 2, 1: 3, 2: 4, 3: 6}[motion]
    p = torch.zeros((n, npar), device=DEV, dtype=F64)
    if motion == 3:
        p[:, 0] = p[:, 4] = 1
    if motion == 2:
        p[:, 3] = 1
    if motion:
        t = align(0, torch.zeros((n, 2), device=DEV, dtype=F64))
        p[:, [2, 5] if motion == 3 else [0, 1]] = t
    p = align(motion, p)
    sx, sy = _map64(motion, p, w, h)
    g, m = _remap64(Cu[0], sx, sy, "zero"), _mask64(sx, sy, w, h, 254).to(F64)
    cnt = m.sum((1, 2))
    a = (R[0] - ((R[0] * m).sum((1, 2)) / cnt)[:, None, None]) * m
    b = (g - ((g * m).sum((1, 2)) / cnt)[:, None, None]) * m
    rho = (a * b).sum((1, 2)) / ((a * a).sum((1, 2)) * (b * b).sum((1, 2))).sqrt()
    out = torch.zeros((n, 6), device=DEV, dtype=F64)
    out[:, :npar] = p
    return out, rho


def _stack64(frames, p, motion, wts=None, wmaps=None, cubic=False):
    """Weighted average of the warped frames (n, h, w[, c]) and its coverage mask."""
    n, h, w = frames.shape[:3]
    planes = frames if frames.dim() == 4 else frames[..., None]
    num = torch.zeros((h, w, planes.shape[3]), device=DEV, dtype=F64)
    den = torch.zeros((h, w), device=DEV, dtype=F64)
    for i in range(n):
        sx, sy = _map64(motion, p[i:i + 1], w, h)
        if cubic:
            ix, iy, _, _ = _taps(sx, sy)
            m = (ix >= 1) & (ix < w - 2) & (iy >= 1) & (iy < h - 2)
        else:
            m = _mask64(sx, sy, w, h, 255)
        m = _erode5(m)[0].to(F64)
        wt = m * (wts[i] if wmaps is None else _remap64(wmaps[i:i + 1].to(F64), sx, sy, "zero", cubic)[0].clamp(min=0))
        den += wt
        for c in range(planes.shape[3]):
            num[..., c] += wt * _remap64(planes[i:i + 1, ..., c].to(F64), sx, sy, "r101", cubic)[0]
    avg = torch.where(den[..., None] > 0, num / den[..., None].clamp(min=1e-300), torch.zeros_like(num))
    return (avg if frames.dim() == 4 else avg[..., 0]), torch.where(den > 0, 255, 0).to(torch.uint8)


def _binned(x, b):
    x = x.to(F64)
    if b == 2:
        h, w = x.shape[0] // 2 * 2, x.shape[1] // 2 * 2
        x = x[:h, :w]
        x = 0.25 * (x[0::2, 0::2] + x[0::2, 1::2] + x[1::2, 0::2] + x[1::2, 1::2])
    return x


def _phase64(ref, frames, b):
    def spec(x):
        x = _binned(x, b)
        h, w = x.shape
        hann = lambda n: 0.5 - 0.5 * torch.cos(2 * math.pi * torch.arange(n, device=DEV, dtype=F64) / (n - 1))
        x = (x - x.mean()) * hann(h)[:, None] * hann(w)[None]
        return torch.fft.fft2(x, (1 << (h - 1).bit_length(), 1 << (w - 1).bit_length()))
    G, out = spec(ref), []
    N, M = G.shape
    ky, kx = (torch.fft.fftfreq(v, device=DEV, dtype=F64) for v in (N, M))
    wt = torch.exp(-2 * math.pi ** 2 * (ky[:, None] ** 2 + kx[None] ** 2))
    for f in frames:
        X = spec(f) * G.conj()
        mag = X.abs()
        r = torch.fft.ifft2(torch.where(mag > 0, X / mag.clamp(min=1e-300), torch.zeros_like(X)) * wt).real
        at = int(r.argmax())
        py, px = at // M, at % M
        v = lambda y, x: float(r[y % N, x % M])

        def fit(a, c, e):
            if min(a, c, e) > 0:
                a, c, e = math.log(a), math.log(c), math.log(e)
            d = a - 2 * c + e
            return 0.0 if d == 0 else 0.5 * (a - e) / d
        c = v(py, px)
        out.append([((px - M if px > M // 2 else px) + fit(v(py, px - 1), c, v(py, px + 1))) * b,
                    ((py - N if py > N // 2 else py) + fit(v(py - 1, px), c, v(py + 1, px))) * b, c])
    return np.array(out)


def _bayer64(s, case):
    w, h = case["w"], case["h"]
    tab = {8: [2, 1, 1, 0], 9: [1, 2, 0, 1], 10: [1, 0, 2, 1], 11: [0, 1, 1, 2]}[case["colorid"]]
    acc, cnt = torch.zeros((3, h, w), device=DEV, dtype=F64), torch.zeros((3, h, w), device=DEV, dtype=F64)
    scale = 2.0 ** -12 if case["u16"] else 1.0
    xs, ys = _grid(w, h, F64)
    for f, (tx, ty) in zip(s["frames"], s["shifts"].astype(np.float64)):
        px, py = xs + tx, ys + ty
        m = _erode5(_mask64(px[None], py[None], w, h, 255))[0]
        sx, sy = px.trunc().long(), py.trunc().long()
        m &= (px.trunc() >= 0) & (sx < w - 1) & (py.trunc() >= 0) & (sy < h - 1)
        img = f.to(F64) * scale
        ax, ay = sx + 1 - px, sy + 1 - py
        for k in range(4):
            xx, yy = (sx + (k & 1)).clamp(0, w - 1), (sy + (k >> 1)).clamp(0, h - 1)
            wt = ((1 - ax) if k & 1 else ax) * ((1 - ay) if k >> 1 else ay) * m
            ch = torch.tensor(tab, device=DEV)[((yy & 1) << 1) | (xx & 1)]
            v = img.reshape(-1)[(yy * w + xx).reshape(-1)].reshape(h, w) * wt
            for c in range(3):
                acc[c] += torch.where(ch == c, v, torch.zeros_like(v))
                cnt[c] += torch.where(ch == c, wt, torch.zeros_like(wt))
    avg = torch.where(cnt > 0, acc / cnt.clamp(min=1e-300), torch.zeros_like(acc)).permute(1, 2, 0)
    return dict(avg=avg, mask=torch.where((cnt > 0).any(0), 255, 0).to(torch.uint8))


def _focus64(fr, shifts, sigma, levels):
    n, h, w = fr.shape[:3]
    planes = fr if fr.dim() == 4 else fr[..., None]
    cn = planes.shape[3]
    sizes = [(w, h)]
    while not (levels and len(sizes) >= levels):
        nw, nh = (sizes[-1][0] + 1) // 2, (sizes[-1][1] + 1) // 2
        if min(nw, nh) <= 8:
            break
        sizes.append((nw, nh))
    acc = [torch.zeros((cn, b, a), device=DEV, dtype=F64) for a, b in sizes]
    ws = [torch.zeros((1, b, a), device=DEV, dtype=F64) for a, b in sizes]
    k = _gk(int(math.floor(sigma * 8 + 1.5)) | 1, sigma)
    for i in range(n):
        p = torch.tensor(shifts[i:i + 1].astype(np.float64), device=DEV)
        sx, sy = _map64(0, p, w, h)
        pl = torch.cat([_remap64(planes[i:i + 1, ..., c].to(F64), sx, sy, "r101") for c in range(cn)])
        gray = pl.mean(0, keepdim=True)
        q = _edge(gray[..., 2:-2, 2:-2], 2, 2, 2, 2, "clamp")  # the outermost results repeat the inner ones

        def conv(rows):
            r = torch.tensor(rows, device=DEV, dtype=F64)
            o = torch.zeros_like(gray[..., 2:-2, 2:-2])
            for y in range(5):
                for x in range(5):
                    if rows[y][x]:
                        o = o + r[y, x] * gray[..., y:h - 4 + y, x:w - 4 + x]
            return _edge(o, 2, 2, 2, 2, "clamp")
        kx = [[-1, 0, 0, 0, 1], [-2, -2, 0, 2, 2], [-4, -4, 0, 4, 4], [-2, -2, 0, 2, 2], [-1, 0, 0, 0, 1]]
        gx, gy = conv(kx), conv([list(r) for r in zip(*kx)])
        lap = conv([[0, 0, -1, 0, 0], [0, -1, -2, -1, 0], [-1, -2, 16, -2, -1], [0, -1, -2, -1, 0], [0, 0, -1, 0, 0]])
        m = 6.0 / 7.0 * 625.0 * lap * lap + 1.0 / 7.0 * (100.0 / 36.0) ** 2 * (gx * gx + gy * gy) + 1e-9
        W = _sep64(m * m, k, k, "r101")
        cur = pl
        for l in range(len(sizes)):
            if l + 1 < len(sizes):
                dn = _down64(cur, *sizes[l + 1])
                lp = cur - _up64(dn, *sizes[l])
            else:
                dn, lp = None, cur
            acc[l] += W * lp
            ws[l] += W
            if dn is not None:
                W, cur = _down64(W, *sizes[l + 1]), dn
    out = acc[-1] / ws[-1]
    for l in range(len(sizes) - 2, -1, -1):
        out = _up64(out, *sizes[l]) + acc[l] / ws[l]
    return out[0] if fr.dim() == 3 else out.permute(1, 2, 0)


def _master64(frame, colorid, kradius, dscale):
    m = frame.to(torch.int64) & 65535
    if colorid:
        m = (2 + m[0::2, 0::2] + m[0::2, 1::2] + m[1::2, 0::2] + m[1::2, 1::2]) >> 2
    for _ in range(dscale):
        if min(m.shape) < 4:
            break
        h, w = m.shape
        m = (_down64(m.to(F64)[None], (w + 1) // 2, (h + 1) // 2)[0] * 256).round().long()
        m = (m + 128) >> 8
    x = m.to(F64)[None, None]
    k, r = 2 * kradius + 1, kradius
    x = torch.nn.functional.pad(x, (r, r, r, r), mode="replicate")
    g = torch.nn.functional.max_pool2d(x, k, 1) + torch.nn.functional.max_pool2d(-x, k, 1)
    ds = 20.0 / 65535.0
    return float(ds ** 3 / g.sum() * (g ** 4).sum()) if float(g.sum()) > 0 else 0.0


def _nn2_64(raw, case):
    h, w = raw.shape
    v = raw.to(torch.int64) & 65535
    p = _edge(v[None], 1, 1, 1, 1, "r101")[0]
    up, dn, lf, rt = p[:-2, 1:-1], p[2:, 1:-1], p[1:-1, :-2], p[1:-1, 2:]
    cross = (up + dn + lf + rt + 2) >> 2
    diag = (p[:-2, :-2] + p[:-2, 2:] + p[2:, :-2] + p[2:, 2:] + 2) >> 2
    hor, ver = (lf + rt + 1) >> 1, (up + dn + 1) >> 1
    tab = {8: [2, 1, 1, 0], 9: [1, 2, 0, 1], 10: [1, 0, 2, 1], 11: [0, 1, 1, 2]}[case["colorid"]]
    t = torch.tensor(tab, device=DEV).reshape(2, 2)
    cm = t.repeat(h // 2 + 1, w // 2 + 1)[:h, :w]
    side = t.flip(1).repeat(h // 2 + 1, w // 2 + 1)[:h, :w]  # the colour of the row's other sites
    out = []
    for c in range(3):
        if c == 1:
            o = torch.where(cm == 1, v, cross)
        else:
            o = torch.where(cm == c, v, torch.where(cm != 1, diag, torch.where(side == c, hor, ver)))
        out.append(o.to(F64) / 2.0 ** case["bpp"])
    return torch.stack(out, -1)


def _inpaint64(img, msk):
    """average_pyramid_inpaint of (c, h, w) and a 0 / 1 mask (h, w)."""
    def box(a):
        h, w = a.shape[-2:]
        p = _edge(a, 1, 1, 1, 1, "clamp")
        return sum(p[..., y:y + h, x:x + w] for y in range(3) for x in range(3))

    def fill(src, m, fb_src, fb_m):
        d, s = box(src), box(m[None])[0]
        fb, div = fb_m != 0, (fb_m == 0) & (s != 0)
        d = torch.where(fb, fb_src, torch.where(div, d / torch.where(div, s, torch.ones_like(s)), d))
        return d, torch.where(fb | div, torch.ones_like(s), s)
    h, w = msk.shape
    if min(h, w) <= 1:
        return img, msk
    a, m = fill(img, msk, img, msk)
    ys = torch.clamp(2 * torch.arange((h + 1) // 2, device=DEV) + 1, max=h - 1)
    xs = torch.clamp(2 * torch.arange((w + 1) // 2, device=DEV) + 1, max=w - 1)
    a, m = a[:, ys][:, :, xs], m[ys][:, xs]
    if not bool((m != 0).all()):
        a, m = _inpaint64(a, m)
    up, one = torch.zeros_like(img), torch.zeros_like(msk)
    up[:, 1::2, 1::2] = a[:, :h // 2, :w // 2]
    one[1::2, 1::2] = 1
    return fill(up, one, img, msk)


def _lowpass64(x, sigma):
    h, w = x.shape[-2:]
    level, ci = 0, 0
    if sigma > 2:
        top, c = int(math.log2(min(w, h))), int(sigma * sigma / 2)
        while level < top and 1 + 4 * ci <= c:
            ci = 1 + 4 * ci
            level += 1
    delta = math.sqrt(sigma * sigma - 2 * ci) / (1 << level) if level else sigma
    sizes = []
    for _ in range(level):
        sizes.append((x.shape[-1], x.shape[-2]))
        x = _down64(x, (x.shape[-1] + 1) // 2, (x.shape[-2] + 1) // 2, "mirror")
    if delta > 0:
        k = _gk(2 * max(1, int(delta * 5)) + 1, delta)
        x = _sep64(x, k, k, "mirror")
    for s in reversed(sizes):
        x = _up64(x, *s)
    return x


def exact(case, seed):
    f = case["family"]
    s = _inputs(case, seed)
    if f in ("frame", "stack", "stack_batch"):
        # the forward-additive aligner at full size; larger batches would take too long
        if case.get("method", 0) or case["scale"] != 1.0 or case.get("n", 1) * case["w"] * case["h"] > 24_000_000:
            return None
        p, rho = _ecc64(s["ref"], s["frames"], case["motion"], case["levels"], case["eps"])
        if f == "frame":
            return dict(ok=None, params=p[0], rho=float(rho[0]))
        x = s["frames"].to(F64)
        q = _edge(x, 1, 1, 1, 1, "clamp")
        lap = q[:, :-2, 1:-1] + q[:, 2:, 1:-1] + q[:, 1:-1, :-2] + q[:, 1:-1, 2:] - 4 * x
        wts = (lap ** 2).mean((1, 2))
        avg, mask = _stack64(s["frames"], p[:, :{0: 2, 1: 3, 2: 4, 3: 6}[case["motion"]]], case["motion"], wts)
        if f == "stack":
            return dict(params=p, rho=rho, weights=wts, avg=avg, mask=mask)
        return dict(params=p, rho=rho, avg=avg, mask=mask)
    if f == "align":
        if case["n"] * case["w"] * case["h"] > 24_000_000 or case["scale"] != 1.0:
            return None
        x = s["frames"].to(F64)
        gray = 0.114 * x[..., 0] + 0.587 * x[..., 1] + 0.299 * x[..., 2]
        p, rho = _ecc64(gray[0], gray, 0, case["levels"], case["eps"])
        return dict(params=p[:, :2], rho=rho)
    if f == "turbulence":
        # the flow's many stages are not restated here; the shifts it starts from are
        return dict(shifts=_phase64(s["ref"], s["frames"], 1), maps=None, avg=None, mask=None)
    if f == "phasecorr":
        return _phase64(s["ref"], s["frames"], case["binning"])
    if f == "bayer":
        return _bayer64(s, case)
    if f == "focus":
        return [_focus64(fr, sh, case["sigma"], case["levels"]) for fr, sh in s["seqs"]]
    if f == "master":
        return np.array([_master64(x, case["colorid"], case["kradius"], case["dscale"]) for x in s["frames"]])
    if f == "input":
        if case["dark"] or case["algorithm"] not in (-1, _lib.DEBAYER_NN2):
            return None
        return torch.stack([_nn2_64(x, case) for x in s["frames"]])
    if f == "accumulate":
        p = torch.tensor(s["params"].astype(np.float64), device=DEV)
        avg, mask = _stack64(s["frames"], p, case["motion"], s.get("weights"), s.get("wmaps"), case["interp"] == 2)
        return dict(avg=avg, mask=mask if case["interp"] == 1 else None)
    x = s["img"].to(F64)
    x = x[None] if x.dim() == 2 else x.permute(2, 0, 1)
    full, m = _inpaint64(x * (s["mask"] != 0), (s["mask"] != 0).to(F64))
    a = case["alpha"]
    out = full / (1 - a) - _lowpass64(full, case["sigma"]) * (a / (1 - a))
    lay = lambda v: v[0] if case["cn"] == 1 else v.permute(1, 2, 0)
    return dict(full=lay(full), mask=(m * 255).round().clamp(0, 255).to(torch.uint8), out=lay(out))
