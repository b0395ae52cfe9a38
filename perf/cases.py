"""Performance cases of the view-synthesis path.

Every case is a piece of work a program using this library has it do, through
the Python binding's public entry points: single views, batches of views,
frames of a video (new sources each pass), requests served to host memory, the
per-stage calls and the loading stages.  Sizes are those of the repository's
own workloads (2 x 640x480 perspective; 4 and 11 equirectangular 4096x2048; 11
perspective 2048x2048; targets from 720p to 8192x4096) or generic ragged ones.

Inputs are synthetic scenes (textured spheres in a box, textured rectangles
before a plane) ray-cast on the GPU for the rig's cameras and handed over as
the raw YUV420 and inverse-depth planes a file would hold.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rvs-cuda_amd", "python"))

import rvs_amd as R  # noqa: E402
import serving as S  # noqa: E402
import workloads as W  # noqa: E402

_BASE = dict(kind="view", scene="spheres", src="erp", ns=4, sw=4096, sh=2048, bd=10, tgt="persp", sizes="1920x1080",
             n=1, exp=1.0, rescale=1.0, tile=0, maps=False, color=False)


def _case(name, **kw):
    c = dict(_BASE, **kw)
    c["name"] = name
    return c


def listed():
    return [
        # the smallest call: a stereo pair of 8-bit perspective VGA views, the
        # view between them, with the float colour map a pipeline's hook reads
        _case("view_vga_persp2", scene="rects", src="persp", ns=2, sw=640, sh=480, bd=8, sizes="640x480", color=True),
        # the plain per-view path: one 1080p viewport of four resident panoramas
        _case("view_1080p_erp4", color=True),
        # a video frame: four panoramas newly loaded, then their 2048x2048 viewport
        _case("frame_2048_erp4", kind="frame", sizes="2048x2048"),
        # a batch of like viewports in one launch set, at the tile edge the autotuner picks
        _case("batch8_1080p_erp4", kind="batch", n=8, tile=32),
        # a batch of uneven viewports, ragged ones among them
        _case("batch16_mixed_erp4", kind="batch", n=16, sizes="1280x720,1920x1080,1366x766,3840x2160,854x482"),
        # 4K viewports of a camera array: many sources, wide disocclusions at the borders
        _case("batch2_4k_persp11", kind="batch", src="persp", ns=11, sw=2048, sh=2048, n=2, sizes="3840x2160"),
        # panoramas from panoramas (wrapping seam, nothing culled)
        _case("batch2_2k_erp_erp4", kind="batch", tgt="erp", n=2, sizes="2048x1024"),
        # the largest view served: an 8K panorama of eleven
        _case("view_8k_erp_erp11", ns=11, tgt="erp", sizes="8192x4096"),
        # an oversampled view with a steep blend and all its maps, from 8-bit views
        _case("view_720p_precision", src="persp", ns=5, sw=1280, sh=960, bd=8, sizes="1280x720", exp=5.0, rescale=1.5,
              maps=True, color=True),
        # the per-stage calls in the reference's order on a new frame of odd-sized
        # views, with multispectral blending
        _case("stages_multispec_persp4", kind="stages", src="persp", ns=4, sw=1021, sh=767, sizes="1366x766"),
        # loading a frame: colour and depth decoded, reprojected into the target
        # camera, and colour encoded again
        _case("load_2048_persp", kind="load", src="persp", ns=1, sw=2048, sh=2048, sizes="2048x2048"),
        # requests served to host memory: batches in flight on two slots
        _case("served16_1080p_erp4", kind="served", n=16),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["view", "view", "view", "batch", "batch", "frame", "stages", "load", "served"])
    c = dict(_BASE, kind=kind)
    c["scene"] = "spheres"
    c["src"] = rng.choice(["persp", "erp"])
    if kind == "load":
        c["src"] = "persp"
    c["bd"] = rng.choice([8, 10, 10])
    c["ns"] = 1 if kind == "load" else rng.choice([2, 3, 4, 4, 5, 7, 11])
    if c["src"] == "erp":
        c["sh"] = int(_log(rng, 256, 2048))
        c["sw"] = 2 * c["sh"] - rng.choice([0, 0, 1])
    else:
        c["sw"] = int(_log(rng, 320, 2048))
        c["sh"] = int(c["sw"] * rng.uniform(0.55, 1.0))
    if kind not in ("stages", "load"):
        c["sw"] -= c["sw"] % 2
        c["sh"] -= c["sh"] % 2
    if c["src"] == "persp" and c["ns"] == 2 and kind == "view" and rng.random() < 0.5:
        c["scene"] = "rects"
    c["tgt"] = rng.choice(["persp", "persp", "erp"]) if c["src"] == "erp" and kind in ("view", "batch") else "persp"
    c["n"] = {"batch": rng.randint(2, 16), "served": rng.randint(4, 16)}.get(kind, 1)
    sizes = []
    for _ in range(rng.randint(1, 4) if c["n"] > 1 else 1):
        w = 2 * int(_log(rng, 160, 1920 if c["n"] > 4 or kind != "view" else 2200) / (1 if c["n"] < 9 else 2))
        h = w // 4 * 2 if c["tgt"] == "erp" else 2 * int(w * rng.uniform(0.25, 0.5))
        sizes.append("%dx%d" % (w, h))
    c["sizes"] = ",".join(sizes)
    if kind == "load":
        c["sizes"] = "%dx%d" % (c["sw"] - c["sw"] % 2, c["sh"] - c["sh"] % 2)
    c["exp"] = rng.choice([1.0, 1.0, 2.0, 5.0])
    c["rescale"] = rng.choice([1.0, 1.0, 1.0, 1.5, 2.0]) if kind == "view" and c["tgt"] == "persp" else 1.0
    c["tile"] = rng.choice([0, 0, 16, 32]) if kind == "batch" else 0
    c["maps"] = kind == "view" and rng.random() < 0.3
    c["color"] = kind == "view" and (c["maps"] or rng.random() < 0.5)
    return c


# ------------------------------------------------------------------ scenes

def _texture(seed):
    """A 1024 x 1024 x 3 periodic map of 3-octave value noise in [0, 1]."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    out = torch.zeros((1024, 1024, 3), dtype=torch.float32, device="cuda")
    at = torch.arange(1024, device="cuda")
    for cell, weight in ((32, 4.0 / 7), (16, 2.0 / 7), (8, 1.0 / 7)):
        n = 1024 // cell
        lat = torch.rand((n, n, 3), generator=g, device="cuda")
        i0, t = at // cell, (at % cell).float() / cell
        t = t * t * (3 - 2 * t)
        i1 = (i0 + 1) % n
        rows = lat[i0] * (1 - t)[:, None, None] + lat[i1] * t[:, None, None]
        out += weight * (rows[:, i0] * (1 - t)[None, :, None] + rows[:, i1] * t[None, :, None])
    return out


def _scene(kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "rects":
        rects = []
        for _ in range(6):
            x = rng.uniform(1.0, 10.0)
            cy, cz = rng.uniform(-0.5, 0.5) * x, rng.uniform(-0.4, 0.4) * x
            hy, hz = rng.uniform(0.08, 0.3, 2) * x
            rects.append((x, cy - hy, cy + hy, cz - hz, cz + hz))
        return dict(rects=rects, spheres=[], planes=[(0, 10.0)], tex=_texture(seed), near=1.0, far=10.0)
    spheres = []
    for _ in range(24):
        u, a = rng.uniform(-1, 1), rng.uniform(0, 2 * math.pi)
        d, r, s = rng.uniform(1.5, 20.0), rng.uniform(0.2, 1.5), math.sqrt(1 - u * u)
        spheres.append((d * s * math.cos(a), d * s * math.sin(a), d * u, r))
    planes = [(ax, p) for ax in range(3) for p in (-14.0, 14.0)]
    return dict(rects=[], spheres=spheres, planes=planes, tex=_texture(seed), near=0.5, far=25.0)


def _render(sc, cam, pos, bd):
    """Raw planes (y, u, v, 16-bit inverse depth) of the scene from an unrotated camera."""
    w, h = cam.w, cam.h
    f64 = dict(dtype=torch.float64, device="cuda")
    uu, vv = torch.arange(w, **f64)[None, :] + 0.5, torch.arange(h, **f64)[:, None] + 0.5
    if cam.proj == 1:
        phi, th = math.pi - 2 * math.pi * uu / w, math.pi / 2 - math.pi * vv / h
        d = (torch.cos(th) * torch.cos(phi), torch.cos(th) * torch.sin(phi), torch.sin(th).expand(h, w))
    else:
        one = torch.ones((h, w), **f64)
        d = (one, (-(uu - cam.p[0]) / cam.f[0]).expand(h, w), (-(vv - cam.p[1]) / cam.f[1]).expand(h, w))
    best = torch.full((h, w), 1e30, **f64)
    tu = torch.zeros((h, w), dtype=torch.float32, device="cuda")
    tv = torch.zeros_like(tu)

    def take(hit, t, a, b):
        m = hit & (t > 1e-6) & (t < best)
        best.copy_(torch.where(m, t, best))
        tu.copy_(torch.where(m, a.float(), tu))
        tv.copy_(torch.where(m, b.float(), tv))

    for k, (ax, p) in enumerate(sc["planes"]):
        t = (p - pos[ax]) / torch.where(d[ax].abs() < 1e-12, torch.full_like(best, 1e-12), d[ax])
        o = [i for i in range(3) if i != ax]
        take(torch.ones_like(t, dtype=torch.bool), t, (pos[o[0]] + t * d[o[0]]) * 40 + 131 * k,
             (pos[o[1]] + t * d[o[1]]) * 40 + 57 * k)
    for k, (x, y0, y1, z0, z1) in enumerate(sc["rects"]):
        t = (x - pos[0]) / d[0]
        y, z = pos[1] + t * d[1], pos[2] + t * d[2]
        take((y >= y0) & (y <= y1) & (z >= z0) & (z <= z1), t, y / x * 500 + 211 * k, z / x * 500)
    dd = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
    for k, (cx, cy, cz, r) in enumerate(sc["spheres"]):
        o = (pos[0] - cx, pos[1] - cy, pos[2] - cz)
        b = o[0] * d[0] + o[1] * d[1] + o[2] * d[2]
        disc = b * b - dd * (o[0] * o[0] + o[1] * o[1] + o[2] * o[2] - r * r)
        t = (-b - torch.sqrt(disc.clamp(min=0.0))) / dd
        q = [o[i] + t * d[i] for i in range(3)]
        take(disc >= 0, t, (q[0] - q[1]) * 85 + 173 * k, (q[2] + 0.5 * (q[0] + q[1])) * 85)
    col = sc["tex"][tv.floor().long() % 1024, tu.floor().long() % 1024]
    s = ((1 << bd) - 1) / 255.0
    dt = np.uint8 if bd <= 8 else np.uint16
    y = ((16 + 219 * col[..., 0]) * s).round()
    he, we = h // 2 * 2, w // 2 * 2
    uv = [((128 + 80 * (col[:he, :we, k].reshape(he // 2, 2, we // 2, 2).mean((1, 3)) - 0.5)) * s).round() for k in (1, 2)]
    z = best.clamp(sc["near"], sc["far"])
    q = (65535 * (1 / z - 1 / sc["far"]) / (1 / sc["near"] - 1 / sc["far"])).round()
    return [x.to(torch.int32).cpu().numpy().astype(t) for x, t in ((y, dt), (uv[0], dt), (uv[1], dt), (q, np.uint16))]


def _positions(case):
    if case["ns"] == 1:
        return [[0.0, 0.0, 0.0]]
    if case["ns"] == 2:
        return [[0.0, 0.05, 0.0], [0.0, -0.05, 0.0]]
    if case["src"] == "erp" and case["ns"] == 4:
        return [[x, y, 0.0] for x in (0.15, -0.15) for y in (0.15, -0.15)]
    return [[0.0, (k % 4 - 1.5) * 0.1, (1 - k // 4) * 0.1] for k in range(case["ns"])]


def _src_cam(case):
    w, h = case["sw"], case["sh"]
    if case["src"] == "erp":
        return R.cam(1, w, h)
    f = w * (500.0 / 640 if case["scene"] == "rects" else 1200.0 / 2048)
    return R.cam(0, w, h, f=(f, f), p=(w / 2.0, h / 2.0))


def _sizes(case):
    s = [tuple(int(x) for x in t.split("x")) for t in case["sizes"].split(",")]
    return [s[k % len(s)] for k in range(case["n"])]


def _targets(case, seed):
    rng = np.random.default_rng(seed + 77)
    walk = W.random_walk(case["n"] + 8, seed + 3)[8:]
    out = []
    for (w, h), (pos, rot) in zip(_sizes(case), walk):
        if case["scene"] == "rects":
            f = w * 500.0 / 640
            c, pos, rot = R.cam(0, w, h, f=(f, f), p=(w / 2.0, h / 2.0)), [0.0, float(rng.uniform(-0.04, 0.04)), 0.0], [0.0] * 3
        else:
            c = R.cam(1, w, h) if case["tgt"] == "erp" else W.perspective_cam(w, h)
            if case["src"] == "persp" or case["tgt"] == "erp":   # stay within the array, look ahead
                pos = [float(x) for x in rng.uniform(-0.1, 0.1, 3)]
                rot = [float(rng.uniform(-20, 20)), float(rng.uniform(-8, 8)), 0.0]
        out.append(R.make_target(c, pos, rot, case["bd"], case["exp"], R.scale_of(case["bd"]), R.scale_of(16),
                                 rescale=case["rescale"], tile=case["tile"]))
    return out


def _sources(case, seed, prep):
    sc, cam = _scene(case["scene"], seed), _src_cam(case)
    src = []
    for p in _positions(case):
        src.append(R.DeviceSource(cam, p, [0.0, 0.0, 0.0], case["bd"], 16, sc["near"], sc["far"],
                                  _render(sc, cam, p, case["bd"])))
        if prep:
            src[-1].prepare(R.scale_of(16))
    return src


# ------------------------------------------------------------------- cases

def prepare(case, seed):
    kind = case["kind"]
    src = _sources(case, seed, kind in ("view", "batch", "served"))
    tgts = _targets(case, seed)
    st = dict(case=case, src=src, tgts=tgts)
    if kind == "view":
        st["syn"] = R.Synthesizer(src, tgts[0], want_maps=case["maps"], want_color=case["color"])
    elif kind == "batch":
        st["syn"] = R.BatchSynthesizer(src, tgts, want_color=False)
    elif kind == "served":
        w, h = map(max, zip(*_sizes(case)))
        st["srv"] = S.Server([src], memory_budget=8 << 30, max_batch=8, slots=2, keep_outputs=True,
                             host_staging_bytes=8 * w * h * 3)
        st["reqs"] = [(0, t) for t in tgts]
    elif kind == "load":
        c, t = src[0].cam, tgts[0]
        f32 = dict(dtype=torch.float32, device="cuda")
        st["pose"] = R.relative_pose(src[0].pos, src[0].rot, list(t.pos), list(t.rot))
        st["out"] = dict(color=torch.empty((c.h, c.w, 3), **f32), depth=torch.empty((c.h, c.w), **f32),
                         uv=torch.empty((c.h, c.w, 2), **f32), vdepth=torch.empty((c.h, c.w), **f32))
        w, h = c.w - c.w % 2, c.h - c.h % 2
        dt = torch.uint8 if case["bd"] <= 8 else torch.int16
        st["planes"] = [torch.empty(s, dtype=dt, device="cuda") for s in ((h, w), (h // 2, w // 2), (h // 2, w // 2))]
        g = torch.Generator(device="cuda").manual_seed(seed)
        st["view"] = torch.rand((h, w, 3), generator=g, device="cuda")   # a synthesized colour map to write
    return st


def run(state):
    case, src, tgts = state["case"], state["src"], state["tgts"]
    kind = case["kind"]
    if kind in ("view", "batch"):
        return state["syn"].run()
    if kind == "frame":
        for s in src:
            s.prepare(R.scale_of(16))
        out = R.Synthesizer(src, tgts[0], want_maps=False, want_color=False).run()
        return [out["y"], out["u"], out["v"]]
    if kind == "served":
        state["srv"].run_closed(state["reqs"], 2 * 8)
        return [np.frombuffer(state["srv"].output(k), np.uint8) for k in range(case["n"])]
    if kind == "stages":
        return R.StagewiseSynthesizer(src, tgts[0], multispectral=(case["exp"], 2.0 * case["exp"])).run()
    s, o, t = src[0], state["out"], tgts[0]
    R.decode_yuv420(*s.planes[:3], s.bd_color, R.scale_of(s.bd_color), o["color"])
    R.decode_depth(s.planes[3], 16, R.scale_of(16), s.znear, s.zfar, True, o["depth"])
    R.reproject(s.cam, t.cam, state["pose"][0], state["pose"][1], o["depth"], None, 1.0, o["uv"], o["vdepth"])
    R.encode_yuv420(state["view"], s.bd_color, *state["planes"])
    return dict(o, planes=state["planes"])


def work(case):
    """Every source sample read once, every output sample written once."""
    b = 1 if case["bd"] <= 8 else 2
    px = case["sw"] * case["sh"]
    total = case["ns"] * px * (1.5 * b + 2)
    if case["kind"] == "load":
        even = (case["sw"] & ~1) * (case["sh"] & ~1)
        return {"bytes": total + px * 4 * (3 + 1 + 2 + 1) + even * (12 + 1.5 * b), "flops": 0}
    for w, h in _sizes(case):
        total += w * h * 1.5 * b
        rpx = int(0.5 + w * case["rescale"]) * int(0.5 + h * case["rescale"])
        if case["kind"] == "stages":
            total += rpx * 24   # colour, quality, depth, validity
        else:
            total += rpx * ((12 if case["color"] else 0) + (12 if case["maps"] else 0))
    return {"bytes": total, "flops": 0}


def exact(case, seed):
    """The loading stages in 64 bits: decoded colour (bilinear chroma without a
    half-pixel offset), metric depth, target coordinates and depth.  Whole
    views (winner-takes-pixel rasters, whole-number planes) have no such value."""
    if case["kind"] != "load":
        return None
    f64 = dict(dtype=torch.float64, device="cuda")
    sc, cam, t = _scene(case["scene"], seed), _src_cam(case), _targets(case, seed)[0]
    y, u, v, q = (torch.from_numpy(p.astype(np.float64)).cuda() for p in _render(sc, cam, [0.0] * 3, case["bd"]))
    h, w = y.shape

    def up(p):
        ph, pw = p.shape
        fy, fx = torch.arange(h, **f64) * (ph / h), torch.arange(w, **f64) * (pw / w)
        y0, x0 = fy.floor().long(), fx.floor().long()
        dy, dx = (fy - y0)[:, None], (fx - x0)[None, :]
        y1, x1 = (y0 + 1).clamp(max=ph - 1), (x0 + 1).clamp(max=pw - 1)
        top = p[y0][:, x0] * (1 - dx) + p[y0][:, x1] * dx
        return top * (1 - dy) + (p[y1][:, x0] * (1 - dx) + p[y1][:, x1] * dx) * dy

    color = torch.stack([y, up(u), up(v)], -1) * R.scale_of(case["bd"])
    near, far = sc["near"], sc["far"]
    d = far * near / (near + q * R.scale_of(16) * (far - near))
    uu, vv = torch.arange(w, **f64)[None, :] + 0.5, torch.arange(h, **f64)[:, None] + 0.5
    p = torch.stack([d, -d / cam.f[0] * (uu - cam.p[0]), -d / cam.f[1] * (vv - cam.p[1])], -1)
    Rm, tr = R.relative_pose([0.0] * 3, [0.0] * 3, list(t.pos), list(t.rot))
    p = p @ torch.from_numpy(Rm.astype(np.float64)).cuda().t() + torch.from_numpy(tr.astype(np.float64)).cuda()
    c = t.cam
    uv = torch.stack([-c.f[0] * p[..., 1] / p[..., 0] + c.p[0], -c.f[1] * p[..., 2] / p[..., 0] + c.p[1]], -1)
    return dict(color=color, depth=d, uv=uv, vdepth=p[..., 0], planes=[None, None, None])
