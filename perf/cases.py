"""The work that programs have this renderer do, as timed cases.

Each case is a call that a program makes through the public entry points
over seeded synthetic maps and cameras (futspace_amd.scene), at the sizes of
this repository's workloads, tests and benchmark:

  frame      one camera over a resident map into a device frame
             (Context.render): the viewer's and the video maker's call
  batch      many cameras over several resident maps in one captured launch
             (Batch.replay): simulators and data-set generation
  session    two ticks of the interactive program with the sun keys held:
             keys, step (which re-shades the map), the frame to the host
  map_load   a host map pair made resident and shaded (Context.map)
  grad       autograd through the differentiable renderer: forward and
             backward with an arbitrary image gradient
  step       the fused L2 fitting step of one view (DiffRenderer.l2_step)
  fit        multi-view colour-map fitting (diff.fit): steps with Adam
  render2    the ray-march renderer (Context.render2) into a device frame
  stateless  the reference's stateless program over device maps
             (fsx_render_stateless), whose own benchmark sweeps its depth,
             columns and rows

One context serves the whole process, as in a user's program.
"""
import ctypes
import math
import random

import numpy as np
import torch

from futspace_amd import Context, View, scene, sky_color
from futspace_amd.diff import DiffRenderer, fit, planes_of
from futspace_amd.renderer import STATELESS_MAIN, Session

SUN = 0.1
TARGET_SUN = 0.3        # the fitting targets show another time of day
LR = 0.5


def listed():
    return [
        # a thumbnail or agent view: latency and a GPU that one frame does not fill
        dict(name="frame_320x240", kind="frame", rows=1024, cols=1024, bits=8, shade=0,
             w=320, h=240, n=1024),
        # the fly-through of the benchmark: the ordinary call
        dict(name="frame_1080p", kind="frame", rows=2048, cols=2048, bits=8, shade=0,
             w=1920, h=1080, n=2048),
        # a window of odd size over a cropped map: no power of two, no whole tile
        dict(name="frame_odd", kind="frame", rows=1000, cols=1500, bits=8, shade=1000,
             w=1363, h=767, n=1531),
        # a large display over a large 16-bit map
        dict(name="frame_4k_u16", kind="frame", rows=4096, cols=4096, bits=16, shade=4096,
             w=3840, h=2160, n=4096),
        # the benchmark's batch: 256 views of mixed size and depth, four maps
        dict(name="batch_256", kind="batch", maps=4, views=256),
        # walking with the sun keys held in the default 1024 x 1024 window
        dict(name="session_sun", kind="session", rows=1024, cols=1024, w=1024, h=1024),
        # loading the benchmark's map
        dict(name="map_load_2048", kind="map_load", rows=2048, cols=2048, bits=8, shade=0),
        # a renderer inside a torch model: forward and backward
        dict(name="grad_800x600", kind="grad", rows=1024, cols=1024, bits=8, w=800, h=600, n=1024),
        # the gradient workload of the benchmark in one fused call
        dict(name="step_720p", kind="step", rows=2048, cols=2048, bits=8, w=1280, h=720, n=2048,
             image=True),
        # fitting a map to 4K photographs
        dict(name="fit_4k_u16", kind="fit", rows=4096, cols=4096, bits=16, w=3840, h=2160, n=4096,
             views=4, steps=3),
        # the ray-march renderer at its default reach
        dict(name="render2_800x600", kind="render2", rows=1024, cols=1024, bits=8, w=800, h=600,
             distance=800.0),
        # the stateless program's row sweep
        dict(name="stateless_rows", kind="stateless", rows=1024, cols=1024, w=800, h=50000,
             distance=800.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _map_sides(rng, hi):
    """A power-of-two square map, or a cropped one of odd sides."""
    if rng.random() < 0.6:
        s = 1 << rng.randint(9, hi.bit_length() - 1)
        return s, s
    return _log(rng, 300, hi), _log(rng, 300, hi)


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "batch", "session", "map_load", "grad", "step",
                       "step", "fit", "render2", "stateless"])
    bits = rng.choice([8, 8, 16])
    if kind == "frame":
        rows, cols = _map_sides(rng, 4096)
        return dict(kind=kind, rows=rows, cols=cols, bits=bits,
                    shade=rng.choice([0, min(rows, cols), _log(rng, 300, 2048)]),
                    w=_log(rng, 64, 3840), h=_log(rng, 48, 2160), n=_log(rng, 256, 4096))
    if kind == "batch":
        return dict(kind=kind, maps=rng.randint(1, 3), views=_log(rng, 4, 200))
    if kind == "session":
        rows, cols = _map_sides(rng, 2048)
        return dict(kind=kind, rows=rows, cols=cols, w=_log(rng, 128, 1920),
                    h=_log(rng, 96, 1080))
    if kind == "map_load":
        rows, cols = _map_sides(rng, 2048)
        return dict(kind=kind, rows=rows, cols=cols, bits=bits,
                    shade=rng.choice([0, min(rows, cols), _log(rng, 300, 2048)]))
    if kind in ("grad", "step"):
        rows, cols = _map_sides(rng, 2048)
        c = dict(kind=kind, rows=rows, cols=cols, bits=bits, w=_log(rng, 64, 1920),
                 h=_log(rng, 48, 1080), n=_log(rng, 256, 2048))
        return dict(c, image=rng.random() < 0.5) if kind == "step" else c
    if kind == "fit":
        rows, cols = _map_sides(rng, 2048)
        return dict(kind=kind, rows=rows, cols=cols, bits=bits, w=_log(rng, 160, 2560),
                    h=_log(rng, 120, 1440), n=_log(rng, 512, 4096), views=rng.randint(1, 4),
                    steps=rng.randint(1, 3))
    if kind == "render2":
        rows, cols = _map_sides(rng, 2048)
        return dict(kind=kind, rows=rows, cols=cols, bits=bits, w=_log(rng, 64, 1280),
                    h=_log(rng, 48, 720), distance=float(_log(rng, 100, 1000)))
    rows, cols = _map_sides(rng, 2048)
    sweep = rng.choice(["depth", "columns", "rows"])
    return dict(kind=kind, rows=rows, cols=cols,
                w=_log(rng, 10, 50000) if sweep == "columns" else 800,
                h=_log(rng, 10, 50000) if sweep == "rows" else 400,
                distance=float(_log(rng, 10, 100000)) if sweep == "depth" else 800.0)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

_context = None


def _ctx():
    global _context
    if _context is None:
        _context = Context()
    return _context


def _max_height(case):
    return 255 if case.get("bits", 8) == 8 else 1024


def _maps(case, seed):
    """(colour u32, height i32) of the case's size, cropped from a square scene."""
    side = 1 << (max(case["rows"], case["cols"]) - 1).bit_length()
    col, hts = scene.scene_maps(seed + 1, side, _max_height(case))
    cut = (slice(0, case["rows"]), slice(0, case["cols"]))
    return np.ascontiguousarray(col[cut]), np.ascontiguousarray(hts[cut])


def _shade_size(case):
    """The differentiable cases fit the full-resolution colour map: its
    planes are square, of the map's smaller side."""
    return min(case["rows"], case["cols"])


def _view(case, rng, hts):
    """A camera above the ground anywhere on the map."""
    rows, cols = hts.shape
    x, y = rng.uniform(0, cols), rng.uniform(0, rows)
    alt = scene.above_ground(rng.uniform(120.0, 400.0), hts, x, y)
    d, z0 = scene.depth_for(case["n"])
    return View(x=x, y=y, height=alt, angle=rng.uniform(0.0, 2.0 * math.pi),
                horizon=rng.uniform(0.1, 0.3) * case["h"], distance=1000.0, fov=1.2,
                sky_color=sky_color(SUN), h=case["h"], w=case["w"], d=d, z0=z0, scale=0.0,
                n_slices=case["n"])


def _frame(h, w):
    return torch.zeros((h, w), dtype=torch.int32, device="cuda")


def prepare(case, seed):
    rng = random.Random(seed)
    kind = case["kind"]
    ctx = _ctx()
    s = dict(kind=kind, ctx=ctx, case=case)
    if kind == "batch":
        sizes = scene.BATCH_MAP_SIZES[:case["maps"]]
        data = [scene.scene_maps(seed + 1 + i, n) for i, n in enumerate(sizes)]
        maps = [ctx.map(c, h) for c, h in data]
        views = scene.batched_views([h for _, h in data], case["views"], seed + 1)
        # the cameras, depths and maps are the seed's, the sizes the case's
        for i, v in enumerate(views):
            v.h, v.w = scene.BATCH_RESOLUTIONS[i % len(scene.BATCH_RESOLUTIONS)]
        offs, total = scene.batch_offsets(views)
        s["out"] = torch.zeros(total, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        s["batch"] = ctx.batch(maps, views, s["out"], offs)
        s["batch"].capture()
        return s
    col, hts = _maps(case, seed)
    if kind == "map_load":
        s.update(col=col, hts=hts)
        return s
    if kind == "session":
        s["session"] = Session(ctx)
        s["session"].update_map(col, hts)
        s["session"].resize(case["h"], case["w"])
        for _ in range(rng.randint(1, 8)):       # walk a little from the fixed start
            for down in (True, False):
                s["session"].key(down, rng.choice("wa"))
                s["session"].step()
        return s
    if kind == "stateless":
        dev = [torch.from_numpy(np.asarray(a, np.uint32).astype(np.int32)).cuda()
               for a in (col & 0xFFFFFF, hts)]
        s.update(color=dev[0], height=dev[1], out=_frame(case["h"], case["w"]))
        m = STATELESS_MAIN
        x, y = rng.uniform(0, case["cols"]), rng.uniform(0, case["rows"])
        s["view"] = View(x=x, y=y, height=scene.above_ground(m.height, hts, x, y),
                         angle=rng.uniform(0.0, 2.0 * math.pi), horizon=m.horizon,
                         distance=case["distance"], fov=m.fov, sky_color=m.sky_color,
                         h=case["h"], w=case["w"])
        torch.cuda.synchronize()
        return s
    if kind == "frame":
        s["map"] = ctx.map(col, hts, case["bits"], case["shade"])
        s["view"] = _view(case, rng, hts)
        s["out"] = _frame(case["h"], case["w"])
        torch.cuda.synchronize()
        return s
    if kind == "render2":
        s["map"] = ctx.map(col, hts, case["bits"])
        x, y = rng.uniform(0, case["cols"]), rng.uniform(0, case["rows"])
        s["view"] = View(x=x, y=y, height=scene.above_ground(rng.uniform(120.0, 300.0), hts, x, y),
                         angle=rng.uniform(0.0, 2.0 * math.pi), horizon=rng.uniform(0.0, 10.0),
                         distance=case["distance"], h=case["h"], w=case["w"])
        s["out"] = _frame(case["h"], case["w"])
        torch.cuda.synchronize()
        return s

    # the differentiable renderer: square planes of the map's smaller side
    side = _shade_size(case)
    s["map"] = ctx.map(col, hts, case["bits"], side)
    r = s["renderer"] = DiffRenderer(ctx, s["map"])
    planes = torch.from_numpy(planes_of(col[:side, :side])).cuda()
    gen = torch.Generator(device="cuda").manual_seed(seed + 1)
    views = s["views"] = [_view(case, rng, hts) for _ in range(case.get("views", 1))]
    s["planes"] = planes
    if kind == "grad":
        v = views[0]
        s["planes"] = planes.requires_grad_(True)
        s["shading"] = torch.tensor([SUN, SUN], requires_grad=True)
        s["gimg"] = torch.randn((3, v.h, v.w), generator=gen, device="cuda")
        torch.cuda.synchronize()
        return s
    noise = torch.randn(planes.shape, generator=gen, device="cuda") * (8.0 / 255.0)
    target_planes = (planes + noise).clamp_(0.0, 1.0)
    s["targets"] = [r.forward_raw(target_planes, TARGET_SUN, v)[0] for v in views]
    if kind == "step":
        v = views[0]
        f32 = dict(dtype=torch.float32, device="cuda")
        s["src"] = _frame(v.h, v.w)
        s["img"] = torch.empty((3, v.h, v.w), **f32) if case["image"] else None
        s["gimg"] = torch.empty((3, v.h, v.w), **f32) if case["image"] else None
        s["gplanes"] = torch.empty_like(planes)
        s["gsky"], s["loss"] = torch.empty(1, **f32), torch.empty(1, **f32)
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def _tick(session, keys):
    """One tick of the interactive loop with `keys` held: events, step, frame."""
    for k in keys:
        session.key(True, k)
    session.step()
    frame = session.render()
    for k in keys:
        session.key(False, k)
    return frame


def run(s):
    kind, ctx = s["kind"], s["ctx"]
    if kind == "frame":
        return ctx.render(s["map"], s["view"], s["out"])
    if kind == "render2":
        return ctx.render2(s["map"], s["view"], s["out"])
    if kind == "batch":
        s["batch"].replay()
        return s["out"]
    if kind == "stateless":
        c, cv = s["case"], s["view"].to_c()
        ctx.check(ctx.lib.fsx_render_stateless(
            ctx.ptr, ctypes.c_void_p(s["color"].data_ptr()),
            ctypes.c_void_p(s["height"].data_ptr()), c["rows"], c["cols"], ctypes.byref(cv),
            ctypes.c_void_p(s["out"].data_ptr())), "fsx_render_stateless")
        return s["out"]
    if kind == "session":
        # forwards under a rising sun, and back under a setting one
        frames = [_tick(s["session"], "wu"), _tick(s["session"], "sj")]
        return {"frames": frames, "text": s["session"].text_content()}
    if kind == "map_load":
        c = s["case"]
        m = ctx.map(s["col"], s["hts"], c["bits"], c["shade"])
        shaded = m.shaded()
        m.close()
        return shaded
    r = s["renderer"]
    if kind == "grad":
        img = r.render(s["planes"], s["shading"], s["views"][0])
        gplanes, gshading = torch.autograd.grad(img, [s["planes"], s["shading"]], s["gimg"])
        return {"img": img.detach(), "gplanes": gplanes, "gshading": gshading}
    if kind == "step":
        img, src, gplanes, gsky, loss = r.l2_step(
            s["planes"], SUN, s["views"][0], s["targets"][0], s["img"], s["src"], s["gimg"],
            s["gplanes"], s["gsky"], s["loss"], outputs=s["case"]["image"])
        return {"img": img, "src": src, "gimg": s["gimg"], "gplanes": gplanes, "gsky": gsky,
                "loss": loss}
    planes = s["planes"].clone()
    losses = fit(r, planes, s["views"], s["targets"], SUN, s["case"]["steps"], lr=LR)
    return {"planes": planes, "losses": losses}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    """bytes: the map texels a pass can touch read once (at most what its
    samples read), its other inputs once, its outputs once.  flops: the
    bilinear height, projection and occlusion of each (slice, column) sample
    (about 25), the colour of each shown pixel's sample (about 60, counted
    once per four pixels), and the passes' own arithmetic."""
    kind = case["kind"]
    if kind == "batch":
        sizes = [scene.BATCH_RESOLUTIONS[i % len(scene.BATCH_RESOLUTIONS)]
                 for i in range(case["views"])]
        px = sum(h * w for h, w in sizes)
        samples = 2560 * sum(w for _, w in sizes)        # of the mean depth
        texels = sum(n * n for n in scene.BATCH_MAP_SIZES[:case["maps"]])
        return {"bytes": min(texels, 4 * samples) + 4 * px + 4 * (1 << 20) * case["maps"],
                "flops": 25 * samples + 15 * px}
    texels = case["rows"] * case["cols"]
    hb = case.get("bits", 8) // 8
    if kind in ("map_load", "session"):
        shade = case.get("shade") or 1024
        # 255 sun-ray steps bound a texel's shadow; a ray above the highest
        # terrain is done, which a quarter of them reaches
        reshade = dict(bytes=8 * shade * shade, flops=64 * 6 * shade * shade)
        if kind == "map_load":
            return {"bytes": 8 * texels + reshade["bytes"], "flops": reshade["flops"]}
        px = 2 * case["w"] * case["h"]
        return {"bytes": 2 * reshade["bytes"] + 4 * px, "flops": 2 * reshade["flops"]}
    px = case["w"] * case["h"]
    if kind == "stateless":
        n = min(600, max(1, int(math.sqrt(400 * case["distance"]))))
        samples = case["w"] * n
        return {"bytes": 4 * px + min(8 * texels, 8 * samples), "flops": 12 * samples}
    if kind == "render2":
        samples = case["w"] * (int(case["distance"] / 4) + 1)
        return {"bytes": 4 * px + min((hb + 4) * texels, 4 * hb * samples + 16 * px),
                "flops": 25 * samples + 15 * px}
    samples = case["w"] * case["n"]
    heights = min(hb * texels, 4 * hb * samples)
    if kind == "frame":
        shade = case["shade"] or 1024
        return {"bytes": 4 * px + heights + min(4 * shade * shade, 16 * px),
                "flops": 25 * samples + 15 * px}
    planes = 3 * _shade_size(case) ** 2
    touched = min(4 * 4 * planes // 3, 16 * px)      # the planes' and shade factors' texels
    if kind == "grad":
        # img out, its gradient in, the visible slice between the two passes
        return {"bytes": heights + touched + (12 + 12 + 4) * px + 4 * planes,
                "flops": 25 * samples + 45 * px}
    image = 24 if case.get("image") else 0
    one = {"bytes": heights + touched + (12 + 4 + image) * px, "flops": 25 * samples + 45 * px}
    if kind == "step":
        return {"bytes": one["bytes"] + 4 * planes, "flops": one["flops"]}
    # fit: the visible slices once per view, the colours and gradients of
    # each step, and Adam over parameter, gradient and moments
    k, v = case["steps"], case["views"]
    return {"bytes": v * heights + k * v * (touched + 12 * px) + k * 4 * 7 * planes,
            "flops": 25 * samples * v + k * v * 45 * px + k * 15 * planes}


# ---------------------------------------------------------------------------
# The same results in 64 bits
# ---------------------------------------------------------------------------

def _coords(v):
    """The f32 map coordinates x, y [n][w] of every (slice, column) sample
    and the slices' inverse depths: they define which texels a frame mixes,
    so they keep the renderer's f32 steps."""
    f = np.float32
    ang, fov = f(v.angle), f(v.fov)
    sin, cos = f(math.sin(float(ang))), f(math.cos(float(ang)))
    lx, ly = f(f(-cos) - f(sin * fov)), f(sin - f(cos * fov))
    rx, ry = f(cos - f(sin * fov)), f(f(-sin) - f(cos * fov))
    i = np.arange(1, v.n_slices + 1, dtype=np.float32)
    z = (i / f(2)) * ((f(2) * f(v.z0)) + ((i - f(1)) * f(v.d)))
    x0, y0, x1, y1 = lx * z, ly * z, rx * z, ry * z
    w = f(v.w)
    table = [x0 + f(v.x), y0 + f(v.y), (x1 - x0) / w, (y1 - y0) / w, (f(1) / z) * f(v.w // 2)]
    sx, sy, dx, dy, iz = (torch.from_numpy(t).cuda()[:, None] for t in table)
    col = torch.arange(v.w, dtype=torch.float32, device="cuda")[None, :]
    return sx + col * dx, sy + col * dy, iz


def _visible(v, hts):
    """The slice shown at each pixel ([h][w], -1 for sky) and the samples'
    coordinates: front to back a sample shows if it rises above everything
    nearer, down to the next shown one; at an integral coordinate it is
    transparent."""
    x, y, iz = _coords(v)
    rows, cols = hts.shape
    fx, cx, fy, cy = x.floor(), x.ceil(), y.floor(), y.ceil()
    h = torch.from_numpy(hts).cuda().float()
    ix, iy = fx.long() % cols, fy.long() % rows
    jx, jy = (fx.long() + 1) % cols, (fy.long() + 1) % rows
    top = (cx - x) * h[iy, ix] + (x - fx) * h[iy, jx]
    low = (cx - x) * h[jy, ix] + (x - fx) * h[jy, jx]
    hgt = (cy - y) * top + (y - fy) * low
    rel = (torch.tensor(v.height, dtype=torch.float32) - hgt) * iz + \
        torch.tensor(v.horizon, dtype=torch.float32)
    row = rel.clamp(0.0, float(v.h)).int()
    front = torch.full_like(row, v.h)
    front[1:] = row.cummin(dim=0).values[:-1].clamp(max=v.h)
    shows = (row < front) & (fx != cx) & (fy != cy)
    k, c = shows.nonzero(as_tuple=True)
    at = torch.full((v.h, v.w), -1, dtype=torch.long, device="cuda")
    at[row[k, c].long(), c] = k
    idx = torch.arange(v.h, device="cuda")[:, None]
    last = torch.where(at >= 0, idx, -1).cummax(dim=0).values
    src = torch.where(last >= 0, at.gather(0, last.clamp(min=0)), -1)
    return src, x, y


def _shade_factor(hts, size):
    """sqrt(1 / (4 count + 1)) in 64 bits; the shadow counts are whole
    numbers, from the f32 rays that define them."""
    f = np.float32
    sh, ch, sa, ca = (f(t(float(f(SUN)))) for t in (math.sin, math.cos, math.sin, math.cos))
    s0, s1, s2 = f(ca * f(-sh)), ch, f(f(-sa) * f(-sh))
    h = torch.from_numpy(hts).cuda().float()
    rows, cols = hts.shape
    g = torch.arange(size, device="cuda")
    fx, fy = g.float()[None, :], g.float()[:, None]
    base = h[(g % rows)[:, None], (g % cols)[None, :]]
    count = torch.zeros((size, size), device="cuda")
    for dist in range(1, 256):
        t = f(dist) * f(4)
        ix = (fx + float(t * s0)).trunc().long() % cols
        iy = (fy + float(t * s2)).trunc().long() % rows
        count += ((base + float(t * s1)) - h[iy, ix]) < -0.5
    return (1.0 / (4.0 * count.double() + 1.0)).sqrt()


class _Exact:
    """The differentiable renderer of one view, in 64 bits."""

    def __init__(self, v, hts, sf):
        self.src, x, y = _visible(v, hts)
        n = sf.shape[0]
        self.sf, self.n = sf.reshape(-1), n
        r, c = (self.src >= 0).nonzero(as_tuple=True)
        k = self.src[r, c]
        self.at = r * v.w + c
        x, y = x[k, c].double(), y[k, c].double()
        fx, cx, fy, cy = x.floor(), x.ceil(), y.floor(), y.ceil()
        wx, wy = ((cx - x) / (cx - fx), (x - fx) / (cx - fx)), \
                 ((cy - y) / (cy - fy), (y - fy) / (cy - fy))
        ax, ay = (fx.long() % n, cx.long() % n), (fy.long() % n, cy.long() % n)
        self.t = [ay[j] * n + ax[i] for j in (0, 1) for i in (0, 1)]
        self.wt = [wy[j] * wx[i] for j in (0, 1) for i in (0, 1)]
        # sums by texel: sorted once, then differences of a running sum (near
        # texels cover whole screens, where adding one by one would queue up)
        self.sums = []
        for t in self.t:
            order = t.argsort()
            key, count = t[order].unique_consecutive(return_counts=True)
            self.sums.append((order, key, count.cumsum(0) - 1))
        self.shape = (v.h, v.w)
        self.base = [144.0 / 255.0, 144.0 / 255.0, 224.0 / 255.0]

    def texel(self, plane, i):
        return plane.reshape(-1)[self.t[i]] * self.sf[self.t[i]]

    def colour(self, plane):
        return sum(self.wt[i] * self.texel(plane, i) ** 2 for i in range(4)).sqrt()

    def image(self, planes, sky):
        img = torch.empty((3,) + self.shape, dtype=torch.float64, device="cuda")
        for ch in range(3):
            img[ch] = self.base[ch] * sky
            img[ch].view(-1)[self.at] = self.colour(planes[ch])
        return img

    def adjoint(self, planes, gimg, gplanes):
        """Adds dL/dplanes into gplanes; returns dL/dsky."""
        shown = self.src >= 0
        gsky = 0.0
        for ch in range(3):
            gsky = gsky + self.base[ch] * gimg[ch][~shown].sum()
            px = self.colour(planes[ch])
            q = torch.where(px > 0, gimg[ch].reshape(-1)[self.at] / px, torch.zeros_like(px))
            for i, (order, key, end) in enumerate(self.sums):
                g = q * self.wt[i] * self.sf[self.t[i]] * self.texel(planes[ch], i)
                total = g[order].cumsum(0)[end]
                total[1:] -= total[:-1].clone()
                gplanes[ch].view(-1)[key] += total
        return gsky


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("grad", "step", "fit"):
        return None                 # whole numbers: equal to the start's
    s = prepare(case, seed)
    _, hts = _maps(case, seed)
    sf = _shade_factor(hts, _shade_size(case))
    views = [_Exact(v, hts, sf) for v in s["views"]]
    planes = s["planes"].detach().double()
    grad = torch.zeros_like(planes)
    sky = float(np.float32(SUN))
    if kind == "grad":
        img = views[0].image(planes, sky)
        gsky = views[0].adjoint(planes, s["gimg"].double(), grad)
        gshading = torch.zeros(2, dtype=torch.float64)
        gshading[0] = gsky.cpu()
        return {"img": img, "gplanes": grad, "gshading": gshading}
    if kind == "step":
        img = views[0].image(planes, sky)
        d = img - s["targets"][0].double()
        gsky = views[0].adjoint(planes, 2.0 * d, grad)
        image = case["image"]
        return {"img": img if image else None, "src": None, "gimg": 2.0 * d if image else None,
                "gplanes": grad, "gsky": gsky.reshape(1), "loss": (d * d).sum().reshape(1)}
    losses = torch.zeros(case["steps"], dtype=torch.float64, device="cuda")
    m, v2 = torch.zeros_like(planes), torch.zeros_like(planes)
    for it in range(case["steps"]):
        grad.zero_()
        for e, t in zip(views, s["targets"]):
            d = e.image(planes, sky) - t.double()
            losses[it] += (d * d).sum()
            e.adjoint(planes, 2.0 * d, grad)
        m = 0.9 * m + 0.1 * grad
        v2 = 0.999 * v2 + 0.001 * grad * grad
        mh, vh = m / (1.0 - 0.9 ** (it + 1)), v2 / (1.0 - 0.999 ** (it + 1))
        planes = (planes - (LR / 255.0) * mh / (vh.sqrt() + 1e-8)).clamp(0.0, 1.0)
    return {"planes": planes, "losses": losses}
