"""What a user of this library has it do, as cases whose speed is measured.

Every case is a dict of plain values; `prepare` makes what the user's program
holds before the call (surfaces in HBM, a prepared batch, a server with its
requests, host buffers), `run` is one pass through the public entry points
and returns the pixels (or the PNG file) it made.

The kinds of work, and the ranges a drawn case comes from:

  fill       one painter.fill on a resident surface (the smallest call: a
             program that draws shape by shape), 64..2048 px, 5..400 nodes
  scene      a frame of an interactive program or a map: a background and n
             ordered paths on one surface as a prepared batch, rendered
             again for every frame, 256..3840 px wide, 20..10,000 paths; with
             mix every operator class, antialiasing mode, precision and paint
             kind that the painter takes, without it the common draw
             (src_over, default antialiasing, solid and gradient paints)
  uneven     many surfaces of uneven sizes (16..1024 px, 80% RGBA8, 20%
             alpha8), each cleared and drawn on by its own 1-50 fills and
             strokes, as one batch (glyph atlases, icons, tiles)
  serve      a burst of requests at the request server: the same surfaces,
             half of them with a clip mask, results in host memory
  text       a page of text, one draw per line
  composite  SurfaceCompositor batches over whole surfaces: one operator, with
             or without an alpha8 mask, 4-byte formats, widths that are and
             are not multiples of four, or a smaller source placed at an
             offset
  paint      a whole surface painted with a (dithered) gradient
  png        a rendered surface encoded to a PNG file in host memory

Results are bytes, so every case is compared exactly."""
import ctypes as C
import math

import numpy as np
import torch

from z2d_amd import abi, gpu

FONT = "tests/golden/fonts/Inter-Regular.ttf"
WORDS = ("The quick brown fox jumps over the lázy dog; façade naïve Ærøskøbing "
         "0123456789 AVATAR Wavy typography kerning ligatures").split()

# operators of the mixed scenes: bounded ones, in integer and in float
INT_OPS = ("src_over", "src_over", "src_over", "multiply", "screen", "overlay", "darken", "lighten",
           "plus", "xor", "src_atop", "dst_out", "hard_light", "difference", "exclusion")
FLOAT_OPS = ("color_dodge", "color_burn", "soft_light", "hue", "saturation", "color", "luminosity")
COMP_OPS = ("src", "src_over", "dst_over", "src_in", "dst_in", "dst_out", "src_atop", "xor", "plus",
            "multiply", "screen", "overlay", "darken", "hard_light", "difference") + FLOAT_OPS

_ctx = None


def _context():
    """One context per program, as the library asks for one per host thread."""
    global _ctx
    if _ctx is None:
        _ctx = gpu.Context()
    return _ctx


_srv = None


def _server():
    """The program's request server, up for as long as the program is."""
    global _srv
    if _srv is None:
        _srv = gpu.Server(_context(), 16 << 30, 64)
    return _srv


# ---- the cases --------------------------------------------------------------
def listed():
    return [
        # one shape drawn by one painter call on a resident 512 px surface
        dict(name="fill_star_512", kind="fill", w=512, h=512, points=5),
        # a small window's frame: 60 shapes and a background, prepared once
        dict(name="frame_800x600_60", kind="scene", w=800, h=600, paths=60, mix=False),
        # the library's headline: a 4K frame of 10,000 paths
        dict(name="scene_4k_10k", kind="scene", w=3840, h=2160, paths=10000, mix=False),
        # a 1080p frame that uses the painter's whole range of options, ragged width
        dict(name="scene_mix_1917x1080_600", kind="scene", w=1917, h=1080, paths=600, mix=True),
        # 1024 uneven surfaces with fills and strokes in one launch
        dict(name="uneven_1024", kind="uneven", surfaces=1024, side=1024),
        # 192 requests that arrive together
        dict(name="serve_192", kind="serve", requests=192, side=1024),
        # a 4K page of text
        dict(name="text_4k_100_lines", kind="text", w=3840, h=2160, lines=100, size=18.0),
        # a layer onto a layer, the most used operator, 4096 px
        dict(name="over_4096", kind="composite", op="src_over", w=4096, h=4096, fmt=abi.RGBA,
             masked=False, x=0, y=0),
        # the same through a mask, a ragged width and another pixel format
        dict(name="overlay_mask_3837x2159", kind="composite", op="overlay", w=3837, h=2159,
             fmt=abi.ARGB, masked=True, x=0, y=0),
        # a blend mode that has to be computed in floating point
        dict(name="luminosity_4096", kind="composite", op="luminosity", w=4096, h=4096,
             fmt=abi.RGBA, masked=False, x=0, y=0),
        # a 4K background: a dithered gradient
        dict(name="gradient_dither_4k", kind="paint", w=3840, h=2160, grad="radial", dither=True),
        # a rendered 4K frame written to a PNG file
        dict(name="png_4k", kind="png", w=3840, h=2160, paths=2000, fmt=abi.RGBA),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("fill", "scene", "scene", "mix", "uneven", "serve", "text", "composite",
                       "composite", "paint", "png"))
    if kind == "fill":
        return dict(kind="fill", w=_log(rng, 64, 2048), h=_log(rng, 64, 2048),
                    points=_log(rng, 3, 200))
    if kind == "scene":
        w = _log(rng, 256, 3840)
        return dict(kind="scene", w=w, h=max(1, min(2160, int(w * rng.uniform(0.4, 1.2)))),
                    paths=_log(rng, 20, 9000), mix=False)
    if kind == "mix":
        w = _log(rng, 256, 1920)
        return dict(kind="scene", w=w, h=max(1, min(1080, int(w * rng.uniform(0.4, 1.2)))),
                    paths=_log(rng, 20, 600), mix=True)
    if kind == "uneven":
        return dict(kind="uneven", surfaces=_log(rng, 16, 1000), side=_log(rng, 64, 1024))
    if kind == "serve":
        return dict(kind="serve", requests=_log(rng, 1, 190), side=_log(rng, 64, 1024))
    if kind == "text":
        w = _log(rng, 320, 3840)
        lines = _log(rng, 1, 95)
        return dict(kind="text", w=w, h=_log(rng, 240, 2160), lines=lines,
                    size=round(rng.uniform(8.0, 40.0), 1))
    if kind == "composite":
        w, h = _log(rng, 32, 4095), _log(rng, 32, 4095)
        at = rng.random() < 0.3
        return dict(kind="composite", op=rng.choice(COMP_OPS), w=w, h=h,
                    fmt=rng.choice((abi.RGBA, abi.RGBA, abi.ARGB, abi.XRGB, abi.RGB)),
                    masked=not at and rng.random() < 0.4,
                    x=rng.randint(0, w // 2) if at else 0, y=rng.randint(0, h // 2) if at else 0)
    if kind == "paint":
        return dict(kind="paint", w=_log(rng, 64, 3840), h=_log(rng, 64, 2160),
                    grad=rng.choice(("linear", "radial", "conic")), dither=rng.random() < 0.5)
    return dict(kind="png", w=_log(rng, 128, 3840), h=_log(rng, 128, 2100),
                paths=_log(rng, 20, 1900), fmt=rng.choice((abi.RGBA, abi.RGB, abi.ALPHA8)))


# ---- inputs -------------------------------------------------------------------
def _solid(rng, fmt=abi.RGBA):
    a = int(rng.integers(64, 256))
    c = [int(round(255 * v)) * a // 255 for v in rng.random(3)]
    if fmt == abi.ALPHA8:
        return abi.solid_pattern(abi.pixel(abi.ALPHA8, a=a))
    return abi.solid_pattern(abi.rgba(c[0], c[1], c[2], a))


def _gradient(rng, x0, y0, s, method=abi.INTERP_LINEAR_RGB, gtype=None):
    gtype = int(rng.integers(0, 3)) if gtype is None else gtype
    u = rng.random(6)
    if gtype == abi.GRADIENT_LINEAR:
        geom = [x0 + s * u[0], y0 + s * u[1], x0 + s * u[2], y0 + s * u[3]]
    elif gtype == abi.GRADIENT_RADIAL:
        geom = [x0 + s * u[0], y0 + s * u[1], s / 4 * u[2], x0 + s * u[3], y0 + s * u[4],
                s * (0.25 + 0.75 * u[5])]
    else:
        geom = [x0 + s * u[0], y0 + s * u[1], 2 * math.pi * u[2]]
    n = int(rng.integers(2, 7))
    cols = rng.random((n, 4))
    stops = [(float(o), abi.color(abi.COLOR_LINEAR_RGB, *map(float, c[:3]), 0.25 + 0.75 * float(c[3])))
             for o, c in zip(np.sort(rng.random(n)), cols)]
    return abi.Gradient(gtype, geom, stops, method)


def _rect(w, h):
    a = np.zeros(6, abi.NODE_DTYPE)
    a["tag"] = [abi.MOVE_TO, abi.LINE_TO, abi.LINE_TO, abi.LINE_TO, abi.CLOSE_PATH, abi.MOVE_TO]
    a["v"][1, 0] = a["v"][2, 0] = w
    a["v"][2, 1] = a["v"][3, 1] = h
    return a


def _paths(rng, n, w, h, max_side=512.0):
    """n closed paths: 3-64 segments, 70% lines and 30% cubics, control points
    uniform in a box of log-uniform side (4..max_side px) placed uniformly.
    Returns [(nodes, x0, y0, side)]."""
    nseg = rng.integers(3, 65, n)
    side = np.exp(rng.uniform(math.log(4.0), math.log(max(4.0, max_side)), n))
    x0 = rng.random(n) * np.maximum(0.0, w - side)
    y0 = rng.random(n) * np.maximum(0.0, h - side)
    cnt = nseg + 3  # move, segments, close, final move
    off = np.concatenate([[0], np.cumsum(cnt)])
    total = int(off[-1])
    own = np.repeat(np.arange(n), cnt)
    a = np.zeros(total, abi.NODE_DTYPE)
    v = rng.random((total, 6)) * side[own][:, None]
    v[:, 0::2] += x0[own][:, None]
    v[:, 1::2] += y0[own][:, None]
    tag = np.where(rng.random(total) < 0.7, abi.LINE_TO, abi.CURVE_TO)
    first, last = off[:-1], off[1:] - 1
    tag[first] = abi.MOVE_TO
    tag[last - 1] = abi.CLOSE_PATH
    tag[last] = abi.MOVE_TO
    v[last] = v[first]
    v[tag != abi.CURVE_TO, 2:] = 0.0
    v[last - 1] = 0.0
    a["tag"] = tag
    a["v"] = v
    return [(a[off[i]:off[i + 1]], float(x0[i]), float(y0[i]), float(side[i])) for i in range(n)]


def _pattern(rng, x0, y0, s, keep, mix=False, fmt=abi.RGBA):
    u = rng.random()
    if u < 0.6:
        return _solid(rng, fmt)
    method = abi.INTERP_LINEAR_RGB
    if mix:
        method = int(rng.choice((abi.INTERP_LINEAR_RGB, abi.INTERP_LINEAR_RGB, abi.INTERP_SRGB,
                                 abi.INTERP_HSL)))
    g = _gradient(rng, x0, y0, s, method)
    keep.append(g)
    if mix and u > 0.9:
        return abi.dither_pattern(int(rng.integers(1, 3)), 8, gradient=g)
    return g.pattern()


def _fill_opts(rng, mix):
    rule = abi.NON_ZERO if rng.random() < 0.5 else abi.EVEN_ODD
    if not mix:
        return abi.fill_opts(abi.AA_DEFAULT, rule, "src_over")
    aa = int(rng.choice((abi.AA_DEFAULT, abi.AA_DEFAULT, abi.AA_DEFAULT, abi.AA_DEFAULT,
                         abi.AA_NONE, abi.AA_SUPERSAMPLE_4X)))
    if rng.random() < 0.2:
        return abi.fill_opts(aa, rule, str(rng.choice(FLOAT_OPS)), abi.PRECISION_FLOAT)
    prec = abi.PRECISION_FLOAT if rng.random() < 0.2 else abi.PRECISION_INTEGER
    return abi.fill_opts(aa, rule, str(rng.choice(INT_OPS)), prec)


def _stroke_opts(rng, keep):
    """Width 0.5-8 px, joins and caps uniform, 25% dashed."""
    o = abi.StrokeOpts()
    o.anti_aliasing_mode = abi.AA_DEFAULT
    o.line_width = float(rng.uniform(0.5, 8.0))
    o.line_join_mode = int(rng.integers(0, 3))
    o.line_cap_mode = int(rng.integers(0, 3))
    o.op = abi.OP["src_over"]
    o.precision = abi.PRECISION_INTEGER
    o.miter_limit = 10.0
    o.tolerance = 0.1
    o.transformation[:] = abi.IDENTITY
    if rng.random() < 0.25:
        n = int(rng.integers(2, 7))
        d = (C.c_double * n)(*map(float, rng.uniform(1.0, 20.0, n)))
        o.dashes = C.cast(d, C.POINTER(C.c_double))
        o.n_dashes = n
        keep.append(d)
    return o


def _jobs(rng, side, keep, fmt):
    """One uneven surface's draws: 1-50 paths, 30% of them stroked."""
    jobs = []
    for nodes, x0, y0, s in _paths(rng, int(rng.integers(1, 51)), side, side, min(512.0, side)):
        keep.append(nodes)
        pat = _pattern(rng, x0, y0, s, keep)
        if rng.random() < 0.3:
            jobs.append(("stroke", pat, nodes, _stroke_opts(rng, keep)))
        else:
            jobs.append(("fill", pat, nodes, _fill_opts(rng, False)))
    return jobs


def _uneven(n, side):
    """(format, side) of the case's n surfaces: sides log-uniform from 16 px
    up.  They belong to the case; the seed decides what is drawn on them."""
    rng = np.random.default_rng((n, side))
    sides = np.exp(rng.uniform(math.log(16.0), math.log(float(side)), n)).round().astype(int)
    return [(abi.RGBA if u < 0.8 else abi.ALPHA8, int(s)) for s, u in zip(sides, rng.random(n))]


class _Pixels:
    """A resident surface's memory as a tensor, where it is.  The tensor keeps
    this object, and so the surface, alive."""

    def __init__(self, surface):
        self.surface = surface
        d = surface.desc()
        self.__cuda_array_interface__ = dict(shape=(surface.nbytes,), typestr="|u1", version=2,
                                             data=(d.data, False), strides=None)


def _tensor(surface):
    t = torch.as_tensor(_Pixels(surface), device="cuda")
    t.surface = surface
    return t


def _surface(ctx, fmt, w, h, data=None):
    s = gpu.DeviceSurface(ctx, fmt, w, h)
    if data is None:
        data = np.zeros(s.nbytes, np.uint8)
    s.upload(data)
    return s


def _premultiplied(seed, w, h):
    """A layer's pixels: alpha uniform, colors uniform up to it."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.randint(0, 256, (h * w, 1), generator=g, device="cuda", dtype=torch.int32)
    u = torch.rand((h * w, 3), generator=g, device="cuda")
    c = torch.floor(u * (a + 1).float()).to(torch.int32).minimum(a)
    return torch.cat([c, a], 1).to(torch.uint8).cpu().numpy().reshape(-1)


def _scene(ctx, rng, w, h, paths, mix, fmt=abi.RGBA):
    """A surface and its prepared batch: an opaque background, then the paths."""
    surf = _surface(ctx, fmt, w, h)
    b = gpu.Batch(ctx)
    keep = [surf]
    if fmt == abi.ALPHA8:
        bg = (abi.solid_pattern(abi.pixel(abi.ALPHA8, a=0)), _rect(w, h),
              abi.fill_opts(abi.AA_DEFAULT, abi.NON_ZERO, "clear"))
    else:
        bg = (abi.solid_pattern(abi.rgba(255, 255, 255, 255)), _rect(w, h),
              abi.fill_opts(abi.AA_DEFAULT, abi.NON_ZERO, "src_over"))
    ctx.check(b.fill(surf, *bg), "fill")
    for nodes, x0, y0, s in _paths(rng, paths, w, h, min(512.0, max(w, h))):
        pat = _pattern(rng, x0, y0, s, keep, mix, fmt)
        ctx.check(b.fill(surf, pat, nodes, _fill_opts(rng, mix)), "fill")
    b.prepare()
    return surf, b, keep


# ---- what the program holds before the call -------------------------------------
def prepare(case, seed):
    ctx = _context()
    rng = np.random.default_rng(seed)
    k = case["kind"]
    st = dict(kind=k, ctx=ctx)
    if k == "fill":
        w, h, n = case["w"], case["h"], case["points"]
        surf = _surface(ctx, abi.RGBA, w, h, np.full(w * h * 4, 255, np.uint8))
        th = -math.pi / 2 + rng.uniform(0, 2 * math.pi) + math.pi / n * np.arange(2 * n)
        r = np.where(np.arange(2 * n) % 2 == 0, 0.47, rng.uniform(0.15, 0.4)) * min(w, h)
        nodes = np.zeros(2 * n + 2, abi.NODE_DTYPE)
        nodes["tag"] = [abi.MOVE_TO] + [abi.LINE_TO] * (2 * n - 1) + [abi.CLOSE_PATH, abi.MOVE_TO]
        nodes["v"][:2 * n, 0] = w / 2 + r * np.cos(th)
        nodes["v"][:2 * n, 1] = h / 2 + r * np.sin(th)
        nodes["v"][-1] = nodes["v"][0]
        c = rng.integers(0, 256, 3)
        st.update(surf=surf, desc=surf.desc(), nodes=nodes, out=_tensor(surf),
                  pattern=abi.solid_pattern(abi.rgba(int(c[0]), int(c[1]), int(c[2]), 255)),
                  opts=abi.fill_opts(abi.AA_DEFAULT, abi.EVEN_ODD, "src_over"))
    elif k == "scene":
        surf, b, keep = _scene(ctx, rng, case["w"], case["h"], case["paths"], case["mix"])
        st.update(batch=b, keep=keep, out=_tensor(surf))
    elif k == "uneven":
        b = gpu.Batch(ctx)
        keep, items, surfs = [], [], []
        for fmt, side in _uneven(case["surfaces"], case["side"]):
            s = gpu.DeviceSurface(ctx, fmt, side, side)
            surfs.append(s)
            if fmt == abi.ALPHA8:  # a mask starts empty
                bg = (abi.solid_pattern(abi.pixel(abi.ALPHA8, a=0)), _rect(side, side),
                      abi.fill_opts(abi.AA_DEFAULT, abi.NON_ZERO, "clear"))
            else:
                bg = (abi.solid_pattern(abi.rgba(250, 250, 245, 255)), _rect(side, side),
                      abi.fill_opts(abi.AA_DEFAULT, abi.NON_ZERO, "src_over"))
            keep.append(bg)
            items.append((s, "fill") + bg)
            items += [(s,) + j for j in _jobs(rng, side, keep, fmt)]
        if any(b.draw_n(items)):
            raise RuntimeError("draw_n")
        b.prepare()
        parts = [_tensor(s) for s in surfs]
        st.update(batch=b, keep=(keep, items, surfs), parts=parts,
                  out=torch.empty(sum(t.numel() for t in parts), dtype=torch.uint8, device="cuda"))
    elif k == "serve":
        keep, preps, sizes = [], [], []
        for fmt, side in _uneven(case["requests"], case["side"]):
            clip = rng.integers(0, 256, side * side, dtype=np.uint8) if rng.random() < 0.5 else None
            preps.append(gpu.Server.prepare(fmt, side, side, [], clear=abi.pixel(fmt), clip=clip,
                                            draws=_jobs(rng, side, keep, fmt)))
            sizes.append(abi.surface_nbytes(fmt, side, side))
        n = len(preps)
        off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
        out = np.zeros(int(off[-1]), np.uint8)
        st.update(server=_server(), keep=(keep, preps), out=out, n=n,
                  reqs=np.array([C.addressof(p[0]) for p in preps], np.uint64),
                  outs=np.uint64(out.ctypes.data) + off[:-1], lens=np.array(sizes, np.uint64),
                  ids=np.zeros(n, np.uint64), status=np.zeros(n, np.int32),
                  done=np.zeros(n, np.uint64), done_status=np.zeros(n, np.int32),
                  t_done=np.zeros(n, np.float64))
    elif k == "text":
        w, h, size = case["w"], case["h"], case["size"]
        font = gpu.Font(open(FONT, "rb").read())
        surf = _surface(ctx, abi.RGBA, w, h)
        b = gpu.Batch(ctx)
        ctx.check(b.fill(surf, abi.solid_pattern(abi.rgba(255, 255, 255, 255)), _rect(w, h),
                         abi.fill_opts()), "fill")
        opts = abi.text_opts(size, fill=abi.fill_opts(abi.AA_DEFAULT))
        pat = abi.solid_pattern(abi.rgba(20, 20, 20, 255))
        chars = max(4, int(min(100, w / (0.55 * size))))
        for i in range(case["lines"]):
            line = ""
            while len(line) < chars:
                line += WORDS[int(rng.integers(0, len(WORDS)))] + " "
            ctx.check(b.text(surf, pat, font, line, 10.0, (i + 1.0) * 1.17 * size, opts), "text")
        b.prepare()
        st.update(batch=b, keep=(surf, font), out=_tensor(surf))
    elif k == "composite":
        w, h, x, y, fmt = case["w"], case["h"], case["x"], case["y"], case["fmt"]
        sw, sh = w - x, h - y
        dst = _surface(ctx, fmt, w, h, _premultiplied(seed, w, h))
        src = _surface(ctx, abi.RGBA, sw, sh, _premultiplied(seed + 1, sw, sh))
        out = _surface(ctx, fmt, w, h)
        keep = [dst, src, out]
        ds, dd, do = src.desc(), dst.desc(), out.desc()
        o = abi.CompOp()
        o.op = abi.OP[case["op"]]
        if case["masked"]:
            mask = _surface(ctx, abi.ALPHA8, w, h, rng.integers(0, 256, w * h, dtype=np.uint8))
            dm = mask.desc()
            m = abi.CompOp()
            m.op = abi.OP["dst_in"]
            m.dst.kind = m.src.kind = abi.PARAM_SURFACE
            m.dst.surface, m.src.surface = C.pointer(ds), C.pointer(dm)
            ops = (abi.CompOp * 2)(m, o)
            keep += [mask, dm]
        else:
            o.src.kind = abi.PARAM_SURFACE
            o.src.surface = C.pointer(ds)
            ops = (abi.CompOp * 1)(o)
        st.update(dst=dd, res=do, ops=ops, n_ops=len(ops), x=x, y=y, keep=(keep, ds),
                  out=_tensor(out))
    elif k == "paint":
        w, h = case["w"], case["h"]
        gtype = dict(linear=abi.GRADIENT_LINEAR, radial=abi.GRADIENT_RADIAL,
                     conic=abi.GRADIENT_CONIC)[case["grad"]]
        g = _gradient(rng, 0.0, 0.0, float(max(w, h)), gtype=gtype)
        surf = _surface(ctx, abi.RGBA, w, h)
        o = abi.CompOp()
        o.op = abi.OP["src"]
        if case["dither"]:
            o.src.kind = abi.PARAM_DITHER
            o.src.dither = abi.dither_pattern(abi.DITHER_BLUE_NOISE, 8, gradient=g).dither
        else:
            o.src.kind = abi.PARAM_GRADIENT
            o.src.gradient = C.pointer(g.desc)
        st.update(dst=surf.desc(), res=None, ops=(abi.CompOp * 1)(o), n_ops=1, x=0, y=0,
                  keep=(surf, g), out=_tensor(surf))
    else:
        surf, b, keep = _scene(ctx, rng, case["w"], case["h"], case["paths"], False, case["fmt"])
        b.render(0)
        b.wait()
        b.close()
        cap = gpu.png_bound(case["fmt"], case["w"], case["h"])
        buf = torch.zeros(cap, dtype=torch.uint8, pin_memory=True)
        st.update(surf=surf, desc=surf.desc(), file=buf, cap=cap, written=C.c_uint64())
    return st


# ---- one pass -------------------------------------------------------------------
def run(st):
    k, ctx = st["kind"], st["ctx"]
    if k in ("scene", "text", "uneven"):
        st["batch"].render(0)
        st["batch"].wait()
        if k == "uneven":  # the atlas: all surfaces in one buffer
            torch.cat(st["parts"], out=st["out"])
        return st["out"]
    if k == "fill":
        ctx.check(gpu.lib().z2d_gpu_fill(ctx.h, C.byref(st["desc"]), C.byref(st["pattern"]),
                                         st["nodes"].ctypes.data, len(st["nodes"]),
                                         C.byref(st["opts"])), "fill")
        return st["out"]
    if k in ("composite", "paint"):
        res = st["res"]
        ctx.check(gpu.lib().z2d_gpu_composite(ctx.h, C.byref(st["dst"]), st["x"], st["y"],
                                              st["ops"], st["n_ops"], abi.PRECISION_INTEGER,
                                              C.byref(res) if res is not None else None),
                  "composite")
        return st["out"]
    if k == "serve":
        srv, n = st["server"], st["n"]
        rc = srv.submit_n_raw(st["reqs"].ctypes.data, st["outs"].ctypes.data,
                              st["lens"].ctypes.data, n, st["ids"].ctypes.data,
                              st["status"].ctypes.data)
        if rc:
            raise RuntimeError("submit %d" % rc)
        got = 0
        while got < n:
            m = srv.wait_some(st["done"][got:], st["done_status"][got:], st["t_done"][got:], 20000.0)
            if m == 0:
                raise RuntimeError("the server did not answer")
            got += m
        if st["done_status"].any():
            raise RuntimeError("a request failed")
        return st["out"]
    ctx.check(gpu.lib().z2d_gpu_png_encode(ctx.h, C.byref(st["desc"]), abi.PNG_PROFILE_NONE,
                                           st["file"].data_ptr(), st["cap"],
                                           C.byref(st["written"])), "png_encode")
    return st["file"], st["written"].value  # the file, in a buffer that any file fits



# ---- what a pass cannot do without -------------------------------------------------
def _surface_bytes(fmt, w, h):
    return w * h * abi.FORMAT_BITS[fmt] // 8


def work(case):
    """Inputs read once, outputs written once."""
    k = case["kind"]
    if k == "fill":  # the surface is read and written under the shape
        n = 4 * case["w"] * case["h"]
        return dict(bytes=2 * n + 56 * 2 * case["points"], flops=0)
    # a path: 36.5 nodes of 56 bytes and its paint
    path = 36.5 * 56 + 100
    if k in ("scene", "png"):
        fmt = case.get("fmt", abi.RGBA)
        n = _surface_bytes(fmt, case["w"], case["h"])
        if k == "png":  # the surface read, the file (about half of it) written
            return dict(bytes=1.5 * n, flops=0)
        return dict(bytes=n + path * case["paths"], flops=0)
    if k in ("uneven", "serve"):
        # the mean square of a log-uniform side, 3.4 bytes a pixel; a stroke's
        # polygon in place of its path (some 1000 edges of 32 bytes)
        s = float(case["side"])
        mean = (s * s - 256.0) / (2.0 * math.log(s / 16.0)) * 3.4
        n = case["surfaces"] if k == "uneven" else case["requests"]
        per = mean + 25.5 * (0.7 * path + 0.3 * 32000)
        if k == "uneven":
            per += 2 * mean  # gathered
        else:
            per += 0.5 * mean / 3.4
        return dict(bytes=n * per, flops=0)
    if k == "text":  # some 26 nodes a glyph
        chars = max(4, int(min(100, case["w"] / (0.55 * case["size"]))))
        return dict(bytes=4 * case["w"] * case["h"] + case["lines"] * chars * 26 * 56, flops=0)
    if k == "paint":
        return dict(bytes=4 * case["w"] * case["h"], flops=0)
    px = (case["w"] - case["x"]) * (case["h"] - case["y"])
    per = (8 if case["op"] == "src" else 12) + (1 if case["masked"] else 0)
    return dict(bytes=per * px, flops=0)


def tolerance(case):
    return "exact"
