"""The work that is timed: calls of the framework's public entry points over
the range of figures, rasters and scenes they are used for.

Kinds of case and their entry points:

  plotter   ft.Plotter.fill / stroke, one call with host ops (and, with
            "read", the raster copied back to the host)
  glyphs    ft_batch_run_noalloc: many small tiles from host ops in one call,
            the entry for serving loops
  walk      Batch.launch of two large fills (NonZero and EvenOdd) whose ops
            are in device memory, pipelined over "depth" workspaces
  atlas     Batch.launch of many tiles of uneven size, replayed as a HIP graph
            or launched eagerly
  diff      DiffRenderer.step, DiffFill.apply + backward, or
            DiffRenderer.forward over images of filled cubic paths

Rasters hold whole numbers (bytes).  The differentiable fill's outputs are
float32; `exact` states its model in float64 torch.
"""
import ctypes
import math

import numpy as np
import torch

import footile_amd as ft
from footile_amd._lib import check, lib
from footile_amd.diff import DiffFill, DiffRenderer, device_array
from footile_amd.path import CLOSE, CUBIC, LINE, MOVE, OP_DTYPE, PEN_WIDTH, QUAD
from footile_amd.pixel import BPP, GRAYA8P, MATTE8, RGBA8P
from footile_amd.plotter import Batch, DeviceBuffer, FillDesc, FillDescC

FMT = {"matte8": MATTE8, "graya8p": GRAYA8P, "rgba8p": RGBA8P}
JOIN = {"miter": ft.JoinStyle.Miter(4.0), "bevel": ft.JoinStyle.Bevel, "round": ft.JoinStyle.Round}


def listed():
    return [
        # an icon: the smallest call, a few curves into 16x16, read back
        {"name": "icon_fill_16", "kind": "plotter", "call": "fill", "w": 16, "h": 16, "fmt": "matte8", "rule": 0,
         "law": "uniform", "lines": 4, "quads": 8, "cubics": 0, "read": True},
        # the plain 256x256 path: 48 lines and 16 cubics, filled
        {"name": "plain_fill_256", "kind": "plotter", "call": "fill", "w": 256, "h": 256, "fmt": "matte8", "rule": 0,
         "law": "uniform", "lines": 48, "quads": 0, "cubics": 16, "read": False},
        # the same path stroked at width 4
        {"name": "plain_stroke_256", "kind": "plotter", "call": "stroke", "w": 256, "h": 256, "fmt": "matte8",
         "rule": 0, "law": "uniform", "lines": 48, "quads": 0, "cubics": 16, "read": False, "width": 4.0,
         "join": "miter"},
        # a drawing of ragged size with more segments than a small figure holds, even-odd, gray
        {"name": "drawing_fill_gray", "kind": "plotter", "call": "fill", "w": 1237, "h": 771, "fmt": "graya8p",
         "rule": 1, "law": "walk", "lines": 300, "quads": 500, "cubics": 700, "read": False},
        # a long route stroked over an HD canvas with round joins
        {"name": "route_stroke_hd", "kind": "plotter", "call": "stroke", "w": 1920, "h": 1080, "fmt": "rgba8p",
         "rule": 0, "law": "route", "lines": 3000, "quads": 0, "cubics": 0, "read": False, "width": 3.0,
         "join": "round"},
        # a line of text: small tiles, ops and descriptors handed over per call
        {"name": "glyphs_384", "kind": "glyphs", "tiles": 384, "lo": 16, "hi": 64, "segs": 12, "fmt": "matte8"},
        # two fills of a 10,000-cubic random walk at 4096x4096, launches pipelined
        {"name": "walk_4096", "kind": "walk", "side": 4096, "cubics": 10000, "sigma": 40.0, "fmt": "rgba8p",
         "depth": 3},
        # 16,384 paths of lognormal length into 32..256 px tiles, one graph replay per launch
        {"name": "atlas_16384", "kind": "atlas", "paths": 16384, "mu": 3.5, "graph": True},
        # a differentiable render with its vector-Jacobian product, small and ragged
        {"name": "diff_vjp_small", "kind": "diff", "mode": "vjp", "images": 1, "w": 200, "h": 120, "paths_lo": 24,
         "paths_hi": 24, "cubics_lo": 1, "cubics_hi": 6, "keep": False},
        # a render alone: one wide image, several blocks across
        {"name": "diff_forward_wide", "kind": "diff", "mode": "forward", "images": 1, "w": 1000, "h": 600,
         "paths_lo": 128, "paths_hi": 128, "cubics_lo": 4, "cubics_hi": 12, "keep": False},
        # one optimisation step of one 512x512 image, 256 paths of 8 cubics
        {"name": "diff_step_512", "kind": "diff", "mode": "step", "images": 1, "w": 512, "h": 512, "paths_lo": 256,
         "paths_hi": 256, "cubics_lo": 8, "cubics_hi": 8, "keep": False},
        # one optimisation step of 64 images in one call
        {"name": "diff_step_64x256", "kind": "diff", "mode": "step", "images": 64, "w": 256, "h": 256, "paths_lo": 32,
         "paths_hi": 512, "cubics_lo": 4, "cubics_hi": 16, "keep": False},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["plotter", "plotter", "plotter", "glyphs", "walk", "atlas", "diff", "diff", "diff"])
    if kind == "plotter":
        call = rng.choice(["fill", "stroke"])
        small = rng.random() < 0.5
        segs = _log(rng, 6, 120) if small else _log(rng, 300, 8000 if call == "fill" else 3000)
        a, b = sorted((rng.random(), rng.random()))
        lines, quads = int(segs * a), int(segs * (b - a))
        w, h = (_log(rng, 12, 700), _log(rng, 12, 700)) if small else (_log(rng, 300, 4096), _log(rng, 300, 4096))
        c = {"kind": "plotter", "call": call, "w": w, "h": h, "fmt": rng.choice(sorted(FMT)),
             "rule": rng.randint(0, 1), "law": "uniform" if small else "walk", "lines": lines, "quads": quads,
             "cubics": segs - lines - quads, "read": small and rng.random() < 0.3}
        if call == "stroke":
            c["rule"] = 0
            c["width"] = round(rng.uniform(0.75, 9.0), 2)
            # round joins go with routes: at a turn straight on or back they have no arc (FT_ERANGE)
            c["join"] = rng.choice(sorted(JOIN))
            if c["join"] == "round":
                c.update(law="route", lines=segs, quads=0, cubics=0)
        return c
    if kind == "glyphs":
        lo = _log(rng, 8, 48)
        return {"kind": "glyphs", "tiles": _log(rng, 8, 900), "lo": lo, "hi": lo + rng.randint(0, 48),
                "segs": rng.randint(6, 24), "fmt": rng.choice(["matte8", "matte8", "rgba8p"])}
    if kind == "walk":
        side = _log(rng, 500, 4096)
        return {"kind": "walk", "side": side, "cubics": _log(rng, 500, 10000), "sigma": round(side / 102.4, 2),
                "fmt": rng.choice(["rgba8p", "rgba8p", "graya8p"]), "depth": rng.randint(1, 3)}
    if kind == "atlas":
        return {"kind": "atlas", "paths": _log(rng, 200, 14000), "mu": round(rng.uniform(2.5, 3.5), 2),
                "graph": rng.random() < 0.5}
    images = _log(rng, 1, 48)
    w, h = _log(rng, 48, 700), _log(rng, 48, 700)
    most = max(8, min(400, int(4.0e8 / (images * w * h))))
    hi = _log(rng, 8, most)
    lo_c = rng.randint(1, 8)
    return {"kind": "diff", "mode": rng.choice(["step", "step", "vjp", "forward"]), "images": images, "w": w, "h": h,
            "paths_lo": max(1, hi // rng.randint(1, 4)), "paths_hi": hi, "cubics_lo": lo_c,
            "cubics_hi": lo_c + rng.randint(0, 8), "keep": rng.random() < 0.25}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
class _DeviceView:
    """Device memory as torch sees it.  The tensor keeps this object, and with
    it the memory's owner (a DeviceBuffer or a Plotter), alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (int(ptr), False),
                                         "version": 2}


def _view(owner, shape, typestr="|u1", ptr=None):
    return torch.as_tensor(_DeviceView(owner, owner.ptr if ptr is None else ptr, shape, typestr), device="cuda")


def _walk(g, n, hi, sigma, start):
    """n points of a random walk reflected into [0, hi] per axis."""
    hi = np.asarray(hi, np.float64)
    p = np.asarray(start) + np.cumsum(g.normal(0.0, sigma, (n, 2)), axis=0)
    p = np.mod(p, 2.0 * hi)
    return np.where(p > hi, 2.0 * hi - p, p)


def _route(g, n, hi, step):
    """n points of a simplified route: every turn between 0.2 and 1.2 rad,
    towards the middle of [0, hi] near its border."""
    turns, steps = g.uniform(0.2, 1.2, n) * np.where(g.random(n) < 0.5, -1.0, 1.0), step * g.uniform(0.5, 1.5, n)
    w, h = hi
    x, y, a = w / 2.0, h / 2.0, float(g.uniform(0.0, 2.0 * math.pi))
    out = []
    for turn, d in zip(turns.tolist(), steps.tolist()):
        if not (0.1 * w < x < 0.9 * w and 0.1 * h < y < 0.9 * h):
            away = math.atan2(h / 2.0 - y, w / 2.0 - x) - a
            turn = math.copysign(max(abs(turn), 0.7), math.sin(away))
        a += turn
        x, y = min(max(x + d * math.cos(a), 0.0), w), min(max(y + d * math.sin(a), 0.0), h)
        out.append((x, y))
    return np.array(out)


def _path_ops(g, kinds, w, h, law):
    """move, the segments `kinds` in order, close."""
    per = np.where(kinds == CUBIC, 3, np.where(kinds == QUAD, 2, 1))
    n = int(per.sum()) + 1
    if law == "uniform":  # margin of 1/32, as a figure drawn for its raster
        m = np.array([w, h]) / 32.0
        pts = m + g.random((n, 2)) * (np.array([w, h]) - 2.0 * m)
    else:
        hi = (w - 0.01, h - 0.01)
        if law == "route":
            pts = _route(g, n, hi, min(w, h) / 70.0)
        else:
            pts = _walk(g, n, hi, max(w, h) / 100.0, (w / 2.0, h / 2.0))
    pts = pts.astype(np.float32)
    ops = np.zeros(len(kinds) + 2, OP_DTYPE)
    ops["tag"][0], ops["tag"][-1] = MOVE, CLOSE
    ops["tag"][1:-1] = kinds
    ops["v"][0, :2] = pts[0]
    first = 1 + np.concatenate([[0], np.cumsum(per)[:-1]])
    for k in range(3):
        has = per > k
        ops["v"][1:-1][has, 2 * k:2 * k + 2] = pts[first[has] + k]
    return ops


def _plotter_ops(case, g):
    kinds = np.array([LINE] * case["lines"] + [QUAD] * case["quads"] + [CUBIC] * case["cubics"])
    ops = _path_ops(g, g.permutation(kinds), case["w"], case["h"], case["law"])
    if case["call"] == "stroke":
        pen = np.zeros(1, OP_DTYPE)
        pen["tag"], pen["v"][0, 0] = PEN_WIDTH, case["width"]
        ops = np.concatenate([pen, ops])
    return ops


def _colour(g, fmt, opaque):
    a = 255 if opaque else int(g.integers(96, 255))
    if fmt == MATTE8:
        return (255,)
    if fmt == GRAYA8P:
        return (int(g.integers(0, a + 1)), a)
    return tuple(int(g.integers(0, a + 1)) for _ in range(3)) + (a,)


def _pack(sides, width, height):
    """Shelf packing, tallest first: x and y of each tile."""
    order = np.argsort(-sides, kind="stable")
    xs, ys = np.zeros(len(sides), np.int64), np.zeros(len(sides), np.int64)
    x = y = shelf = 0
    for t in order:
        s = int(sides[t])
        if x + s > width:
            x, y, shelf = 0, y + shelf, 0
        xs[t], ys[t] = x, y
        x += s
        shelf = max(shelf, s)
    if y + shelf > height:
        raise ValueError("the tiles do not fit")
    return xs, ys


def _tile_ops(g, seg_counts, cum_kinds, sides, closes_every=None):
    """Closed paths of random segments, each uniform in its own tile; with
    closes_every, a path is several outlines of that many segments.  Returns
    the ops and each path's (begin, count)."""
    n_seg = np.asarray(seg_counts, np.int64)
    subs = np.ones_like(n_seg) if closes_every is None else -(-n_seg // closes_every)
    counts = n_seg + 2 * subs
    begins = np.concatenate([[0], np.cumsum(counts)[:-1]])
    total = int(counts.sum())
    path = np.repeat(np.arange(len(n_seg)), counts)
    local = np.arange(total) - begins[path]
    per = n_seg[path] + 2 if closes_every is None else np.full(total, closes_every + 2)
    pos = local % per
    last = (pos == per - 1) | (local == counts[path] - 1)
    u = g.random(total)
    tag = np.where(u < cum_kinds[0], CUBIC, np.where(u < cum_kinds[1], QUAD, LINE))
    tag = np.where(pos == 0, MOVE, np.where(last, CLOSE, tag))
    n_val = np.array([0, 2, 2, 4, 6, 0])[tag]
    s = np.asarray(sides, np.float64)[path][:, None]
    v = 1.0 + g.random((total, 6)) * (s - 2.0)
    v[np.arange(6)[None, :] >= n_val[:, None]] = 0.0
    ops = np.zeros(total, OP_DTYPE)
    ops["tag"], ops["v"] = tag, v.astype(np.float32)
    return ops, begins, counts


def _glyph_inputs(case, g):
    n = case["tiles"]
    sides = g.integers(case["lo"], case["hi"] + 1, n)
    segs = np.maximum(4, g.integers(case["segs"] // 2, case["segs"] * 3 // 2 + 1, n))
    ops, begins, counts = _tile_ops(g, segs, (0.1, 0.65), sides, closes_every=max(4, case["segs"] // 2))
    height = 2 * case["hi"] + int(1.5 * n * case["hi"] ** 2 / 1024)
    xs, ys = _pack(sides, 1024, height)
    return ops, begins, counts, sides, xs, ys, height


def _atlas_inputs(case, g):
    n = case["paths"]
    segs = np.clip(np.rint(np.exp(case["mu"] + g.normal(size=n))), 4, 2000).astype(np.int64)
    sides = np.clip(np.ceil(12.0 * np.sqrt(segs) / 8.0).astype(np.int64) * 8, 32, 256)
    ops, begins, counts = _tile_ops(g, segs, (0.6, 0.9), sides)
    side = 16384 if n > 1200 else 4096
    xs, ys = _pack(sides, side, side)
    return ops, begins, counts, sides, xs, ys, side


def _walk_ops(case, g):
    side = case["side"]
    pts = _walk(g, 3 * case["cubics"], (side - 0.01, side - 0.01), case["sigma"], (side / 2.0, side / 2.0))
    ops = np.zeros(case["cubics"] + 2, OP_DTYPE)
    ops["tag"][0], ops["tag"][-1], ops["tag"][1:-1] = MOVE, CLOSE, CUBIC
    ops["v"][0, :2] = side / 2.0
    ops["v"][1:-1] = pts.reshape(-1, 6).astype(np.float32)
    return ops


def _diff_layout(case):
    """The scene's layout: a program's plan, the same for every seed."""
    g = np.random.default_rng(17)
    n = g.integers(case["paths_lo"], case["paths_hi"] + 1, case["images"])
    image = np.repeat(np.arange(case["images"], dtype=np.uint32), n)
    cubics = g.integers(case["cubics_lo"], case["cubics_hi"] + 1, len(image)).astype(np.uint32)
    return image, cubics


def _diff_inputs(case, seed):
    """Control points uniform over the canvas, premultiplied colours, and a
    smooth target (or, for a VJP, a cotangent) with noise."""
    image, cubics = _diff_layout(case)
    g = np.random.default_rng(seed)
    w, h = case["w"], case["h"]
    n_pts = int(np.sum(1 + 3 * cubics.astype(np.int64)))
    points = (g.random((n_pts, 2)) * (w, h)).astype(np.float32)
    a = g.uniform(0.3, 0.9, (len(image), 1))
    colours = np.concatenate([a * g.random((len(image), 3)), a], axis=1).astype(np.float32)
    if case["mode"] == "vjp":
        pixels = g.normal(size=(case["images"], h, w, 4)).astype(np.float32)
    else:
        y, x = np.mgrid[0:h, 0:w].astype(np.float32)
        f = g.uniform(1.0, 9.0, (case["images"], 4, 2)).astype(np.float32)
        pixels = np.stack([np.stack([0.5 + 0.4 * np.sin(f[i, c, 0] * x / w + f[i, c, 1] * y / h)
                                     for c in range(4)], -1) for i in range(case["images"])])
        pixels = (pixels + g.normal(0.0, 0.02, pixels.shape)).astype(np.float32)
    return image, cubics, points, colours, pixels


# ---------------------------------------------------------------------------
# What a program holds before the call, and the call
# ---------------------------------------------------------------------------
def prepare(case, seed):
    g = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "plotter":
        fmt = FMT[case["fmt"]]
        p = ft.Plotter(ft.Raster.with_clear(case["w"], case["h"], fmt))
        if case["call"] == "stroke":
            p.set_join(JOIN[case["join"]])
        ops = _plotter_ops(case, g)
        ptr, pitch = p.device_ptr()
        return {"kind": kind, "p": p, "ops": ops, "clr": _colour(g, fmt, opaque=seed % 2 == 0), "rule": case["rule"],
                "stroke": case["call"] == "stroke", "read": case["read"], "out": _view(p, (case["h"], pitch), ptr=ptr)}
    if kind == "glyphs":
        fmt = FMT[case["fmt"]]
        ops, begins, counts, sides, xs, ys, height = _glyph_inputs(case, g)
        bpp = BPP[fmt]
        pitch = 1024 * bpp
        dst = DeviceBuffer(pitch * height)
        dst.zero()
        clr = _colour(g, fmt, opaque=True)
        descs = [FillDesc(int(b), int(c), dst.ptr + int(y) * pitch + int(x) * bpp, int(s), int(s), pitch, fmt,
                          clr=clr, fresh=True) for b, c, x, y, s in zip(begins, counts, xs, ys, sides)]
        n = len(descs)
        return {"kind": kind, "ops": ops, "descs": (FillDescC * n)(*[d.c for d in descs]), "n": n, "dst": dst,
                "offered": np.zeros(n, np.uint64), "stored": np.zeros(n, np.uint64),
                "out": _view(dst, (height, pitch))}
    if kind == "walk":
        fmt = FMT[case["fmt"]]
        side, bpp = case["side"], BPP[fmt]
        ops = _walk_ops(case, g)
        clr = (200, 120, 40, 255) if fmt == RGBA8P else (140, 255)
        bufs = [DeviceBuffer(side * side * bpp) for _ in range(2)]
        descs = [FillDesc(k * len(ops), len(ops), bufs[k].ptr, side, side, side * bpp, fmt, rule=k, clr=clr)
                 for k in range(2)]
        batch = Batch(np.concatenate([ops, ops]), descs)
        batch.run()  # sizes the workspace
        batch.set_pipeline(case["depth"])
        for b in bufs:
            b.zero()
        return {"kind": kind, "batch": batch, "bufs": bufs,
                "out": [_view(b, (side, side * bpp)) for b in bufs]}
    if kind == "atlas":
        ops, begins, counts, sides, xs, ys, side = _atlas_inputs(case, g)
        dst = DeviceBuffer(side * side)
        dst.zero()
        descs = [FillDesc(int(b), int(c), dst.ptr + int(y) * side + int(x), int(s), int(s), side, fresh=True)
                 for b, c, x, y, s in zip(begins, counts, xs, ys, sides)]
        batch = Batch(ops, descs)
        batch.run()  # sizes the workspace
        if case["graph"]:
            batch.set_graph(True)
        return {"kind": kind, "batch": batch, "bufs": [dst], "out": [_view(dst, (side, side))]}
    image, cubics, points, colours, pixels = _diff_inputs(case, seed)
    r = DiffRenderer(case["images"], case["w"], case["h"], image, cubics, keep_coverage=case["keep"])
    s = {"kind": kind, "mode": case["mode"], "r": r, "points": device_array(points),
         "colours": device_array(colours), "pixels": device_array(pixels), "canvas": r.new_canvas(),
         "gcan": r.new_canvas(), "gp": DeviceBuffer(8 * r.n_points), "gc": DeviceBuffer(16 * r.n_paths)}
    s["out"] = {"canvas": _view(s["canvas"], r.canvas_shape, "<f4"),
                "grad_points": _view(s["gp"], (r.n_points, 2), "<f4"),
                "grad_colours": _view(s["gc"], (r.n_paths, 4), "<f4")}
    return s


def run(state):
    kind = state["kind"]
    if kind == "plotter":
        p = state["p"]
        if state["stroke"]:
            p.stroke(state["ops"], state["clr"])
        else:
            p.fill(state["rule"], state["ops"], state["clr"])
        return p.raster().pixels if state["read"] else state["out"]
    if kind == "glyphs":
        ops = state["ops"]
        check(lib().ft_batch_run_noalloc(ops.ctypes.data_as(ctypes.c_void_p), len(ops), state["descs"], state["n"],
                                         None, state["offered"].ctypes.data_as(ctypes.c_void_p),
                                         state["stored"].ctypes.data_as(ctypes.c_void_p)), "ft_batch_run_noalloc")
        return {"tiles": state["out"], "offered": state["offered"].view(np.int64),
                "stored": state["stored"].view(np.int64)}
    if kind in ("walk", "atlas"):
        state["batch"].launch()
        return state["out"]
    r, out = state["r"], state["out"]
    if state["mode"] == "step":
        loss = r.step(state["points"], state["colours"], state["pixels"], state["canvas"], state["gcan"], state["gp"],
                      state["gc"])
        return dict(out, loss=loss)
    if state["mode"] == "forward":
        r.forward(state["points"], state["colours"], state["canvas"])
        return {"canvas": out["canvas"]}
    canvas, ctx = DiffFill.apply(r, state["points"], state["colours"])
    _, gp, gc = DiffFill.backward(ctx, state["pixels"])
    state["last"] = (canvas, gp, gc)
    return {"canvas": _view(canvas, r.canvas_shape, "<f4"), "grad_points": _view(gp, (r.n_points, 2), "<f4"),
            "grad_colours": _view(gc, (r.n_paths, 4), "<f4")}


# ---------------------------------------------------------------------------
# Work and the float64 model
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: the raster written (and, where the fill blends, read) and the
    ops' points.  Flops of the differentiable fill: the composite of every
    path over every pixel and, with gradients, its adjoint."""
    kind = case["kind"]
    if kind == "plotter":
        bpp = BPP[FMT[case["fmt"]]]
        px = case["w"] * case["h"] * bpp * (1 if bpp == 1 else 2)
        return {"bytes": px + 8 * (case["lines"] + 2 * case["quads"] + 3 * case["cubics"] + 1), "flops": 0}
    if kind == "glyphs":
        side2 = ((case["lo"] + case["hi"]) / 2.0) ** 2
        return {"bytes": case["tiles"] * (side2 * BPP[FMT[case["fmt"]]] + 8 * 1.8 * case["segs"]), "flops": 0}
    if kind == "walk":
        return {"bytes": 2 * (case["side"] ** 2 * 2 * BPP[FMT[case["fmt"]]] + 24 * case["cubics"]), "flops": 0}
    if kind == "atlas":
        mean = math.exp(case["mu"] + 0.5)
        return {"bytes": case["paths"] * (144.0 * mean + 8 * 2.5 * mean), "flops": 0}
    image, _ = _diff_layout(case)
    px = case["w"] * case["h"]
    canvases = {"forward": 1, "vjp": 2, "step": 3}[case["mode"]]
    per = {"forward": 12, "vjp": 42, "step": 42}[case["mode"]]
    return {"bytes": 16 * px * case["images"] * canvases, "flops": per * px * len(image)}


def _pieces(P, q, path, H):
    """Edge pieces per row: edges p -> q of `path`, split over the rows they
    overlap.  P, q: [E, 2].  Returns x at top and bottom, signed height, the
    row and the path of each piece."""
    down = q[:, 1] > P[:, 1]
    t, b = torch.where(down[:, None], P, q), torch.where(down[:, None], q, P)
    with torch.no_grad():
        lo, hi = t[:, 1].clamp(0, H), b[:, 1].clamp(0, H)
        r0 = lo.floor().long()
        n = torch.where((b[:, 1] > t[:, 1]) & (hi > lo), hi.ceil().long() - r0, torch.zeros_like(r0))
        e = torch.repeat_interleave(torch.arange(len(n), device=n.device), n)
        Y = r0[e] + torch.arange(len(e), device=n.device) - (torch.cumsum(n, 0) - n)[e]
    tx, ty, bx, by = t[e, 0], t[e, 1], b[e, 0], b[e, 1]
    Yf = Y.to(P.dtype)
    ya, yb = torch.maximum(ty, Yf), torch.minimum(by, Yf + 1.0)
    sl = (bx - tx) / (by - ty)
    sign = torch.where(down[e], 1.0, -1.0).to(P.dtype)
    return tx + (ya - ty) * sl, tx + (yb - ty) * sl, sign * (yb - ya), Y, path[e]


def _coverage(pts, first, cubics, k0, k1, H, W):
    """Signed coverage [k1 - k0, H, W] of the paths k0..k1 from their control
    points."""
    dev, P, Q, owner = pts.device, [], [], []
    t = torch.arange(1, 17, dtype=pts.dtype, device=dev)[:, None] / 16.0
    wts = torch.cat([(1 - t) ** 3, 3 * (1 - t) ** 2 * t, 3 * (1 - t) * t ** 2, t ** 3], 1)
    ids = torch.arange(k0, k1, device=dev)
    n = torch.as_tensor(cubics[k0:k1].astype(np.int64), device=dev)
    c_path = torch.repeat_interleave(ids - k0, n)
    c_local = torch.arange(len(c_path), device=dev) - (torch.cumsum(n, 0) - n)[c_path]
    base = torch.as_tensor(first[k0:k1], device=dev)[c_path] + 3 * c_local
    ctrl = pts[base[:, None] + torch.arange(4, device=dev)]           # [C, 4, 2]
    v = torch.einsum("jk,ckd->cjd", wts, ctrl)                        # [C, 16, 2]
    prev = torch.cat([ctrl[:, :1], v[:, :-1]], 1)
    # a cubic's first vertex is the previous cubic's last (the path's start for the first)
    follows = (c_local > 0).nonzero()[:, 0]
    prev = prev.index_put((follows, torch.zeros_like(follows)), v[follows - 1, -1])
    last = torch.cumsum(n, 0) - 1
    start = pts[torch.as_tensor(first[k0:k1], device=dev)]
    P = torch.cat([prev.reshape(-1, 2), v[last, -1]])
    Q = torch.cat([v.reshape(-1, 2), start])
    owner = torch.cat([torch.repeat_interleave(c_path, 16), ids - k0])
    xa, xb, z, Y, path = _pieces(P, Q, owner, H)
    X = torch.arange(W, dtype=pts.dtype, device=dev)
    ua, ub = X[None, :] + 1.0 - xa[:, None], X[None, :] + 1.0 - xb[:, None]
    lo, hi = torch.minimum(ua, ub), torch.maximum(ua, ub)
    narrow = hi - lo < 1e-5
    wd = torch.where(narrow, torch.ones_like(lo), hi - lo)
    a, b = lo.clamp(0.0, 1.0), hi.clamp(0.0, 1.0)
    m = ((b - a) * (a + b) * 0.5 + (hi - 1.0).clamp(min=0.0)) / wd
    m = torch.where(narrow, ((lo + hi) * 0.5).clamp(0.0, 1.0), m)
    m = torch.where(hi <= 0.0, torch.zeros_like(m), torch.where(lo >= 1.0, torch.ones_like(m), m))
    A = torch.zeros((k1 - k0) * H, W, dtype=pts.dtype, device=dev)
    return A.index_add(0, path * H + Y, z[:, None] * m).reshape(k1 - k0, H, W)


def _composite(A, col):
    al = A.abs().clamp(max=1.0)[..., None]
    C = torch.zeros(A.shape[1], A.shape[2], 4, dtype=A.dtype, device=A.device)
    for k in range(len(A)):
        C = col[k] * al[k] + C * (1.0 - col[k, 3] * al[k])
    return C


def exact(case, seed):
    """The differentiable fill's outputs in float64 torch; rasters are bytes
    and have no such value."""
    if case["kind"] != "diff":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    image, cubics, points, colours, pixels = _diff_inputs(case, seed)
    first = np.concatenate([[0], np.cumsum(1 + 3 * cubics.astype(np.int64))])
    pts = torch.as_tensor(points, dtype=torch.float64, device=dev)
    col = torch.as_tensor(colours, dtype=torch.float64, device=dev)
    pix = torch.as_tensor(pixels, dtype=torch.float64, device=dev)
    H, W = case["h"], case["w"]
    grads = case["mode"] != "forward"
    canvas = torch.zeros_like(pix)
    gp, gc = torch.zeros_like(pts), torch.zeros_like(col)
    n_all = pix.numel()
    loss = 0.0
    for i in range(case["images"]):
        ks = np.nonzero(image == i)[0]
        if not len(ks):
            if case["mode"] == "step":
                loss += float(((canvas[i] - pix[i]) ** 2).sum()) / n_all
            continue
        k0, k1 = int(ks[0]), int(ks[-1]) + 1
        # paths in runs whose [pieces, W] arrays stay small
        cost = np.cumsum(cubics[k0:k1].astype(np.int64) * (0.6 * H + 20) * W)
        run_of = (cost // 60_000_000).astype(np.int64)
        cuts = [k0] + [k0 + int(j) for j in np.nonzero(np.diff(run_of))[0] + 1] + [k1]
        with torch.no_grad():
            A = torch.cat([_coverage(pts, first, cubics, a, b, H, W) for a, b in zip(cuts, cuts[1:])])
        if not grads:
            with torch.no_grad():
                canvas[i] = _composite(A, col[k0:k1])
            continue
        A.requires_grad_(True)
        c = col[k0:k1].clone().requires_grad_(True)
        C = _composite(A, c)
        canvas[i] = C.detach()
        if case["mode"] == "step":
            part = ((C - pix[i]) ** 2).sum() / n_all
            loss += float(part.detach())
        else:
            part = (C * pix[i]).sum()
        part.backward()
        gc[k0:k1] = c.grad
        dA = A.grad
        del C, part, A
        for a, b in zip(cuts, cuts[1:]):
            p = pts[int(first[a]):int(first[b])].clone().requires_grad_(True)
            _coverage(p, first[a:b + 1] - first[a], cubics[a:b], 0, b - a, H, W).backward(dA[a - k0:b - k0])
            gp[int(first[a]):int(first[b])] = p.grad
    out = {"canvas": canvas}
    if grads:
        out.update(grad_points=gp, grad_colours=gc)
    if case["mode"] == "step":
        out["loss"] = torch.tensor(loss, dtype=torch.float64)
    return out
