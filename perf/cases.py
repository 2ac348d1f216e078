"""What is timed of this framework: the work its users have it do, through its public
entry points (resvg_amd.Context and resvg_amd.diff.Renderer).

Kinds of case, and what each stands for:

* ``document``: Context.render of a whole document onto a device pixmap (resvg::render),
  the framework's main path.  The full-filter scene at 4096 x 4096 is the headline; the
  plain documents (5-200 paths, a 1-6 primitive filter) are ordinary pages; the
  blur -> offset -> composite document is the smallest filtered one.
* ``clipmask``: Context.render of a document whose groups are clipped and masked.
* ``host``: Context.render_host, the resvg_render twin a C caller uses: an icon drawn
  into host memory, where latency and the number of launches count.
* ``batch``: Context.render_batch of many documents of uneven sizes (thumbnailing).
* ``filter``: Context.filter_apply of a filter graph on a layer: blurs of the IIR and the
  box branch, morphology, chains of the other primitives.
* ``png``: Context.png_filter_rows, the device's part of PNG output.
* ``planes`` / ``analytic``: one training step's forward and backward of the
  differentiable f32 form: paint, blur and colour matrix over fixed coverage, and the
  batched form with geometry (image fitting).

Rendered and filtered pixels are bytes and stay the same bytes.  Only the differentiable
form returns floating results; ``exact`` restates it in float64.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import resvg_amd
from resvg_amd import abi, diff, workloads
from resvg_amd.filters import SOURCE_ALPHA, SOURCE_GRAPHIC, FilterGraph, distant_light, point_light, spot_light

SPACES = {"linear": abi.CI_LINEAR_RGB, "srgb": abi.CI_SRGB}
_CTX = None


def _ctx():
    """The process's one context, as a program that renders keeps it."""
    global _CTX
    if _CTX is None:
        _CTX = resvg_amd.Context(0)
    return _CTX


# --- the cases -------------------------------------------------------------------
def listed():
    return [
        # the headline scene: 2000 gradient paths in opacity groups, 8 filter regions
        {"name": "full_filter_4096", "kind": "document", "doc": "full_filter", "w": 4096, "h": 4096, "paths": 2000,
         "prims": 0},
        # an ordinary page: tens of paths and a filter chain, odd sides
        {"name": "page_1201x843", "kind": "document", "doc": "plain", "w": 1201, "h": 843, "paths": 64, "prims": 3},
        # one filtered path, the smallest document with a filter
        {"name": "blur_path_512", "kind": "document", "doc": "blur_path", "w": 512, "h": 512, "paths": 1, "prims": 3},
        # clip paths and masks, each rendered for every group that uses it
        {"name": "clip_mask_2048", "kind": "clipmask", "w": 2048, "h": 2048, "groups": 150},
        # an icon into host memory (the C entry point): the smallest call
        {"name": "icon_host_61x47", "kind": "host", "w": 61, "h": 47, "paths": 6, "prims": 1},
        # thumbnails: documents with sides 64-2048 in one call
        {"name": "batch_64", "kind": "batch", "docs": 64, "max_side": 2048},
        # every other filter primitive and a blur of the IIR branch in one graph, on an odd-sized layer
        {"name": "chain_1601x1131", "kind": "filter", "w": 1601, "h": 1131, "space": "linear", "sx": 1.5, "sy": 1.5,
         "prims": "blur,turbulence,displacement,lighting,convolve,transfer,matrix,arithmetic,shadow,tile,blend"},
        # a large feGaussianBlur (box branch), colour conversions included
        {"name": "blur_4096_s6", "kind": "filter", "w": 4096, "h": 4096, "space": "linear", "prims": "blur",
         "sx": 6.0, "sy": 6.0},
        # morphology, ragged sides, both directions of the range of radii
        {"name": "dilate_2051x1537", "kind": "filter", "w": 2051, "h": 1537, "space": "srgb", "prims": "dilate",
         "sx": 5.0, "sy": 2.0},
        # PNG rows of a finished page
        {"name": "png_3001x2003", "kind": "png", "w": 3001, "h": 2003},
        # one fitting step of one large picture with fixed outlines
        {"name": "planes_1024", "kind": "planes", "w": 1024, "h": 1024, "paths": 256, "segments": 8, "sigma": 4.0},
        # one step of many small fits at once, outlines fitted too
        {"name": "analytic_16x512", "kind": "analytic", "batch": 16, "w": 512, "h": 512, "paths": 128,
         "segments": 8, "sigma": 2.5},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["document", "document", "clipmask", "host", "batch", "filter", "filter", "filter", "png",
                       "planes", "analytic"])
    if kind == "document":
        doc = rng.choice(["full_filter", "plain", "plain", "blur_path"])
        if doc == "full_filter":
            s = _log(rng, 128, 4096)
            return {"kind": kind, "doc": doc, "w": s, "h": s, "paths": _log(rng, 20, 2000), "prims": 0}
        if doc == "blur_path":
            s = _log(rng, 64, 2048)
            return {"kind": kind, "doc": doc, "w": s, "h": s, "paths": 1, "prims": 3}
        return {"kind": kind, "doc": doc, "w": _log(rng, 64, 2048), "h": _log(rng, 64, 2048),
                "paths": rng.randint(5, 200), "prims": rng.randint(1, 6)}
    if kind == "clipmask":
        s = _log(rng, 128, 2048)
        return {"kind": kind, "w": s, "h": s, "groups": _log(rng, 8, 150)}
    if kind == "host":
        return {"kind": kind, "w": _log(rng, 16, 512), "h": _log(rng, 16, 512), "paths": rng.randint(1, 40),
                "prims": rng.randint(1, 3)}
    if kind == "batch":
        return {"kind": kind, "docs": _log(rng, 4, 64), "max_side": _log(rng, 128, 2048)}
    if kind == "filter":
        case = {"kind": kind, "w": _log(rng, 24, 4096), "h": _log(rng, 24, 4096),
                "space": rng.choice(["linear", "srgb"])}
        if rng.random() < 0.4:
            names = ["blur", "turbulence", "displacement", "lighting", "convolve", "transfer", "matrix", "arithmetic",
                     "shadow", "tile", "blend"]
            rng.shuffle(names)
            s = round(math.exp(rng.uniform(math.log(0.5), math.log(24.0))), 3)
            case.update(w=min(case["w"], 2048), h=min(case["h"], 2048), prims=",".join(names[:rng.randint(1, 6)]),
                        sx=s, sy=s)
        else:
            prim = rng.choice(["blur", "blur", "dilate", "erode"])
            hi = 24.0 if prim == "blur" else 8.0
            r = [round(math.exp(rng.uniform(math.log(0.5), math.log(hi))), 3) for _ in range(2)]
            if rng.random() < 0.4:
                r[1] = r[0]
            case.update(prims=prim, sx=r[0], sy=r[1])
        return case
    if kind == "png":
        return {"kind": kind, "w": _log(rng, 16, 4096), "h": _log(rng, 16, 4096)}
    if kind == "planes":
        return {"kind": kind, "w": _log(rng, 100, 1024), "h": _log(rng, 100, 1024), "paths": _log(rng, 5, 256),
                "segments": rng.randint(3, 8), "sigma": round(rng.uniform(0.5, 12.0), 3)}
    return {"kind": kind, "batch": rng.randint(1, 16), "w": _log(rng, 100, 512), "h": _log(rng, 100, 512),
            "paths": _log(rng, 5, 128), "segments": rng.randint(3, 8), "sigma": round(rng.uniform(0.5, 4.0), 3)}


# --- inputs ----------------------------------------------------------------------
def _document(case, seed):
    if case["kind"] == "clipmask":
        return workloads.clip_mask_doc(seed=seed, size=case["w"], n_groups=case["groups"])[0]
    doc = case.get("doc", "plain")
    if doc == "full_filter":
        return workloads.full_filter_doc(seed=seed, size=case["w"], n_paths=case["paths"])[0]
    if doc == "blur_path":
        return workloads.blur_offset_composite_doc(seed=seed, size=case["w"])[0]
    return workloads.batch_doc(seed, case["w"], case["h"], case["paths"], case["prims"])


def _batch_specs(case):
    """(width, height, paths, filter primitives) of a batch's documents: the same shapes for
    every seed, other contents."""
    return [sp[1:] for sp in workloads.document_specs(case["docs"], seed=case["docs"], max_side=case["max_side"])]


def _layer(w, h, seed):
    """A premultiplied RGBA8 layer as a group of drawn shapes leaves it: about a third
    transparent, a third opaque, soft edges between, colours that vary slowly with a
    little noise on them."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    low = torch.rand((1, 4, h // 48 + 3, w // 48 + 3), generator=gen, device="cuda")
    up = torch.nn.functional.interpolate(low, size=(h, w), mode="bicubic", align_corners=False)[0]
    noise = torch.rand((3, h, w), generator=gen, device="cuda") * 0.04
    a = ((up[3] - 0.42) * 8.0).clamp(0.0, 1.0)
    rgb = (up[:3] + noise).clamp(0.0, 1.0) * a
    return (torch.cat([rgb, a[None]]) * 255.0).floor().to(torch.uint8).permute(1, 2, 0).contiguous()


def _graph(case, seed):
    rng = np.random.default_rng(seed)
    w, h = float(case["w"]), float(case["h"])
    g = FilterGraph((0.0, 0.0, w, h))
    cs = SPACES[case["space"]]
    prev = SOURCE_GRAPHIC
    for name in case["prims"].split(","):
        if name == "blur":
            prev = g.gaussian_blur(case["sx"], case["sy"], in1=prev, cs=cs)
        elif name in ("dilate", "erode"):
            op = abi.MORPH_DILATE if name == "dilate" else abi.MORPH_ERODE
            prev = g.morphology(op, case["sx"], case["sy"], in1=prev, cs=cs)
        elif name == "turbulence":
            f = rng.uniform(0.01, 0.1, 2)
            t = g.turbulence(float(f[0]), float(f[1]), 4, int(rng.integers(1000)), False, True, cs=cs)
            prev = g.composite(abi.COMPOSITE_IN, in1=t, in2=prev, cs=cs)
        elif name == "displacement":
            prev = g.displacement_map(float(rng.uniform(5.0, 40.0)), abi.CHANNEL_R, abi.CHANNEL_G, in1=prev,
                                      in2=SOURCE_GRAPHIC, cs=cs)
        elif name == "lighting":
            d = g.lighting(False, distant_light(float(rng.uniform(0, 360)), float(rng.uniform(10, 80))), 2.0, 1.0,
                           in1=SOURCE_ALPHA, cs=cs)
            p = g.lighting(True, point_light(w / 2, h / 2, 0.2 * w), 2.0, 1.0, 12.0, in1=prev, cs=cs)
            s = g.lighting(False, spot_light(0.0, 0.0, 0.3 * w, w, h, 0.0, 2.0, 35.0), 2.0, 1.0, in1=prev, cs=cs)
            prev = g.merge([d, s, p], cs=cs)
        elif name == "convolve":
            k = rng.integers(-4, 5, 25).astype(float)
            prev = g.convolve_matrix(5, 5, k.tolist(), in1=prev, cs=cs)
        elif name == "transfer":
            prev = g.component_transfer([("table", rng.uniform(0, 1, 5).tolist()), ("gamma", 1.2, 0.8, 0.05),
                                         ("discrete", rng.uniform(0, 1, 4).tolist()), ("linear", 0.9, 0.1)],
                                        in1=prev, cs=cs)
        elif name == "matrix":
            prev = g.color_matrix(abi.COLOR_MATRIX_MATRIX, rng.uniform(-1, 1, 20).tolist(), in1=prev, cs=cs)
        elif name == "arithmetic":
            k = rng.uniform(0.0, 0.8, 4)
            prev = g.composite(abi.COMPOSITE_ARITHMETIC, k=tuple(map(float, k)), in1=prev, in2=SOURCE_GRAPHIC, cs=cs)
        elif name == "shadow":
            prev = g.drop_shadow(6.0, 4.0, 3.0, 3.0, (20, 30, 60), 0.7, in1=prev, cs=cs)
        elif name == "tile":
            o = g.offset(5.0, 3.0, in1=prev, cs=cs, rect=(0.1 * w, 0.2 * h, 0.4 * w + 1.0, 0.3 * h + 1.0))
            prev = g.tile(in1=o, cs=cs)
        else:
            prev = g.blend("multiply", in1=prev, in2=SOURCE_GRAPHIC, cs=cs)
    return g


def _fits(case, seed):
    """The scenes (paths, gradient ends), parameters, geometry and dL/d(image) of one
    training step; outlines partly leave a canvas that is not square."""
    w, h, k = case["w"], case["h"], case["segments"]
    scenes, params, geoms = [], [], []
    for b in range(case.get("batch", 1)):
        _, _, paths, ends, p, _ = workloads.diff_scene(seed=seed * 1009 + b, size=max(w, h), n_paths=case["paths"],
                                                       segments=k, sigma=case["sigma"])
        scenes.append((paths, ends))
        params.append(p)
        geoms.append(diff.geometry(paths, k))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    shape = (len(scenes), h, w, 4)
    # the gradient of a mean squared error against another picture
    grad = torch.randn(shape, generator=gen, device="cuda") * (2.0 / (h * w * 4))
    return scenes, np.stack(params), np.stack(geoms), grad


def prepare(case, seed):
    kind = case["kind"]
    ctx = _ctx()
    if kind in ("document", "clipmask"):
        return {"kind": kind, "scene": _document(case, seed).to_abi(),
                "px": torch.zeros((case["h"], case["w"], 4), dtype=torch.uint8, device="cuda")}
    if kind == "host":
        return {"kind": kind, "scene": _document(case, seed).to_abi(),
                "px": np.zeros((case["h"], case["w"], 4), np.uint8)}
    if kind == "batch":
        specs = _batch_specs(case)
        docs = [workloads.batch_doc(seed * 4099 + i, *sp) for i, sp in enumerate(specs)]
        return {"kind": kind, "scenes": [sc.to_abi() for sc in docs],
                "px": [torch.zeros((sp[1], sp[0], 4), dtype=torch.uint8, device="cuda") for sp in specs]}
    if kind == "filter":
        src = _layer(case["w"], case["h"], seed)
        return {"kind": kind, "graph": _graph(case, seed), "src": src, "px": torch.empty_like(src)}
    if kind == "png":
        w, h = case["w"], case["h"]
        return {"kind": kind, "src": _layer(w, h, seed),
                "rows": torch.empty(h * (4 * w + 1), dtype=torch.uint8, device="cuda")}
    scenes, params, geoms, grad = _fits(case, seed)
    if kind == "planes":
        r = diff.Renderer(ctx, case["w"], case["h"], *scenes[0])
        return {"kind": kind, "r": r, "params": torch.as_tensor(params[0], device="cuda"), "grad": grad[0]}
    r = diff.Renderer.batched(ctx, case["w"], case["h"], scenes, cubics=case["segments"])
    return {"kind": kind, "r": r, "params": torch.as_tensor(params, device="cuda"),
            "geom": torch.as_tensor(geoms, device="cuda"), "grad": grad}


# --- one pass --------------------------------------------------------------------
def run(state):
    ctx, kind = _ctx(), state["kind"]
    ts = abi.Transform.identity()
    if kind in ("document", "clipmask"):
        state["px"].zero_()  # render composites: a new picture starts from a clear pixmap
        ctx.render(state["scene"], ts, state["px"])
        return state["px"]
    if kind == "host":
        state["px"].fill(0)
        ctx.render_host(state["scene"], ts, state["px"])
        return state["px"]
    if kind == "batch":
        for px in state["px"]:
            px.zero_()
        ctx.render_batch(state["scenes"], ts, state["px"])
        return state["px"]
    if kind == "filter":
        state["px"].copy_(state["src"])  # the filter works on the layer in place
        ctx.filter_apply(state["graph"], ts, state["px"])
        return state["px"]
    if kind == "png":
        ctx.png_filter_rows(state["src"], state["rows"])
        return state["rows"]
    r = state["r"]
    if kind == "planes":
        out = r.forward(state["params"])
        return {"image": out, "params": r.backward(state["params"], state["grad"])}
    out = r.forward(state["params"], state["geom"])
    gp, gg = r.backward(state["params"], state["grad"], state["geom"])
    return {"image": out, "params": gp, "geom": gg}


# --- work and tolerance ----------------------------------------------------------
# operations per painted pixel of a path: a gradient colour and one SourceOver of four
# channels; paths with points uniform in the canvas paint about half of it
PAINT_FLOPS = 20.0
# per pixel of a pass: what the primitives of a graph need (octaves of noise, taps)
PRIM_FLOPS = {"blur": 60.0, "dilate": 24.0, "erode": 24.0, "turbulence": 600.0, "displacement": 12.0,
              "lighting": 180.0, "convolve": 100.0, "transfer": 8.0, "matrix": 40.0, "arithmetic": 24.0,
              "shadow": 70.0, "tile": 2.0, "blend": 20.0}


def work(case):
    kind = case["kind"]
    if kind in ("document", "host"):
        px = case["w"] * case["h"]
        return {"bytes": 8.0 * px + 2000.0 * case["paths"],
                "flops": PAINT_FLOPS * 0.5 * case["paths"] * px + 60.0 * case["prims"] * px}
    if kind == "clipmask":
        px = case["w"] * case["h"]
        # two paths, a clip path of two and a mask of two for about half of the groups
        return {"bytes": 8.0 * px + 2000.0 * 2 * case["groups"], "flops": PAINT_FLOPS * 2.0 * case["groups"] * px}
    if kind == "batch":
        specs = _batch_specs(case)
        return {"bytes": sum(8.0 * w * h + 2000.0 * n for w, h, n, _ in specs),
                "flops": sum(w * h * (PAINT_FLOPS * 0.5 * n + 60.0 * k) for w, h, n, k in specs)}
    if kind == "filter":
        px = case["w"] * case["h"]
        return {"bytes": 8.0 * px, "flops": px * sum(PRIM_FLOPS[p] for p in case["prims"].split(","))}
    px = case["w"] * case["h"]
    if kind == "png":
        return {"bytes": 8.0 * px, "flops": 40.0 * px}
    n, b = case["paths"], case.get("batch", 1)
    per_path = 30.0 + 90.0  # paint and composite, and their adjoint
    blur = 4 * 2 * 4 * (2 * min(math.ceil(3.0 * case["sigma"]), 48) + 1)
    cover = n if kind == "planes" else 0
    return {"bytes": b * px * (32.0 + cover), "flops": b * px * (n * per_path * 0.5 + blur)}


def tolerance(case):
    # Four times the largest distance from exact() seen over the declared ranges (the listed
    # cases and twelve drawn ones, two seeds each): images are within 1e-5, but the gradients
    # have kinks (the clamped colour, coverage min(1, |area|), a pixel's side of an edge), and
    # a last-bit difference that takes one pixel over one of them moves a gradient by that
    # pixel's share: 5e-4 of the paint gradients (2e-3 over analytic coverage), 5.6e-3 of the geometry's, single
    # entries 0.21.
    if case["kind"] == "planes":
        return {"rel": 2e-3, "max": 0.05}
    if case["kind"] == "analytic":
        return {"rel": 2.2e-2, "max": 0.84}
    return "exact"


# --- the differentiable form in float64 ------------------------------------------
def _paint(cov, ends, q, px, py, s):
    """SourceOver of one path: coverage, tint, opacity and a 4-stop pad gradient."""
    tint, opacity, col, off = q[0:3], q[3], q[4:20].reshape(4, 4), q[20:24]
    x0, y0, x1, y1 = ends
    dx, dy = x1 - x0, y1 - y0
    dd = dx * dx + dy * dy
    t = (((px - x0) * dx + (py - y0) * dy) / dd).clamp(0.0, 1.0) if dd > 0 else torch.zeros_like(px)
    before, after = t <= off[0], t >= off[3]
    after = after & ~before
    k = torch.where(t < off[1], 0, torch.where(t < off[2], 1, 2))
    k = torch.where(before, 0, torch.where(after, 2, k))
    lo, hi = torch.zeros_like(t), torch.zeros_like(t)
    for j in range(3):
        lo = torch.where(k == j, off[j], lo)
        hi = torch.where(k == j, off[j + 1], hi)
    span = hi - lo
    u = torch.where(span > 0, (t - lo) / torch.where(span > 0, span, 1.0), 0.0)
    u = torch.where(before, 0.0, torch.where(after, 1.0, u))
    zero = torch.zeros_like(u)
    wts = torch.stack([torch.where(k == j, 1.0 - u, zero) + torch.where(k + 1 == j, u, zero) for j in range(4)])
    c = (col.t() @ wts.reshape(4, -1)).reshape(4, *t.shape)
    a = cov * opacity * c[3]
    src = torch.cat([c[:3] * tint[:, None, None] * a, a[None]])
    return src + (1.0 - a) * s


def _paint_run(cov, ends, params, px, py, s, i0):
    for j in range(cov.shape[0]):
        q = params[(i0 + j) * diff.PATH_PARAMS:(i0 + j + 1) * diff.PATH_PARAMS]
        s = _paint(cov[j], ends[i0 + j], q, px, py, s)
    return s


def _picture(cov, ends, params):
    """Paths, then blur, colour matrix and the composite over the paths."""
    from torch.utils.checkpoint import checkpoint
    n, h, w = cov.shape
    dev = cov.device
    py, px = torch.meshgrid(torch.arange(h, device=dev, dtype=torch.float64) + 0.5,
                            torch.arange(w, device=dev, dtype=torch.float64) + 0.5, indexing="ij")
    s = torch.zeros((4, h, w), dtype=torch.float64, device=dev)
    for i in range(0, n, 16):
        s = checkpoint(_paint_run, cov[i:i + 16], ends, params, px, py, s, i, use_reentrant=False)
    sigma = params[n * diff.PATH_PARAMS].clamp(0.05, 16.0)
    r = min(math.ceil(float(np.float32(3.0) * np.float32(float(sigma.detach())))), 48)
    j = torch.arange(-r, r + 1, device=dev, dtype=torch.float64)
    g = torch.exp(-j * j / (2.0 * sigma * sigma))
    g = g / g.sum()
    pad = torch.nn.functional.pad(s, (r, r))
    x = sum(g[m] * pad[:, :, m:m + w] for m in range(2 * r + 1))
    pad = torch.nn.functional.pad(x, (0, 0, r, r))
    b = sum(g[m] * pad[:, m:m + h] for m in range(2 * r + 1))
    m = params[n * diff.PATH_PARAMS + 1:].reshape(4, 5)
    v = torch.cat([b[:3] / b[3].clamp(min=1.0 / 255.0), b[3:4]])
    o = (m[:, :4] @ v.reshape(4, -1)).reshape(4, h, w) + m[:, 4][:, None, None]
    q = o.clamp(0.0, 1.0)
    f = torch.cat([q[:3] * q[3], q[3:4]])
    return (f + (1.0 - q[3]) * s).permute(1, 2, 0)


def _antiderivative(u):
    """The integral of clamp(u, 0, 1)."""
    c = u.clamp(0.0, 1.0)
    return 0.5 * c * c + (u - 1.0).clamp(min=0.0)


def _winding_area(geom, k, w, h):
    """The integral of the winding number over every pixel, of each path's cubics
    flattened at 16 uniform parameters and closed: (paths, h, w)."""
    n, dev = geom.shape[0], geom.device
    a, pts = geom[:, :6], geom[:, 6:].reshape(n, 3 * k + 1, 2)
    jj = torch.arange(k * 16 + 1, device=dev)
    c = (jj // 16).clamp(max=k - 1)
    t = ((jj - 16 * c).to(torch.float64) / 16.0)[:, None]
    u = 1.0 - t
    v = (u * u * u * pts[:, 3 * c] + 3.0 * u * u * t * pts[:, 3 * c + 1] + 3.0 * u * t * t * pts[:, 3 * c + 2] +
         t * t * t * pts[:, 3 * c + 3])
    x = a[:, 0:1] * v[..., 0] + a[:, 2:3] * v[..., 1] + a[:, 4:5]
    y = a[:, 1:2] * v[..., 0] + a[:, 3:4] * v[..., 1] + a[:, 5:6]
    xa, ya = x.reshape(-1), y.reshape(-1)
    xb, yb = x.roll(-1, 1).reshape(-1), y.roll(-1, 1).reshape(-1)
    path = torch.arange(n, device=dev).repeat_interleave(k * 16 + 1)
    # every (edge, row) the edge spans
    r0 = torch.minimum(ya, yb).detach().floor().clamp(0, h).long()
    r1 = torch.maximum(ya, yb).detach().ceil().clamp(0, h).long()
    cnt = (r1 - r0).clamp(min=0)
    cnt = torch.where((ya == yb).detach(), torch.zeros_like(cnt), cnt)
    e = torch.arange(xa.numel(), device=dev).repeat_interleave(cnt)
    row = r0[e] + torch.arange(e.numel(), device=dev) - (cnt.cumsum(0) - cnt)[e]
    up = yb[e] > ya[e]
    yt, yl = torch.where(up, ya[e], yb[e]), torch.where(up, yb[e], ya[e])
    t0, t1 = torch.maximum(yt, row.to(torch.float64)), torch.minimum(yl, row.to(torch.float64) + 1.0)
    slope = (xb[e] - xa[e]) / (yb[e] - ya[e])
    p, q = xa[e] + slope * (t0 - ya[e]), xa[e] + slope * (t1 - ya[e])
    d = (t1 - t0) * torch.where(up, 1.0, -1.0)
    lo, hi = torch.minimum(p, q), torch.maximum(p, q)
    j0, j1 = lo.detach().floor().clamp(0, w).long(), hi.detach().floor().clamp(-1, w - 1).long()
    # every pixel right of the stretch takes the whole of it
    plane = path[e] * h + row
    step = torch.zeros(n * h * (w + 1), dtype=torch.float64, device=dev)
    step = step.index_add(0, plane * (w + 1) + torch.maximum(j1 + 1, torch.zeros_like(j1)).clamp(max=w), d)
    area = step.reshape(n, h, w + 1).cumsum(2)[..., :w]
    # the pixels it crosses take the part right of it
    num = (j1 - j0 + 1).clamp(min=0)
    f = torch.arange(e.numel(), device=dev).repeat_interleave(num)
    col = j0[f] + torch.arange(f.numel(), device=dev) - (num.cumsum(0) - num)[f]
    edge = col.to(torch.float64) + 1.0
    width = hi[f] - lo[f]
    flat = width < 1e-9
    part = torch.where(flat, (edge - 0.5 * (lo[f] + hi[f])).clamp(0.0, 1.0),
                       (_antiderivative(edge - lo[f]) - _antiderivative(edge - hi[f])) / torch.where(flat, 1.0, width))
    some = torch.zeros(n * h * w, dtype=torch.float64, device=dev).index_add(0, plane[f] * w + col, part * d[f])
    return area + some.reshape(n, h, w)


def exact(case, seed):
    """The differentiable form in float64; the bytes of the other kinds have no value
    beside themselves.  The u8 coverage planes are an input of the planes form."""
    kind = case["kind"]
    if kind not in ("planes", "analytic"):
        return None
    scenes, params, geoms, grad = _fits(case, seed)
    p = torch.as_tensor(params, device="cuda").double()
    images, gps, ggs = [], [], []
    for b, (_, ends) in enumerate(scenes):
        q = p[b].clone().requires_grad_(True)
        e = [tuple(float(v) for v in row) for row in ends]
        leaves = [q]
        if kind == "planes":
            cov = prepare(case, seed)["r"].coverage.double() / 255.0
        else:
            g = torch.as_tensor(geoms[b], device="cuda").double().requires_grad_(True)
            leaves.append(g)
            cov = _winding_area(g, case["segments"], case["w"], case["h"]).abs().clamp(max=1.0)
        img = _picture(cov, e, q)
        got = torch.autograd.grad(img, leaves, grad[b].double())
        images.append(img.detach())
        gps.append(got[0])
        if kind == "analytic":
            ggs.append(got[1])
    if kind == "planes":
        return {"image": images[0], "params": gps[0]}
    return {"image": torch.stack(images), "params": torch.stack(gps), "geom": torch.stack(ggs)}
