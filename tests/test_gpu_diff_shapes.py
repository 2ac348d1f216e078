"""The differentiable form at the edges of its kernels' blocks (64 x 4 pixels of 16 x 4 waves,
segments of 8 paths, blur blocks of 64 x 32 and 256 x 4, rows of winding area in LDS), at
stop intervals without width, and its area rows that are too long for LDS."""
import numpy as np
import pytest

from oracle import diff_ref as D
from resvg_amd import diff
from resvg_amd.workloads import diff_scene

pytestmark = pytest.mark.gpu


def _planes(ctx, w, h, n, seed, sigma=1.3, equal_offsets=False):
    import torch
    _, _, paths, ends, p0, _ = diff_scene(seed=seed, size=max(w, h), n_paths=n, segments=3, sigma=sigma)
    if equal_offsets:
        for i in range(n):  # one interval without width, or all of them
            o = p0[i * diff.PATH_PARAMS + 20:i * diff.PATH_PARAMS + 24]
            o[:] = o[0] if i % 3 == 0 else (np.float32([o[0], o[1], o[1], o[3]]) if i % 3 == 1 else o)
    r = diff.Renderer(ctx, w, h, paths, ends)
    return r, torch.as_tensor(p0, device="cuda"), r.coverage.cpu().numpy(), np.asarray(ends, np.float32)


@pytest.mark.parametrize("w,h", [(1, 1), (3, 63), (63, 3), (64, 4), (65, 5), (16, 33), (17, 129), (256, 32), (257, 33)])
@pytest.mark.parametrize("n", [1, 8, 9])
def test_shapes_forward(ctx, w, h, n):
    r, params, cov, ends = _planes(ctx, w, h, n, seed=w + h + n)
    out = r.forward(params).cpu().numpy()
    # 2e-5: f32 sums of up to 9 composites, 9 x 9 taps and a matrix, as for the oracle tests
    assert np.abs(out - D.forward(cov, ends, params.cpu().numpy(), w, h)).max() < 2e-5


@pytest.mark.parametrize("sigma", [0.05, 0.4, 6.0, 16.0])
def test_blur_radii(ctx, sigma):
    r, params, cov, ends = _planes(ctx, 70, 37, 4, seed=5, sigma=sigma)
    out = r.forward(params).cpu().numpy()
    assert np.abs(out - D.forward(cov, ends, params.cpu().numpy(), 70, 37)).max() < 2e-5


def test_stop_intervals_without_width(ctx):
    r, params, cov, ends = _planes(ctx, 65, 40, 9, seed=3, equal_offsets=True)
    out = r.forward(params).cpu().numpy()
    assert np.abs(out - D.forward(cov, ends, params.cpu().numpy(), 65, 40)).max() < 2e-5


def test_gradient_through_stop_intervals_without_width(ctx):
    # the offsets of a path with such an interval have no derivative there; every other
    # parameter, and the other paths' offsets, do
    import torch
    w, h, n = 65, 17, 9
    r, params, cov, ends = _planes(ctx, w, h, n, seed=4, equal_offsets=True)
    go = np.random.default_rng(4).normal(0.0, 1.0, (h, w, 4)).astype(np.float32)
    r.forward(params)
    g = r.backward(params, torch.as_tensor(go, device="cuda")).cpu().numpy().astype(np.float64)
    assert np.isfinite(g).all()
    P = diff.PATH_PARAMS
    idx = [j for j in range(len(g)) if j >= n * P or j % P < 20 or (j // P) % 3 == 2]
    ref = D.grad_fd(cov, ends, params.cpu().numpy(), w, h, go, idx)
    assert np.linalg.norm(g[idx] - ref[idx]) / np.linalg.norm(ref[idx]) < 1e-3  # as for the oracle tests


@pytest.mark.parametrize("w,h,n", [(63, 5, 3), (66, 9, 9)])
def test_shapes_gradient(ctx, w, h, n):
    import torch
    r, params, cov, ends = _planes(ctx, w, h, n, seed=w)
    go = np.random.default_rng(w).normal(0.0, 1.0, (h, w, 4)).astype(np.float32)
    r.forward(params)
    g = r.backward(params, torch.as_tensor(go, device="cuda")).cpu().numpy().astype(np.float64)
    ref = D.grad_fd(cov, ends, params.cpu().numpy(), w, h, go)
    assert np.linalg.norm(g - ref) / np.linalg.norm(ref) < 1e-3  # as for the oracle tests


@pytest.mark.parametrize("w", [8189, 8190, 8191, 8300])
def test_long_area_rows_match_short_ones(ctx, w):
    # the same paths on canvases whose rows do and do not fit LDS: the areas are exact
    # integer sums, so every pixel away from the right edge has the same bits
    import torch
    _, _, paths, ends, p0, _ = diff_scene(seed=2, size=600, n_paths=2, segments=2, sigma=0.5)
    paths = [(v, np.asarray(p, np.float32) * np.float32([14.0, 0.05])) for v, p in paths]
    outs = []
    for width in (8100, w):
        r = diff.Renderer(ctx, width, 19, paths, ends, cubics=2)
        outs.append(r.forward(torch.as_tensor(p0, device="cuda"), r.geom0).cpu().numpy()[:, :8000])
    assert np.abs(outs[0]).max() > 0.1
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("k", [1, 31, 32, 33, 511, 512, 600])
@pytest.mark.parametrize("kind", ["outline", "wild", "nan"])
def test_areas_of_many_cubics(ctx, k, kind):
    # bands gather the cubics, then the edges, that meet them (512 at a time): the areas have
    # the bits of the form for long rows, which visits every edge's own rows
    import torch
    from resvg_amd import abi
    rng = np.random.default_rng(k)
    t = np.linspace(0.0, 2.0 * np.pi, 3 * k + 1)
    paths = []
    for i in range(3):
        r = 0.4 + 0.05 * np.sin(7 * t + i) + (rng.uniform(-0.4, 0.4, t.size) if kind != "outline" else 0.0)
        pts = np.stack([150.0 + 180.0 * r * np.cos(t), 18.0 + 60.0 * r * np.sin(t)], 1).astype(np.float32)
        if kind == "nan" and i == 1:
            pts[3 * k // 2, 1] = np.nan
        paths.append(([abi.VERB_MOVE] + [abi.VERB_CUBIC] * k + [abi.VERB_CLOSE], pts))
    p = np.zeros(diff.n_params(3), np.float32)
    p[:72] = 0.5
    p[72] = 0.05  # no colour matrix: the picture is the paths' canvas
    outs = []
    for width in (300, 8200):
        r = diff.Renderer(ctx, width, 37, paths, np.zeros((3, 4), np.float32), cubics=k)
        outs.append(r.forward(torch.as_tensor(p, device="cuda"), r.geom0).cpu().numpy()[:, :299])
    assert outs[0][..., 3].max() > 0.1
    assert np.array_equal(outs[0], outs[1], equal_nan=True)


# ---- non-finite values stay where they are -----------------------------------------
def _rect(x0, x1, y1, y0=0):
    from resvg_amd import abi
    pts = [(x0, y0), (x1, y0), (x1, y1), (x0, y1)]
    return [abi.VERB_MOVE, abi.VERB_LINE, abi.VERB_LINE, abi.VERB_LINE, abi.VERB_CLOSE], np.asarray(pts, np.float32)


def _columns(ctx, w, h, spans, wide):
    """Opaque-edged columns x0 <= x < x1 under a zero colour matrix: the picture is the paths'
    canvas and, within the blur's reach of finite pixels, dL/d(canvas) is dL/d(picture), so a
    path's gradient comes from its pixels alone.
    `wide`: the gradients' stops far apart (a wave in one interval) or close (in several)."""
    n = len(spans)
    rng = np.random.default_rng(7)
    ends = np.float32([(-200.0, 0.0, 300.0, 0.0) if wide else (x0, 0.0, x1, 0.0) for x0, x1 in spans])
    p = np.zeros(diff.n_params(n), np.float32)
    for i in range(n):
        q = p[i * diff.PATH_PARAMS:(i + 1) * diff.PATH_PARAMS]
        q[:20] = rng.uniform(0.3, 0.9, 20)
        q[20:24] = (0.1, 0.3, 0.6, 0.9)
    p[n * diff.PATH_PARAMS] = 0.05  # radius 1
    return diff.Renderer(ctx, w, h, [_rect(x0, x1, h) for x0, x1 in spans], ends), p


def _grad(r, p, go):
    import torch
    params = torch.as_tensor(p, device="cuda")
    r.forward(params)
    return r.backward(params, torch.as_tensor(go, device="cuda")).cpu().numpy()


@pytest.mark.parametrize("wide", [True, False])
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_upstream_at_uncovered_pixels(ctx, value, wide):
    # the gradient of a path does not depend on dL/d(picture) where it has no coverage, also
    # where its wave of 16 x 4 pixels has some
    r, p = _columns(ctx, 16, 4, [(0, 8)], wide)
    go = np.random.default_rng(1).normal(0.0, 1.0, (4, 16, 4)).astype(np.float32)
    want = _grad(r, p, go)[:diff.PATH_PARAMS]
    go[1, 12] = value
    assert np.isfinite(want).all() and want.any()
    assert np.array_equal(_grad(r, p, go)[:diff.PATH_PARAMS], want)


@pytest.mark.parametrize("wide", [True, False])
@pytest.mark.parametrize("param,value", [(0, np.nan), (3, np.inf), (3, np.nan), (7, np.inf), (11, np.nan)])
def test_paint_at_uncovered_pixels(ctx, param, value, wide):
    # nor on the paint of another path over other pixels of the wave
    r, p = _columns(ctx, 16, 4, [(10, 16), (0, 2)], wide)
    go = np.random.default_rng(2).normal(0.0, 1.0, (4, 16, 4)).astype(np.float32)
    want = _grad(r, p, go)[:diff.PATH_PARAMS]
    p[diff.PATH_PARAMS + param] = value
    assert np.isfinite(want).all() and want.any()
    assert np.array_equal(_grad(r, p, go)[:diff.PATH_PARAMS], want)


def test_overflowing_slope_is_infinite(ctx):
    # finite values whose product overflows along the gradient: the offsets of the stops on
    # either side take an infinity of its sign, not a NaN
    r, p = _columns(ctx, 16, 4, [(0, 8)], True)
    p[:4] = 1.0
    p[4:20] = np.float32([[0, 0, 0, 1], [0, 0, 0, 1], [100, 0, 0, 1], [0, 0, 0, 1]]).ravel()
    p[20:24] = (0.1, 0.39, 0.6, 0.9)
    go = np.zeros((4, 16, 4), np.float32)
    go[1, 3, 0] = 1e37  # at u = 0.08 of the second interval: times 100 past the largest float
    g = _grad(r, p, go)
    assert g[21] == g[22] == -np.inf
    go[1, 3, 0] = -1e37
    g = _grad(r, p, go)
    assert g[21] == g[22] == np.inf


@pytest.mark.parametrize("k", [0, 1, 2, 3])
def test_offsets_that_are_no_numbers(ctx, k):
    # a pixel is in the interval whose upper offset it is below; an interval with a NaN end
    # has no width (the lower stop's colour), and no pixel lies between stops of which the
    # first or last is one
    r, p = _columns(ctx, 32, 4, [(0, 32)], False)
    p[20 + k] = np.nan
    go = np.random.default_rng(3).normal(0.0, 1.0, (4, 32, 4)).astype(np.float32)
    import torch
    out = r.forward(torch.as_tensor(p, device="cuda")).cpu().numpy()
    with np.errstate(invalid="ignore"):
        ref = D.forward(r.coverage.cpu().numpy(), r.ends.cpu().numpy()[0], p, 32, 4)
    assert np.abs(out - ref).max() < 2e-5  # as in the tests above
    g = _grad(r, p, go)[:diff.PATH_PARAMS]
    assert np.isfinite(g).all() and (k in (1, 2) or not g[20:24].any())


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("sigma,radius", [(0.05, 1), (0.6, 2), (1.0, 3), (2.5, 8)])
def test_blur_reaches_its_radius_only(ctx, sigma, radius, value):
    # a blur thread makes several outputs from each input it reads; those further than the
    # radius from a non-finite pixel keep their bits, in the picture and in the gradients
    import torch
    n, bad = 45, 21
    lo, hi = bad - radius, bad + radius + 1
    rects = [_rect(bad, bad + 1, bad + 1, bad), _rect(0, lo, n), _rect(hi, n, n), _rect(0, n, lo), _rect(0, n, n, hi)]
    r = diff.Renderer(ctx, n, n, rects, np.float32([(-90.0, -80.0, 120.0, 90.0)] * 5))
    P = diff.PATH_PARAMS
    p = np.zeros(diff.n_params(5), np.float32)
    for i in range(5):
        p[i * P:i * P + 20] = np.random.default_rng(i).uniform(0.3, 0.6, 20)
        p[i * P + 20:i * P + 24] = (0.1, 0.3, 0.6, 0.9)
    p[5 * P] = sigma
    p[5 * P + 1:] = np.float32([[0.8, 0, 0, 0, 0.1], [0, 0.8, 0, 0, 0.1], [0, 0, 0.8, 0, 0.1], [0, 0, 0, 0.8, 0.1]]).ravel()

    def run(p, go):
        params = torch.as_tensor(p, device="cuda")
        img = r.forward(params).cpu().numpy()
        return img, r.backward(params, torch.as_tensor(go, device="cuda")).cpu().numpy()

    go = np.random.default_rng(9).normal(0.0, 1.0, (n, n, 4)).astype(np.float32)
    go[lo:hi, lo:hi] = 0.0
    img, grad = run(p, go)
    assert np.isfinite(img).all() and np.isfinite(grad).all() and grad[P:2 * P].any()
    q = p.copy()
    q[0] = value  # the tint of the path that covers the pixel alone
    far = np.ones((n, n), bool)
    far[lo:hi, lo:hi] = False
    assert np.array_equal(run(q, go)[0][far], img[far])
    go[bad, bad] = value
    assert np.array_equal(run(p, go)[1][P:5 * P], grad[P:5 * P])


@pytest.mark.parametrize("w,h", [(1024, 1024), (2048, 1536), (1000, 700)])
def test_rounding_of_the_sum_over_pixels(ctx, w, h):
    # every pixel of a full canvas adds the same value to the tint's gradient, so all rounding
    # is that of the sum.  A pixel's value passes the wave's tree (6 additions), the block's
    # 4 waves, one of 8 sums of up to `chain` partial rows, 3 and 6 levels of pairs; each
    # rounds by at most half a unit, 2^-24 of the sum
    r = diff.Renderer(ctx, w, h, [_rect(0, w, h)], np.zeros((1, 4), np.float32))
    P = diff.PATH_PARAMS
    p = np.zeros(diff.n_params(1), np.float32)
    p[:20] = 1.0
    p[20:24] = (0.1, 0.3, 0.6, 0.9)
    p[P] = 0.05  # no colour matrix: dL/d(canvas) is dL/d(picture)
    tiles = -(-w // 64) * -(-h // 4)
    chain = -(-tiles // 512)
    for seed in range(4):
        g = np.random.default_rng(seed).uniform(1.0, 2.0, 3).astype(np.float32)
        go = np.zeros((h, w, 4), np.float32)
        go[..., :3] = g
        rel = np.abs(_grad(r, p, go)[:3].astype(np.float64) / (g.astype(np.float64) * (w * h)) - 1.0)
        assert rel.max() <= (6 + 3 + chain + 9) * 2.0 ** -24
