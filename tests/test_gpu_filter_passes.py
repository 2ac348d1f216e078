"""Filter passes where their kernels' cases change: every channel value at every alpha
through the corrected quotients, widths that leave remainders of the four pixels a thread
takes, and graphs whose results are used several times (an image that its last user takes
over must not be one that another still reads).  Byte for byte against the oracle."""
import numpy as np
import pytest

from oracle import bindings as orc
from resvg_amd import abi
from resvg_amd.filters import SOURCE_ALPHA, SOURCE_GRAPHIC, FilterGraph

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _random(h, w, seed, holes=0.5):
    rng = np.random.default_rng(seed)
    px = rng.integers(0, 256, (h, w, 4))
    px[rng.random((h, w)) < holes] = 0
    px[..., :3] = px[..., :3] * px[..., 3:] // 255
    return px.astype(np.uint8)


@pytest.mark.parametrize("name", ["into_linear_rgb", "into_srgb", "demultiply_alpha", "multiply_alpha"])
def test_every_channel_at_every_alpha(ctx, name):
    a, c = np.meshgrid(np.arange(256), np.arange(256), indexing="ij")
    px = np.stack([c, 255 - c, (c * 7) % 256, a], -1).astype(np.uint8).reshape(1, -1, 4)[:, 1:]
    t, e = _dev(px), px.copy()
    getattr(ctx, name)(t)
    getattr(orc, name)(e)
    assert np.array_equal(t.cpu().numpy(), e)


@pytest.mark.parametrize("values", [[0.3] * 20, [1.7, -0.4, 0.0, 0.2, 0.01] * 4])
def test_matrix_of_every_channel_at_every_alpha(ctx, values):
    a, c = np.meshgrid(np.arange(256), np.arange(256), indexing="ij")
    px = np.stack([c, 255 - c, (c * 7) % 256, a], -1).astype(np.uint8)
    g = FilterGraph((0, 0, 256, 256))
    g.color_matrix(abi.COLOR_MATRIX_MATRIX, values, cs=abi.CI_SRGB)
    t, e = _dev(px), px.copy()
    ts = abi.Transform(1.0, 0.0, 0.0, 1.0, 0.0, 0.0)
    assert ctx.filter_apply(g, ts, t) == orc.filter_apply(g, ts, e)
    assert np.array_equal(t.cpu().numpy(), e)


@pytest.mark.parametrize("mode", ["source_over", "multiply", "xor", "destination"])
@pytest.mark.parametrize("dw,sw,x", [(7, 7, 0), (1029, 1029, 0), (61, 30, 5), (300, 259, 17), (20, 50, -13)])
def test_draw_widths(ctx, mode, dw, sw, x):
    names = [m.replace("-", "_").lower() for m in abi.BLEND_MODES]
    m = names.index(mode)
    for opacity in (1.0, 0.37, 0.0):
        d, s = _random(9, dw, 1), _random(11, sw, 2)
        t, e = _dev(d), d.copy()
        ctx.draw_pixmap(t, x, -1, _dev(s), opacity, m)
        orc.draw_pixmap(e, x, -1, s, opacity, m)
        assert np.array_equal(t.cpu().numpy(), e), opacity


@pytest.mark.parametrize("rect", [(0, 0, 61, 4), (3, 1, 7, 5), (1, 0, 300, 9), (-4, 2, 9, 100)])
def test_clear_widths(ctx, rect):
    px = _random(9, 61, 3, 0.0)
    t, e = _dev(px), px.copy()
    ctx.clear_rect(t, *rect)
    x0, y0 = max(rect[0], 0), max(rect[1], 0)
    e[y0:rect[1] + rect[3], x0:rect[0] + rect[2]] = 0
    assert np.array_equal(t.cpu().numpy(), e)


def _reusing_graph(rng, region):
    g = FilterGraph(region)
    ids = [SOURCE_GRAPHIC, SOURCE_ALPHA]
    for _ in range(int(rng.integers(4, 10))):
        a, b = (int(ids[rng.integers(len(ids))]) for _ in range(2))
        kw = {"cs": int(rng.integers(2))}
        if rng.random() < 0.2:
            x, y, w, h = region
            kw["rect"] = (x + w * 0.25, y + h * 0.125, w * 0.5, h * 0.5)
        k = int(rng.integers(12))
        if k == 0:
            r = g.gaussian_blur(float(rng.uniform(2, 6)), float(rng.uniform(2, 6)), in1=a, **kw)
        elif k == 1:
            r = g.gaussian_blur(0.0, 0.0, in1=a, **kw)
        elif k == 2:
            r = g.offset(float(rng.integers(0, 4)), 0.0, in1=a, **kw)
        elif k == 3:
            r = g.blend(int(rng.integers(len(abi.BLEND_MODES))), in1=a, in2=b, **kw)
        elif k == 4:
            r = g.composite(int(rng.integers(6)), k=(0.3, -0.2, 0.9, 0.0), in1=a, in2=b, **kw)
        elif k == 5:
            r = g.merge([a, b, a, int(ids[rng.integers(len(ids))])][:int(rng.integers(0, 5))], **kw)
        elif k == 6:
            r = g.displacement_map(9.0, abi.CHANNEL_R, abi.CHANNEL_A, in1=a, in2=b, **kw)
        elif k == 7:
            r = g.convolve_matrix(3, 2, rng.integers(-3, 4, 6).astype(float), in1=a, **kw)
        elif k == 8:
            r = g.color_matrix(abi.COLOR_MATRIX_SATURATE, [0.4], in1=a, **kw)
        elif k == 9:
            r = g.drop_shadow(2.0, 1.0, 2.5, float(rng.integers(2)), (9, 200, 30), 0.6, in1=a, **kw)
        elif k == 10:
            r = g.turbulence(0.06, 0.03, 3, 5, bool(rng.integers(2)), bool(rng.integers(2)), **kw)
        else:
            r = g.morphology(int(rng.integers(2)), 1.0, 2.0, in1=a, **kw)
        ids.append(r)
    return g


@pytest.mark.parametrize("seed", range(24))
def test_results_used_again(ctx, seed):
    rng = np.random.default_rng(seed)
    h, w = int(rng.integers(3, 70)), int(rng.integers(3, 150))
    layer = _random(h, w, seed, 0.3)
    # the layer's own size (images written whole), or a part of it
    region = (0.0, 0.0, float(w), float(h)) if seed % 3 else (1.0, 2.0, float(w) * 0.75, float(h))
    g = _reusing_graph(rng, region)
    ts = abi.Transform(1.0, 0.0, 0.0, 1.0, 0.0, 0.0)
    t, e = _dev(layer), layer.copy()
    assert ctx.filter_apply(g, ts, t) == orc.filter_apply(g, ts, e)
    assert np.array_equal(t.cpu().numpy(), e)


@pytest.mark.parametrize("order", [(5, 5), (7, 9), (64, 1), (1, 64), (1, 1)])
@pytest.mark.parametrize("edge", [abi.EDGE_NONE, abi.EDGE_DUPLICATE, abi.EDGE_WRAP])
@pytest.mark.parametrize("shape", [(1, 1), (3, 2), (17, 65), (33, 130)])
def test_convolution_tiles(ctx, order, edge, shape):
    # images smaller and larger than a block's 64 x 4 pixels and than the matrix, an infinite
    # coefficient; images large enough for tiles in LDS are in the test below
    rng = np.random.default_rng(order[0] * 100 + order[1] + edge)
    k = rng.uniform(-1, 1, order[0] * order[1])
    for k0, preserve in ((k[0], False), (k[0], True), (float("inf"), False)):
        k[0] = k0
        g = FilterGraph((0, 0, 1, 1))
        g.convolve_matrix(order[0], order[1], k, 1.5, 0.1, edge_mode=edge, preserve_alpha=preserve)
        px = _random(*shape, 7)
        t, e = _dev(px), px.copy()
        ctx.convolve_matrix(t, g.primitives[0], g.values)
        orc.convolve_matrix(e, g.primitives[0], g.values)
        assert np.array_equal(t.cpu().numpy(), e), (k0, preserve)


@pytest.mark.parametrize("edge", [abi.EDGE_NONE, abi.EDGE_DUPLICATE, abi.EDGE_WRAP])
@pytest.mark.parametrize("shape", [(1021, 1029), (1025, 1023), (1023, 1025), (17, 61681), (1031, 1018),
                                   (17, 15421), (513, 511), (514, 511)])
def test_convolution_by_size(ctx, edge, shape):
    # from memory a thread takes one pixel, or four from 2^20 pixels on, with every remainder
    # of a row (matrices of more than 64 entries and with an infinite one); the others are
    # tiled from 2^18 pixels on
    rng = np.random.default_rng(edge)
    px = _random(*shape, 7)
    inf = rng.uniform(-1, 1, 6)
    inf[1] = float("inf")
    for order, k in (((5, 13), rng.uniform(-1, 1, 65)), ((3, 2), inf), ((5, 5), rng.uniform(-1, 1, 25)),
                     ((40, 1), rng.uniform(-1, 1, 40)), ((1, 23), rng.uniform(-1, 1, 23))):
        g = FilterGraph((0, 0, 1, 1))
        g.convolve_matrix(order[0], order[1], k, 1.5, 0.1, edge_mode=edge)
        t, e = _dev(px), px.copy()
        ctx.convolve_matrix(t, g.primitives[0], g.values)
        orc.convolve_matrix(e, g.primitives[0], g.values)
        assert np.array_equal(t.cpu().numpy(), e), order


@pytest.mark.parametrize("sig", [(1.2, 0.7), (0.0, 1.1), (1.4, 0.0)])
@pytest.mark.parametrize("shape", [(38, 125), (5, 3)])
def test_small_blur_of_a_shared_image(ctx, sig, shape):
    # the IIR blur reads the layer, or a result that is used again, and writes its own image
    h, w = shape
    g = FilterGraph((0, 0, w, h))
    a = g.gaussian_blur(*sig, cs=abi.CI_SRGB)
    b = g.gaussian_blur(*sig, in1=a, cs=abi.CI_SRGB)
    g.merge([a, b, SOURCE_GRAPHIC], cs=abi.CI_SRGB)
    layer = _random(h, w, 5, 0.3)
    t, e = _dev(layer), layer.copy()
    ts = abi.Transform(1.0, 0.0, 0.0, 1.0, 0.0, 0.0)
    assert ctx.filter_apply(g, ts, t) == orc.filter_apply(g, ts, e)
    assert np.array_equal(t.cpu().numpy(), e)
