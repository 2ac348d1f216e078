"""PNG rows where the kernel's cases change: rows past the LDS width, every channel value
at every alpha (also above it) and smooth rows on which each filter type wins, byte for
byte against the oracle."""
import numpy as np
import pytest

from oracle import bindings as orc

pytestmark = pytest.mark.gpu


def _rows(ctx, px):
    import torch
    h, w = px.shape[:2]
    out = torch.full((h * (4 * w + 1),), 77, dtype=torch.uint8, device="cuda")
    ctx.png_filter_rows(torch.from_numpy(np.ascontiguousarray(px)).cuda(), out)
    ctx.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("w", [2, 63, 64, 65, 4095, 4097, 5001])
def test_widths(ctx, w):
    px = np.random.default_rng(w).integers(0, 256, (4, w, 4)).astype(np.uint8)
    assert np.array_equal(_rows(ctx, px), orc.png_filter_rows(px))


def test_every_channel_at_every_alpha(ctx):
    a, c = np.meshgrid(np.arange(256), np.arange(256), indexing="ij")
    px = np.stack([c, 255 - c, (c * 7) % 256, a], -1).astype(np.uint8)
    assert np.array_equal(_rows(ctx, px), orc.png_filter_rows(px))


def test_smooth_rows_of_every_filter(ctx):
    y, x = np.mgrid[0:200, 0:300].astype(np.float64)
    rng = np.random.default_rng(1)
    bands = [np.full_like(x, 9.0), x * 0.9, y * 1.2, (x + y) * 0.5, 60 * np.sin(x / 9) + 60 * np.sin(y / 7) + 120,
             rng.integers(0, 5, x.shape).astype(np.float64)]
    px = np.zeros((200, 300, 4), np.uint8)
    for k, f in enumerate(bands):  # a band of rows for each pattern, opaque
        px[k * 33:(k + 1) * 33, :, :3] = (np.clip(f, 0, 255)[k * 33:(k + 1) * 33, :, None] * [1.0, 0.8, 0.6])
    px[..., 3] = 255
    got = _rows(ctx, px)
    assert np.array_equal(got, orc.png_filter_rows(px))
    assert len(set(got.reshape(200, -1)[:, 0].tolist())) >= 4
