"""The forward interpolation over images at and around its 16x16-pixel tile, ids
and indices out of range, channel counts that move one and four at a time:
against FP64 barycentrics."""
import numpy as np
import pytest

from test_gpu_diff_tiles import _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,channels", [(1, 1, 4), (16, 16, 8), (15, 17, 3), (33, 31, 12), (300, 5, 1),
                                                   (5, 300, 4)])
def test_every_pixel(width, height, channels):
    import torch
    from cudaraster.diff import DiffRasterizer
    pos, attr, tri, ids, _ = _case(width, width, height, channels, 60, 3)
    seen = (ids >= 0) & (ids < len(tri))
    seen[seen] = (tri[ids[seen]] < len(pos)).all(1)
    v = np.minimum(tri[np.where(seen, ids, 0)], len(pos) - 1)                    # [h, w, 3]
    p = pos.astype(np.float64)[v]
    qx = ((2.0 * np.arange(width) + 1.0) / width - 1.0)[None, :, None]
    qy = ((2.0 * np.arange(height) + 1.0) / height - 1.0)[:, None, None]
    xs, ys = p[..., 0] - qx * p[..., 3], p[..., 1] - qy * p[..., 3]
    c = np.stack([xs[..., (k + 1) % 3] * ys[..., (k + 2) % 3] - ys[..., (k + 1) % 3] * xs[..., (k + 2) % 3]
                  for k in range(3)], -1)
    total = c.sum(-1, keepdims=True)
    scale = np.abs(c).sum(-1, keepdims=True)
    # Near-degenerate projections (one triangle in ten repeats a vertex): the
    # barycentrics' FP64 rounding is not the subject here.
    sure = ~seen | (np.abs(total) > 1e-6 * scale)[..., 0]
    b = c / np.where(total == 0.0, 1.0, total)
    a = attr.astype(np.float64)[v]
    want = np.where(seen[..., None], (b[..., None] * a).sum(-2), 0.0)
    # One rounding to FP32, and FP64 roundings that the barycentrics' size and
    # the cancellation in their sum scale.
    bound = 2.0 ** -23 * np.abs(want) + 1e-14 * (np.abs(b[..., None] * a).sum(-2) *
                                                 (scale / np.maximum(np.abs(total), 1e-300)) + 1.0)
    dr = DiffRasterizer(width, height)
    try:
        got = dr.render(*(torch.from_numpy(t).cuda() for t in (pos, attr, tri)),
                        tri_image=torch.from_numpy(ids).cuda()).cpu().numpy()
    finally:
        dr.close()
    assert got.shape == (height, width, channels)
    assert (np.abs(got - want) <= bound)[sure].all()
