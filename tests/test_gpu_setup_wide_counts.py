"""Boxes of several bins in some of a wave's lanes: images against the oracle
around the rule by which the wave walks them together, and the time of a few such
lanes against that of a whole wave of them."""
import numpy as np
import pytest

from test_gpu_setup_waves import _check

pytestmark = pytest.mark.gpu


def _mixed(n, w, h, per_wave, bw, bh, seed):
    """Right triangles of 6 x 6 pixels, the first per_wave of each 64 of bw x bh."""
    from cudaraster import scenes
    r = np.random.default_rng(seed)
    big = np.arange(n) % 64 < per_wave
    bw, bh = np.where(big, bw, 6.0), np.where(big, bh, 6.0)
    x, y = r.random(n) * (w - bw), r.random(n) * (h - bh)
    t = np.zeros((n, 3, 8), np.float32)
    t[:, 0, 0], t[:, 1, 0], t[:, 2, 0] = x, x + bw, x
    t[:, 0, 1], t[:, 1, 1], t[:, 2, 1] = y, y, y + bh
    t[..., 0], t[..., 1] = t[..., 0] / w * 2 - 1, t[..., 1] / h * 2 - 1
    t[..., 2] = r.uniform(-0.9, 0.9, (n, 1))
    t[..., 3] = 1.0
    t[..., 4:] = r.random((n, 3, 4))
    return scenes.Scene("wide", w, h, 0, scenes.FLAG_DEPTH | scenes.FLAG_LERP, scenes.BLEND_REPLACE,
                        scenes.SHADER_GOURAUD, t.reshape(-1, 8), np.arange(3 * n, dtype=np.int32).reshape(n, 3))


@pytest.mark.parametrize("bins", [3, 4, 6, 15])
@pytest.mark.parametrize("per_wave", [1, 2, 4, 31, 33, 64])
def test_some_wide_boxes(bins, per_wave):
    # 256x256: 16x16 bins of 16 pixels
    _check(_mixed(200, 256, 256, per_wave, 16.0 * bins - 8, 16.0 * bins - 8, seed=bins + per_wave))


def test_some_wide_boxes_cost_no_more_than_all():
    """1024 triangles, 36 of each 64 over 8 to 12 bins: 33 us of setup with the boxes one
    after another, 16.5 with all 64."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import cudaraster
    times = []
    for per_wave in (36, 64):
        r = cudaraster.SceneRenderer(_mixed(1024, 2048, 2048, per_wave, 250.0, 400.0, seed=3), triangle_ids=False)
        try:
            s = []
            for _ in range(20):
                r.draw(clear=True)
                s.append(r.cr.getStats()["setupTime"])
            times.append(sorted(s)[10])
        finally:
            r.close()
    assert times[0] < 1.35 * times[1], times
