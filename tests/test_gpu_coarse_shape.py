"""The plain draw's choice of coarse workgroup: the same images on both sides of
the rule, and never a multiple of the large workgroups' time where a few thousand
triangles reach many bins each."""
import numpy as np
import pytest

from test_gpu_setup_waves import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tris,width,height", [(16, 2040, 2000), (17, 2040, 2000), (127, 200, 120), (128, 200, 120),
                                               (129, 200, 120)])
def test_around_the_rule(tris, width, height):
    from cudaraster import scenes
    _check(scenes.random_tris(tris, width, height, samples_log2=0, seed=tris, area_range=(4.0, 0.3 * width * height)))


def test_many_large_triangles():
    """5000 triangles of half the view's width at 2048x2048: 1523 us in workgroups of
    256 lanes, 703 in those of 1024."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import cudaraster
    from cudaraster import scenes
    rng = np.random.default_rng(6)
    n = 5000
    t = np.zeros((n, 3, 4), np.float32)
    t[..., 3] = 1.0
    t[:, :, :2] = rng.uniform(-1.0, 0.0, (n, 1, 2))
    t[:, 1, 0] += 1.0
    t[:, 2, 1] += 1.0
    t[..., 2] = rng.uniform(-0.9, 0.9, (n, 1))
    sc = scenes.Scene("large", 2048, 2048, 0, scenes.FLAG_DEPTH, scenes.BLEND_REPLACE, scenes.SHADER_CONSTANT,
                      t.reshape(-1, 4), np.arange(3 * n, dtype=np.int32).reshape(n, 3))
    r = cudaraster.SceneRenderer(sc, triangle_ids=False)
    try:
        times = {}
        for threads in (1024, 0):
            r.cr.setDebugParams(coarse_threads=threads)
            s = []
            for _ in range(12):
                r.draw(clear=True)
                s.append(r.cr.getStats()["coarseTime"])
            times[threads] = sorted(s)[6]
        assert times[0] < 1.25 * times[1024], times
    finally:
        r.close()
