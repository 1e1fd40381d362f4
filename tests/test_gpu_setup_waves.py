"""Triangle setup's wave-wide paths against the oracle, bit for bit: clipping
(every triangle of a wave, some, one; polygons of up to nine vertices; counts
around the wave and the workgroup's chunk) and boxes of many bins."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(sc, ids=True):
    import cudaraster
    import oracle
    ref = oracle.render(sc)
    r = cudaraster.SceneRenderer(sc)
    try:
        r.draw(clear=True)
        got = r.read()
    finally:
        r.close()
    for k in ("depth", "triid", "color"):
        assert np.array_equal(got[k], ref[k]), k


@pytest.mark.parametrize("tris", [1, 63, 64, 65, 1023, 1024, 1025, 2500])
@pytest.mark.parametrize("samples_log2", [0, 3])
def test_clipped_triangles(tris, samples_log2):
    from cudaraster import scenes
    _check(scenes.clip_mix(tris, 120, 104, samples_log2=samples_log2, seed=tris + samples_log2))


@pytest.mark.parametrize("every", [2, 17, 300])
def test_clipped_between_unclipped(every):
    """One clipped triangle in `every`: waves with one and without any."""
    from cudaraster import scenes
    sc = scenes.random_tris(1500, 120, 104, samples_log2=1, seed=every)
    cl = scenes.clip_mix(1500, 120, 104, samples_log2=1, seed=every + 1)
    v = sc.vertices.reshape(1500, 3, -1).copy()
    v[::every] = cl.vertices.reshape(1500, 3, -1)[::every]
    sc.vertices = np.ascontiguousarray(v.reshape(4500, -1))
    _check(sc)


def test_frustum_corners():
    """Triangles around the whole frustum, cut by all six planes."""
    from cudaraster import scenes
    rng = np.random.default_rng(8)
    n = 400
    ang = rng.uniform(0, 2 * np.pi, (n, 1)) + np.array([0.0, 2.1, 4.2])
    r = rng.uniform(1.2, 4.0, (n, 3))
    w = rng.uniform(0.5, 2.0, (n, 3))
    clip = np.stack([r * np.cos(ang) * w, r * np.sin(ang) * w, rng.uniform(-1.6, 1.6, (n, 3)) * w, w], -1)
    verts = np.concatenate([clip, rng.random((n, 3, 4))], -1).reshape(-1, 8).astype(np.float32)
    _check(scenes.Scene("corners", 200, 136, 2, scenes.FLAG_DEPTH | scenes.FLAG_LERP, scenes.BLEND_REPLACE,
                        scenes.SHADER_GOURAUD, verts, np.arange(3 * n, dtype=np.int32).reshape(n, 3)))


@pytest.mark.parametrize("width,height", [(136, 2040), (2040, 136), (1000, 900)])
def test_boxes_of_many_bins(width, height):
    """From one bin to all of them, around the size at which a wave takes over."""
    from cudaraster import scenes
    sc = scenes.random_tris(1100, width, height, samples_log2=0, seed=width, area_range=(20.0, 0.5 * width * height))
    _check(sc)
