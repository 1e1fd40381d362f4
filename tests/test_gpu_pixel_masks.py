"""Deferred shading walks each pixel's own records, chosen by a conservative
mask per record: every sample count against the oracle, bit for bit, on the
shapes where such a mask could miss a pixel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(kind, samples_log2, seed):
    from cudaraster import scenes
    rng = np.random.default_rng(seed)
    W = H = 64
    n = 900
    base = rng.uniform(-8, W + 8, (n, 1, 2))
    if kind == "axis":          # horizontal and vertical edges on the 1/16 pixel lattice
        size = rng.integers(1, 64, (n, 2)) / 16.0
        p = np.repeat(np.round(base * 16) / 16, 3, 1)
        p[:, 1, 0] += size[:, 0]
        p[:, 2, 1] += size[:, 1]
    elif kind == "sliver":      # long and thinner than a pixel, any direction
        a = rng.uniform(0, 2 * np.pi, n)
        d = np.stack([np.cos(a), np.sin(a)], -1)
        length, width = rng.uniform(4, 90, (n, 1)), rng.uniform(0.05, 0.9, (n, 1))
        p = np.stack([base[:, 0], base[:, 0] + d * length,
                      base[:, 0] + d * length * 0.5 + d[:, ::-1] * [-1, 1] * width], 1)
    elif kind == "huge":        # edges that cross the viewport far from the vertices
        p = base + rng.uniform(-1, 1, (n, 3, 2)) * 900
    else:                       # "tiny": a pixel or less
        p = base + rng.uniform(-0.8, 0.8, (n, 3, 2))
    area = (p[:, 1, 0] - p[:, 0, 0]) * (p[:, 2, 1] - p[:, 0, 1]) - (p[:, 2, 0] - p[:, 0, 0]) * (p[:, 1, 1] - p[:, 0, 1])
    p = np.where((area < 0)[:, None, None], p[:, ::-1], p)
    w = rng.uniform(1, 20, (n, 3))
    clip = scenes._to_clip(p[..., 0], p[..., 1], w, W, H)
    verts = np.concatenate([clip, rng.random((n, 3, 4))], -1).reshape(-1, 8).astype(np.float32)
    return scenes.Scene(kind, W, H, samples_log2, scenes.FLAG_DEPTH | scenes.FLAG_LERP, scenes.BLEND_REPLACE,
                        scenes.SHADER_GOURAUD, verts, np.arange(3 * n, dtype=np.int32).reshape(n, 3))


@pytest.mark.parametrize("kind", ["axis", "sliver", "huge", "tiny"])
@pytest.mark.parametrize("samples_log2", [0, 1, 2, 3])
@pytest.mark.parametrize("tris", [900, 4])
def test_masked_walk_matches_oracle(kind, samples_log2, tris):
    """tris = 4: batches short enough to be walked without masks, and tiles
    whose texels are stored wide."""
    import cudaraster
    import oracle
    sc = _scene(kind, samples_log2, 17 + samples_log2)
    sc.indices = np.ascontiguousarray(sc.indices[:tris])
    ref = oracle.render(sc)
    r = cudaraster.SceneRenderer(sc)
    try:
        r.draw(clear=True)
        got = r.read()
    finally:
        r.close()
    for k in ("depth", "triid", "color"):
        assert np.array_equal(got[k], ref[k]), k
