"""The backward pass's sums over a tile: shared and repeated vertices, ids and
indices out of range, images at and around the tile size, channel counts at
and around the staged block, against the FP64 reference tile by tile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILE = 16


def _case(seed, width, height, channels, tris, spread):
    """Random ids over a mesh whose vertex indices are `spread` apart, with
    ids past the triangle count, vertices past the vertex count, and
    triangles that use a vertex twice."""
    rng = np.random.default_rng(seed)
    used = max(3, tris // 2)
    V = (used - 1) * spread + 1
    w = rng.uniform(1.0, 3.0, V)
    pos = np.stack([rng.uniform(-1, 1, V) * w, rng.uniform(-1, 1, V) * w, rng.uniform(-1, 1, V) * w, w], -1)
    tri = rng.integers(0, used, (tris, 3)) * spread
    tri[rng.random(tris) < 0.1, 1] = V + 7
    twice = rng.random(tris) < 0.1
    tri[twice, 2] = tri[twice, 0]
    # Neighbouring pixels mostly see one triangle.
    ids = rng.integers(-1, tris + 3, (height // 3 + 1, width // 3 + 1)).repeat(3, 0).repeat(3, 1)[:height, :width]
    noise = rng.random(ids.shape) < 0.2
    ids = np.where(noise, rng.integers(-1, tris + 3, ids.shape), ids)
    return (pos.astype(np.float32), rng.uniform(-1, 1, (V, channels)).astype(np.float32), tri.astype(np.int32),
            np.ascontiguousarray(ids, dtype=np.int32), rng.normal(size=(height, width, channels)).astype(np.float32))


def _reference(pos, attr, tri, ids, g):
    """FP64 gradients, and per value the bound on their FP32 summation: every
    tile's sum is rounded once and added with one rounding, each at most 2^-24
    of the sums' magnitudes so far."""
    import diff_ref
    seen = (ids >= 0) & (ids < len(tri))
    seen[seen] = (tri[ids[seen]] < len(pos)).all(1)
    ids = np.where(seen, ids, -1).astype(np.int64)
    safe = np.minimum(tri, len(pos) - 1)
    total = [np.zeros((len(pos), 4)), np.zeros(attr.shape, np.float64)]
    size = [np.zeros_like(t) for t in total]
    tiles = 0
    for y in range(0, ids.shape[0], TILE):
        for x in range(0, ids.shape[1], TILE):
            part = np.full_like(ids, -1)
            part[y:y + TILE, x:x + TILE] = ids[y:y + TILE, x:x + TILE]
            tiles += 1
            for k, v in enumerate(diff_ref.backward(pos, attr, safe, part, g)):
                total[k] += v
                size[k] += np.abs(v)
    return total, [2 * tiles * 2.0 ** -24 * s + 1e-9 * (1 + s.max()) for s in size]


CASES = [(1, 1, 1, 1, 1), (16, 16, 8, 300, 1), (17, 15, 7, 40, 1024), (33, 48, 9, 200, 64), (5, 70, 16, 25, 512),
         (48, 48, 3, 5000, 3), (40, 24, 20, 2, 1)]


@pytest.mark.parametrize("deterministic", [False, True])
@pytest.mark.parametrize("width,height,channels,tris,spread", CASES)
def test_tile_sums(width, height, channels, tris, spread, deterministic):
    import torch
    from cudaraster.diff import DiffRasterizer
    case = _case(width + tris, width, height, channels, tris, spread)
    (gp, ga), (bp, ba) = _reference(*case)
    pos, attr, tri, ids, g = (torch.from_numpy(a).cuda() for a in case)
    dr = DiffRasterizer(width, height, deterministic=deterministic)
    try:
        runs = []
        for _ in range(2):
            p, a = pos.clone().requires_grad_(True), attr.clone().requires_grad_(True)
            dr.render(p, a, tri, ids).backward(g)
            runs.append((p.grad.cpu().numpy(), a.grad.cpu().numpy()))
        for got_p, got_a in runs:
            assert (np.abs(got_p - gp) <= bp).all()
            assert (np.abs(got_a - ga) <= ba).all()
        if deterministic:
            assert all(np.array_equal(u, v) for u, v in zip(*runs))
    finally:
        dr.close()
