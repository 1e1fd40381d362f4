"""Backward over meshes whose rows fall on one another in the tiles' tables of
vertices and triangles: gradients against FP64, and no such width costs a multiple
of its neighbours."""
import numpy as np
import pytest

from test_gpu_diff_tiles import _reference

pytestmark = pytest.mark.gpu


def _mesh(cols, rows, sx, sy):
    """A grid of cols x rows vertices over [-sx, sx] x [-sy, sy], two triangles per cell."""
    x, y = np.meshgrid(np.linspace(-sx, sx, cols), np.linspace(-sy, sy, rows))
    n = cols * rows
    pos = np.stack([x.ravel(), y.ravel(), np.zeros(n), np.ones(n)], -1).astype(np.float32)
    i = np.arange(n).reshape(rows, cols)
    a, b, c, d = i[:-1, :-1].ravel(), i[:-1, 1:].ravel(), i[1:, :-1].ravel(), i[1:, 1:].ravel()
    tri = np.stack([np.stack([a, b, c], -1), np.stack([b, d, c], -1)], 1).reshape(-1, 3).astype(np.int32)
    return pos, tri


@pytest.mark.parametrize("deterministic", [False, True])
@pytest.mark.parametrize("cols", [240, 478, 717, 988, 1000, 1024])
def test_gradients(cols, deterministic):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cudaraster.diff import DiffRasterizer
    W, H, C = 36, 33, 5
    # Half a pixel to a vertex, the mesh wider than the image.
    pos, tri = _mesh(cols, 2 * H, cols / (2 * W), 1.0)
    rng = np.random.default_rng(cols)
    attr = rng.uniform(-1, 1, (len(pos), C)).astype(np.float32)
    g = rng.normal(size=(H, W, C)).astype(np.float32)
    dr = DiffRasterizer(W, H, deterministic=deterministic)
    try:
        p, a = torch.from_numpy(pos).cuda().requires_grad_(True), torch.from_numpy(attr).cuda().requires_grad_(True)
        t = torch.from_numpy(tri).cuda()
        ids = dr.rasterize(p.detach(), t)
        assert int((ids >= 0).sum()) > 0.9 * W * H
        dr.render(p, a, t, ids).backward(torch.from_numpy(g).cuda())
        (gp, ga), (bp, ba) = _reference(pos, attr, tri, ids.cpu().numpy(), g)
        assert (np.abs(p.grad.cpu().numpy() - gp) <= bp).all()
        assert (np.abs(a.grad.cpu().numpy() - ga) <= ba).all()
    finally:
        dr.close()


def test_time():
    """512x512, meshes of 988 columns against 800: with the tables' slots tried one
    after the other 170 against 47 us."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cudaraster.diff import DiffRasterizer
    times = {}
    for cols in (800, 988):
        dr = DiffRasterizer(512, 512)
        try:
            pos, tri = (torch.from_numpy(x).cuda() for x in _mesh(cols, cols, 1.0, 1.0))
            attr = torch.rand(len(pos), 3, device="cuda", requires_grad=True)
            ids = dr.rasterize(pos, tri)
            g = torch.rand(512, 512, 3, device="cuda")
            s = []
            for _ in range(9):
                a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                torch.cuda.synchronize()
                a.record()
                for _ in range(8):
                    dr._interpolate_backward(pos, attr.detach(), tri, ids, g)
                b.record()
                torch.cuda.synchronize()
                s.append(a.elapsed_time(b) / 8)
            times[cols] = sorted(s)[4]
        finally:
            dr.close()
    assert times[988] < 2.0 * times[800], times
