"""The forward interpolation's two workgroup shapes, chosen by triangles per pixel:
triangles that no pixel shows change the shape and not a bit of the image; and
large triangles with many channels take the shape of longer stores."""
import numpy as np
import pytest

from test_gpu_diff_tiles import _case

pytestmark = pytest.mark.gpu


def _more(tri, pixels):
    return np.concatenate([tri, np.tile(tri[:1], (pixels, 1))])


@pytest.mark.parametrize("width,height", [(1, 1), (31, 7), (32, 8), (33, 9), (255, 2), (256, 1), (257, 17), (64, 300)])
@pytest.mark.parametrize("channels", [1, 4, 5, 24])
def test_same_bits(width, height, channels):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cudaraster.diff import DiffRasterizer
    few = max(1, width * height // 8)
    pos, attr, tri, ids, _ = _case(width + channels, width, height, channels, few, 2)
    ids = np.where(ids < few, ids, -1).astype(np.int32)
    dr = DiffRasterizer(width, height)
    try:
        p, a, i = (torch.from_numpy(x).cuda() for x in (pos, attr, ids))
        rows, tiles = (dr.render(p, a, torch.from_numpy(t).cuda(), tri_image=i).cpu().numpy()
                       for t in (tri, _more(tri, width * height)))
    finally:
        dr.close()
    assert np.array_equal(rows.view(np.uint32), tiles.view(np.uint32))


def test_large_triangles_in_rows():
    """1024x1024, 8k triangles, 24 channels: 62 us in 16 x 16 pixels, 45 in rows."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cudaraster.diff import DiffRasterizer
    from test_gpu_diff_mesh_widths import _mesh
    S, C = 1024, 24
    pos, tri = _mesh(65, 65, 1.0, 1.0)
    dr = DiffRasterizer(S, S)
    try:
        p = torch.from_numpy(pos).cuda()
        attr, out = torch.rand(len(pos), C, device="cuda"), torch.empty(S, S, C, device="cuda")
        ids = dr.rasterize(p, torch.from_numpy(tri).cuda())
        times = []
        for t in (tri, _more(tri, S * S // 4)):
            t = torch.from_numpy(t).cuda()
            s = []
            for _ in range(11):
                a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                torch.cuda.synchronize()
                a.record()
                for _ in range(20):
                    dr._interpolate_ids(p, attr, t, out, ids)
                b.record()
                torch.cuda.synchronize()
                s.append(a.elapsed_time(b))
            times.append(sorted(s)[5])
    finally:
        dr.close()
    assert times[0] < 0.93 * times[1], times
