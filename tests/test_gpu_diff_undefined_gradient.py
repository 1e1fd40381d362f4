"""A function behind the image that returns no gradient for it: pos and attr get
zeros, from render() and from render_views() alike."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("views", [0, 1, 3])
def test_zeros(views):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cudaraster import scenes
    from cudaraster.diff import DiffRasterizer

    class Dropped(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x.sum()

        @staticmethod
        def backward(ctx, g):
            return None

    vs = scenes.diff_views(max(views, 1), num_tris=300, width=48, height=40, channels=3)
    pos = [torch.from_numpy(v.pos).cuda().requires_grad_(True) for v in vs]
    attr = [torch.from_numpy(v.attr).cuda().requires_grad_(True) for v in vs]
    tris = [torch.from_numpy(v.tris).cuda() for v in vs]
    dr = DiffRasterizer(48, 40)
    try:
        out = dr.render_views(pos, attr, tris)[0] if views else dr.render(pos[0], attr[0], tris[0])
        grads = torch.autograd.grad(Dropped.apply(out), [*pos, *attr])
        for x, g in zip([*pos, *attr], grads):
            assert g is not None and g.shape == x.shape and not g.any()
    finally:
        dr.close()
