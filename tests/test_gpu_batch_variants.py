"""Fine stages of several pipe variants, one after the other in a batch's first
draw and side by side in the later ones' graph: every draw against the plain
draws of the same views."""
import numpy as np
import pytest

from test_gpu_batch import mixed_views, plain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("num_views,groups", [(1, 1), (2, 1), (9, 1), (14, 1), (10, 2)])
def test_every_draw_of_a_batch(num_views, groups):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import cudaraster
    views = [v for v in mixed_views(2 * num_views, seed=31) if v.deferred_clear][:num_views]
    refs = [plain(v) for v in views]
    br = cudaraster.BatchRenderer(views)
    try:
        br.batch.configure(4, 0, 256, groups)
        for rep in range(4):
            print(f"{len(views)} views, draw {rep}", flush=True)
            br.draw()
            x = torch.ones(1 << 20, device="cuda")
            assert float((x * 2).sum()) == 2.0 * (1 << 20)
            for i in range(len(views)):
                got = br.read(i)
                for k in ("color", "depth", "triid"):
                    assert np.array_equal(got[k], refs[i][k]), f"draw {rep}: view {i} {k}"
    finally:
        br.close()
