"""Replays of a batch's graph in the configurations that the tuner does not
always choose: three and four view groups, banded placement, two and eight tiles
per group, 1024 coarse lanes.  The first draw is launched; every later one is a
replay, over surfaces overwritten before it."""
import numpy as np
import pytest

from test_gpu_batch import mixed_views, plain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [(2, 1, 1024, 1), (8, 0, 256, 2), (4, 1, 256, 4), (4, 0, 1024, 3), (8, 1, 1024, 4),
                                 (2, 0, 256, 3)])
def test_replays(cfg):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import cudaraster
    views = [v for v in mixed_views(12, seed=12) if v.deferred_clear][:9]
    refs = [plain(v) for v in views]
    br = cudaraster.BatchRenderer(views)
    try:
        br.batch.configure(*cfg)
        br.batch.use_graph(True)
        for draw in range(4):
            for trio in br.surfaces:
                for s in trio:
                    s.upload(np.full(s.shape, 0x51 + draw, np.uint32))
            br.draw()
            x = torch.ones(1 << 20, device="cuda")
            assert float((x * 2).sum()) == 2.0 * (1 << 20)
            info = br.batch.info()
            assert info["uses_graph"] == 1 and info["retries"] == 0
            assert (info["fine_tiles_per_group"], info["fine_banded"], info["coarse_threads"],
                    info["view_groups"]) == cfg
            for i in range(len(views)):
                got = br.read(i)
                for k in ("color", "depth", "triid"):
                    assert np.array_equal(got[k], refs[i][k]), f"{cfg}, draw {draw}: view {i} {k}"
    finally:
        br.close()
