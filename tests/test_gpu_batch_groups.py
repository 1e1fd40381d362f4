"""View groups on any stream, through the graph (side by side) and launched
directly (one after the other), with tables rebuilt between the draws: every view
as its plain draw."""
import numpy as np
import pytest

from test_gpu_batch import mixed_views, plain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups", [1, 2, 3, 4])
@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("own_stream", [False, True])
def test_groups_with_rebuilt_tables(groups, graph, own_stream):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import cudaraster
    views = [v for v in mixed_views(12, seed=77) if v.deferred_clear][:7]
    refs = [plain(v) for v in views]
    stream = torch.cuda.Stream() if own_stream else None
    br = cudaraster.BatchRenderer(views)
    try:
        br.batch.use_graph(graph)
        br.batch.configure(4, 0, 256, groups)
        for rep in range(4):
            print(f"{groups} groups, graph {graph}, own stream {own_stream}, draw {rep}", flush=True)
            if rep == 2:                     # other places for every view's queues
                for i, v in enumerate(views):
                    br.batch.reserve(i, v.num_tris + 9000 + 64 * i, 1 << 17, 1 << 18)
            for trio in br.surfaces:
                for s in trio:
                    s.upload(np.full(s.shape, 11 + rep, np.uint32))
            br.draw(stream)
            for i in range(len(views)):
                got = br.read(i)
                assert all(np.array_equal(got[k], refs[i][k]) for k in refs[i]), (rep, i)
        assert br.batch.info()["view_groups"] == groups
    finally:
        br.close()
