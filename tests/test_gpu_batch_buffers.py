"""Batch.set_buffers: views pointed at other vertex and index buffers draw
what plain draws of those buffers draw, through the graph and without it, in
one group and in several, and for more views than one launch can update."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scenes(n, seed, tris, size):
    from cudaraster import scenes
    return [scenes.random_tris(tris, size, size, samples_log2=(k % 2) * 2, seed=seed + k) for k in range(n)]


def _plain(scene):
    import cudaraster
    r = cudaraster.SceneRenderer(scene)
    try:
        r.draw(clear=True)
        return r.read()
    finally:
        r.close()


@pytest.mark.parametrize("views,tris,size,groups,graph", [(3, 700, 72, 1, True), (3, 700, 72, 2, True),
                                                         (5, 300, 40, 4, False), (131, 20, 16, 2, True)])
def test_set_buffers(views, tris, size, groups, graph):
    import cudaraster
    sets = [_scenes(views, 100 * k, tris, size) for k in range(2)]
    buffers = [[cudaraster.device_buffers(sc) for sc in s] for s in sets]
    br = cudaraster.BatchRenderer(sets[0])
    try:
        br.batch.configure(view_groups=groups)
        br.batch.use_graph(graph)
        look = range(views) if views < 10 else (0, 63, 127, 128, views - 1)
        want = [[_plain(s[i]) for i in look] for s in sets]
        for k in (0, 1, 1, 0):
            br.batch.set_buffers([v.data_ptr() for v, _ in buffers[k]], [t.data_ptr() for _, t in buffers[k]])
            br.draw()
            for i, w in zip(look, want[k]):
                got = br.read(i)
                assert all(np.array_equal(got[c], w[c]) for c in w), (k, i)
    finally:
        br.close()


def test_set_buffers_refuses_bad_pointers():
    import cudaraster
    br = cudaraster.BatchRenderer(_scenes(2, 7, 50, 24))
    try:
        br.draw()
        want = br.read(1)
        v, t = ([b[k].data_ptr() for b in br.buffers] for k in (0, 1))
        for bad in (([v[0], v[1] + 4], t), ([v[0], None], t), (v, [t[0], t[1] + 2]), (v[:1], t[:1])):
            with pytest.raises(cudaraster.CrError):
                br.batch.set_buffers(*bad)
        br.draw()
        got = br.read(1)
        assert all(np.array_equal(got[c], want[c]) for c in want)
    finally:
        br.close()
