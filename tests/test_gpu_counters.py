"""The counter block is handed to the host and cleared at the end of every
draw: draws that follow one another in any mixture of entry points, contexts
and graph replays start from cleared counters and report their own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _renderer(seed, tris=3000, clip=False):
    import cudaraster
    from cudaraster import scenes
    if clip:   # clipped triangles take slots past the triangle count
        return cudaraster.SceneRenderer(scenes.clip_mix(tris, 200, 120, samples_log2=1, seed=seed))
    return cudaraster.SceneRenderer(scenes.random_tris(tris, 200, 120, samples_log2=1, seed=seed))


@pytest.mark.parametrize("clip", [False, True])
def test_counters_of_consecutive_draws(clip):
    """Plain, asynchronous, no-allocation and profiling draws in turn: each
    reports the counters of the first plain draw and draws its frame."""
    import cudaraster
    r = _renderer(3, clip=clip)
    try:
        sc = r.scene
        r.draw(clear=True)
        want, counters = r.read(), r.cr.getCounters()
        assert counters["num_subtris"] >= sc.num_tris and (counters["num_subtris"] > sc.num_tris) == clip
        for name in ("plain", "async", "noalloc", "profiling", "plain", "async"):
            r.cr.setDebugParams(profiling_mode=cudaraster.PROFILING_COUNTERS if name == "profiling" else 0)
            r.cr.deferredClear(sc.clear_color, sc.clear_depth)
            if name == "async":
                r.cr.drawTrianglesAsync()
                stats = r.cr.getStats()              # waits for the draw
                assert r.cr.drawCheck() == cudaraster.CR_OK
            elif name == "noalloc":
                r.cr.drawTrianglesNoAlloc()
                stats = r.cr.getStats()
            else:
                r.cr.drawTriangles()
                stats = r.cr.getStats()
            got = r.cr.getCounters()
            for k in ("num_tris", "num_subtris", "bin_entries", "tile_list_entries"):
                assert got[k] == counters[k], (name, k)
            assert all(0.0 < stats[k] < 1.0 for k in ("setupTime", "coarseTime", "fineTime")), (name, stats)
            frame = r.read()
            assert all(np.array_equal(frame[k], want[k]) for k in want), name
    finally:
        r.close()


def test_captured_draw_replays_between_other_draws():
    """An asynchronous draw captured in a graph: every replay equals the eager
    frame, with another context's draws between the replays."""
    import torch
    a, b = _renderer(4), _renderer(5, clip=True)
    try:
        sc = a.scene
        a.draw(clear=True)
        want = a.read()
        g = torch.cuda.CUDAGraph()
        side = torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=side):
            a.cr.deferredClear(sc.clear_color, sc.clear_depth)
            a.cr.drawTrianglesAsync(torch.cuda.current_stream())
        for rep in range(4):
            for s in (a.color, a.depth, a.triid):
                s.upload(np.full(s.shape, 7 + rep, np.uint32))
            b.draw(clear=True)
            g.replay()
            torch.cuda.synchronize()
            got = a.read()
            assert all(np.array_equal(got[k], want[k]) for k in want), rep
        del g
    finally:
        a.close()
        b.close()
