"""getStats is about its own draw: it does not wait for other work, can be called
while a stream captures, keeps to the last draw around captured ones, and its fine
time covers every tile of a workgroup."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STAGES = ("setupTime", "coarseTime", "fineTime")


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _renderer(tris=3000, seed=3):
    import cudaraster
    from cudaraster import scenes
    return cudaraster.SceneRenderer(scenes.random_tris(tris, 200, 120, samples_log2=1, seed=seed))


def test_does_not_wait_for_other_work():
    torch = _torch()
    side = torch.cuda.Stream()
    r = _renderer()
    try:
        for _ in range(2):
            r.draw(clear=True, stream=side)
            r.cr.getStats()
        a = torch.rand(8192, 8192, device="cuda")
        a @ a
        torch.cuda.synchronize()
        r.draw(clear=True, stream=side)
        for _ in range(30):                  # some 100 ms on the default stream
            a = a @ a
            a = a / a.abs().amax()
        assert not torch.cuda.default_stream().query()
        stats = r.cr.getStats()
        assert not torch.cuda.default_stream().query()
        assert all(stats[k] > 0.0 for k in STAGES), stats
        torch.cuda.synchronize()
    finally:
        r.close()


@pytest.mark.parametrize("mode", ["global", "thread_local", "relaxed"])
@pytest.mark.parametrize("asked_before", [False, True])
def test_while_a_stream_captures(mode, asked_before):
    torch = _torch()
    r = _renderer()
    try:
        r.draw(clear=True)
        if asked_before:
            want = r.cr.getStats()
        x = torch.zeros(64, device="cuda")
        g = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=torch.cuda.Stream(), capture_error_mode=mode):
            x.add_(1.0)
            stats = r.cr.getStats()
        assert all(0.0 < stats[k] < 1.0 for k in STAGES), stats
        assert not asked_before or stats == want
        for rep in range(2):
            g.replay()
            torch.cuda.synchronize()
            assert float(x.sum()) == 64.0 * (rep + 1)
        del g
    finally:
        r.close()


def test_around_captured_draws():
    """The last eager draw's times after a capture, and whole times after replays."""
    torch = _torch()
    r = _renderer()
    try:
        sc = r.scene
        for _ in range(3):
            r.draw(clear=True)
        want = r.cr.getStats()
        g = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=torch.cuda.Stream()):
            r.cr.deferredClear(sc.clear_color, sc.clear_depth)
            r.cr.drawTrianglesAsync(torch.cuda.current_stream())
        assert r.cr.getStats() == want
        for _ in range(3):
            g.replay()
            torch.cuda.synchronize()
            stats = r.cr.getStats()
            assert all(0.0 < stats[k] < 0.01 for k in STAGES), stats
            r.draw(clear=True)
            stats = r.cr.getStats()
            assert all(0.0 < stats[k] < 0.01 for k in STAGES), stats
        del g
    finally:
        r.close()


@pytest.mark.parametrize("clear", [True, False])
def test_fine_time_covers_every_tile(clear):
    """Four tiles, one workgroup: the same long list in its first and in its last
    tile takes the same time."""
    _torch()
    import cudaraster
    from cudaraster import scenes
    times = []
    for tile in (0, 3):
        n = 4000
        rng = np.random.default_rng(2)
        t = np.zeros((n, 3, 8), np.float32)
        t[:, 0, :2], t[:, 1, :2], t[:, 2, :2] = (1.0, 1.0), (7.0, 1.0), (1.0, 7.0)
        t[..., 0] = (t[..., 0] + 8.0 * tile) / 32.0 * 2.0 - 1.0
        t[..., 1] = t[..., 1] / 8.0 * 2.0 - 1.0
        t[..., 2] = np.linspace(0.9, -0.9, n, dtype=np.float32)[:, None]       # every one in front of the last
        t[..., 3] = 1.0
        t[..., 4:] = rng.random((n, 3, 4))
        sc = scenes.Scene("deep", 32, 8, 0, scenes.FLAG_DEPTH | scenes.FLAG_LERP, scenes.BLEND_SRCOVER,
                          scenes.SHADER_GOURAUD, t.reshape(-1, 8), np.arange(3 * n, dtype=np.int32).reshape(n, 3))
        r = cudaraster.SceneRenderer(sc)
        try:
            s = []
            for k in range(15):
                if not clear:                # (without a clear a tile without entries ends at once)
                    r.depth.upload(np.full(r.depth.shape, 0xFFFFFFFF, np.uint32))
                r.draw(clear=clear)
                s.append(r.cr.getStats()["fineTime"])
            times.append(sorted(s)[7])
        finally:
            r.close()
    assert 0.7 < times[1] / times[0] < 1.4, times
