"""Waves with none, one, two, several and 64 clipped triangles, side by side and
alone, against the oracle, bit for bit; slots past the reserved ones; and what a
wave full of clipped triangles costs against one with a single one."""
import numpy as np
import pytest

from test_gpu_setup_waves import _check

pytestmark = pytest.mark.gpu


def _clipped(n, counts, seed, samples_log2=1, size=(120, 104)):
    """n triangles, the first counts[w % len(counts)] of each 64 to be clipped."""
    from cudaraster import scenes
    sc = scenes.random_tris(n, *size, samples_log2=samples_log2, seed=seed)
    cl = scenes.clip_mix(n, *size, samples_log2=samples_log2, seed=seed + 1)
    t = np.arange(n)
    m = t % 64 < np.asarray(counts)[t // 64 % len(counts)]
    v = sc.vertices.reshape(n, 3, -1).copy()
    v[m] = cl.vertices.reshape(n, 3, -1)[m]
    sc.vertices = np.ascontiguousarray(v.reshape(3 * n, -1))
    return sc


@pytest.mark.parametrize("counts", [(1,), (2,), (3,), (64,), (0, 1, 2, 64, 5, 0, 63)])
@pytest.mark.parametrize("tris", [64, 127, 1500])
def test_clipped_per_wave(counts, tris):
    _check(_clipped(tris, counts, seed=sum(counts) + tris))


def test_slots_past_the_reserved_ones():
    """More subtriangles than there are slots: the draw runs again with more."""
    import cudaraster
    import oracle
    sc = _clipped(12000, (64, 1, 2), seed=9, samples_log2=0)
    ref = oracle.render(sc)
    br = cudaraster.BatchRenderer([sc])
    try:
        br.batch.reserve(0, 1, 1 << 20, 1 << 20)              # a slot per triangle and none for the others
        br.draw()
        got = br.read(0)
        assert br.batch.info()["retries"] >= 1 and br.batch.view_counters(0)["num_subtris"] > sc.num_tris
    finally:
        br.close()
    for k in ("depth", "triid", "color"):
        assert np.array_equal(got[k], ref[k]), k


def test_many_clipped_cost_little_more_than_one():
    """One after another, 64 clipped triangles of a wave took 13 times the setup
    time of one (540 against 40 us)."""
    import cudaraster
    from cudaraster import scenes
    times = []
    for per_wave in (1, 64):
        rng = np.random.default_rng(4)
        n = 1024
        t = np.zeros((n, 3, 4), np.float32)
        t[..., 3] = 1.0
        t[:, :, :2] = rng.uniform(-0.9, 0.9, (n, 1, 2))
        t[:, 1, 0] += 0.02
        t[:, 2, 1] += 0.02
        t[np.arange(n) % 64 < per_wave, 0, 2] = -1.3          # a corner before the near plane
        sc = scenes.Scene("clipped", 1024, 1024, 0, scenes.FLAG_DEPTH, scenes.BLEND_REPLACE, scenes.SHADER_CONSTANT,
                          t.reshape(-1, 4), np.arange(3 * n, dtype=np.int32).reshape(n, 3))
        r = cudaraster.SceneRenderer(sc, triangle_ids=False)
        try:
            s = []
            for _ in range(20):
                r.draw(clear=True)
                s.append(r.cr.getStats()["setupTime"])
            times.append(sorted(s)[10])
        finally:
            r.close()
    assert times[1] < 4.0 * times[0], times
