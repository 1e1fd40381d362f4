"""The autotuner times what later draws run: the captured graph with its parallel
fine branches, not the launches one after the other."""
import pytest

pytestmark = pytest.mark.gpu


def test_tuned_time_is_the_replayed_graphs():
    """8 small views of two pipe variants: 92 us tuned without the branches, 81
    drawn with them."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import cudaraster
    from cudaraster import scenes
    views = scenes.multi_view(8, seed=11, resolutions=(256,), tri_range=(2000, 20000), samples_choices=(0, 2))
    br = cudaraster.BatchRenderer(views)
    try:
        br.batch.autotune()
        tuned = br.batch.info()["tuned_gpu_ms"]
        times = []
        for _ in range(21):
            br.draw()
            times.append(br.batch.info()["last_gpu_ms"])
        assert tuned < 1.08 * sorted(times)[10], (tuned, sorted(times))
    finally:
        br.close()
