"""A batch draw on a capturing stream is refused and changes nothing: the capture
goes on, and the batch's next draw starts from cleared counters and reads the
buffers set before the refusal."""
import numpy as np
import pytest

from test_gpu_batch import plain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("drawn", [0, 1, 3])
@pytest.mark.parametrize("tune", [False, True])
def test_refused_under_capture(drawn, tune):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import cudaraster
    from cudaraster import scenes
    sets = [[scenes.random_tris(900, 96, 72, samples_log2=2 * (k % 2), seed=50 * s + k) for k in range(3)]
            for s in range(2)]
    buffers = [cudaraster.device_buffers(sc) for sc in sets[1]]
    want = [plain(sc) for sc in sets[1]]
    br = cudaraster.BatchRenderer(sets[0])
    try:
        for _ in range(drawn):
            br.draw()
        br.batch.set_buffers([v.data_ptr() for v, _ in buffers], [t.data_ptr() for _, t in buffers])
        x = torch.zeros(64, device="cuda")
        g = torch.cuda.CUDAGraph()
        side = torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=side, capture_error_mode="relaxed"):
            x.add_(1.0)
            with pytest.raises(cudaraster.CrError):
                (br.batch.autotune if tune else br.draw)(torch.cuda.current_stream())
        for rep in range(3):
            g.replay()
            torch.cuda.synchronize()
            assert float(x.sum()) == 64.0 * (rep + 1)
            br.draw()
            for i in range(3):
                got = br.read(i)
                assert all(np.array_equal(got[k], want[i][k]) for k in want[i]), (rep, i)
        del g
    finally:
        br.close()
