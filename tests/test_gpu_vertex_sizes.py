"""The passthrough vertex shader on either side of the size from which its
records bypass the caches: every clip position against the fused FP32 chain in
FP64, the rest of every record untouched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LINE = (64 << 20) // (12 + 48)


@pytest.mark.parametrize("count", [1, 255, 257, LINE - 1, LINE + 2])
def test_records(count):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import cudaraster
    rng = np.random.default_rng(count)
    m = rng.uniform(-2, 2, (4, 4)).astype(np.float32)
    gen = torch.Generator(device="cuda").manual_seed(7)
    p = torch.rand((count, 3), generator=gen, device="cuda") * 4 - 2
    out = torch.full((count, 12), 7.0, device="cuda")
    cr = cudaraster.CudaRaster().init()
    try:
        cr.vertexShaderPassthrough(p, m, out, out_stride=48)
        torch.cuda.synchronize()
    finally:
        cr.close()
    h = torch.cat([p, torch.ones_like(p[:, :1])], 1).double()
    md = torch.from_numpy(m).double().cuda()
    want, size = h @ md.T, h.abs() @ md.abs().T
    # Four fused multiply-adds, each rounded once, at most the terms' size.
    assert bool(((out[:, :4].double() - want).abs() <= 4 * 2.0 ** -24 * size).all())
    assert bool((out[:, 4:] == 7.0).all())
