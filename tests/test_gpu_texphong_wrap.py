"""Texture coordinates around the whole textures at which the texel index
changes from the addition to the division, and beyond the range in which an
index exists: against the oracle, colour within 1 LSB per channel."""
import numpy as np
import pytest

from test_gpu_parity import assert_parity, render_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("samples_log2", [0, 3])
@pytest.mark.parametrize("offset", [-2.0, -1.0, 0.0, 1.0, 2.0, 300.0, 1e10])
def test_tex_phong_coordinate_range(oracle_lib, offset, samples_log2):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cudaraster import scenes
    sc = scenes.tex_phong(2000, 136, 104, samples_log2=samples_log2, seed=120, quads=True, tex_scale=(0.5, 1.0))
    uv = sc.vertices[:, 12:14]
    uv -= np.floor(uv.min(axis=0))
    uv *= 0.25
    uv += np.float32(offset)
    print(f"texPhong offset={offset} s={samples_log2}", flush=True)
    assert_parity(render_gpu(sc), oracle_lib.render(sc), f"texPhong offset {offset}")
