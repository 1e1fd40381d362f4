"""Waves with few, half and all of their triangles over many bins, below and
above the count from which every lane walks its own box: against the oracle, bit
for bit."""
import numpy as np
import pytest

from test_gpu_setup_waves import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wide", [16, 35, 36, 37, 64, 130])
@pytest.mark.parametrize("every", [1, 2])
def test_wide_boxes(wide, every):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cudaraster import scenes
    n = max(wide * every, 200)
    sc = scenes.random_tris(n, 368, 145, samples_log2=1, seed=wide + every)
    big = scenes.random_tris(n, 368, 145, samples_log2=1, seed=wide + 7, area_range=(20000.0, 50000.0))
    v = sc.vertices.reshape(n, 3, -1).copy()
    v[:wide * every:every] = big.vertices.reshape(n, 3, -1)[:wide * every:every]
    sc.vertices = np.ascontiguousarray(v.reshape(3 * n, -1))
    _check(sc)
