"""The per-depth kernels' ray queues at the edges of their blocks.

k_shade appends a block's rays with one counter update per queue, from per-wave counts: images of
fewer pixels than a wave, exactly a block, a block and one, and several blocks with a partial last
wave must give the same bits as the tail kernel, which uses no queue after its first."""
import numpy as np
import pytest

from tests.test_gpu_render import render_gpu
from vlr_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(1, 1), (63, 1), (16, 16), (257, 1), (37, 41)])
@pytest.mark.parametrize("spectral", [False, True])
def test_block_appends_keep_every_path(torch_gpu, W, H, spectral):
    desc = scenes.cornell_box()
    imgs, st, rng, acc = render_gpu(desc, W, H, 2, 6, spectral, wavefront_depth=64, want_accum=True)
    imgs0, st0, rng0, acc0 = render_gpu(desc, W, H, 2, 6, spectral, wavefront_depth=0, want_accum=True)
    assert st["closestRays"] == st0["closestRays"] and st["shadowRays"] == st0["shadowRays"]
    assert np.array_equal(rng, rng0)
    assert np.array_equal(np.asarray(acc), np.asarray(acc0))
    assert all(np.array_equal(np.asarray(a), np.asarray(b)) for a, b in zip(imgs, imgs0))
