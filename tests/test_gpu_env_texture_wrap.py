"""A surface that emits the environment texture, with texture coordinates outside [0, 1].

Directions map into [0, 1] x [0, 1], a mesh's texture coordinates need not: the texture repeats
there (reference shader_nodes.cpp:1910-1919).  Rays that hit the emitter and light samples on it
must read the texels that the oracle reads."""
import math

import numpy as np
import pytest

from oracle import binding as ob
from tests.test_gpu_render import assert_pixels_match_where_paths_match, render_gpu
from vlr_amd import scenes

pytestmark = pytest.mark.gpu


def emitter_wall(lo, hi, env_size=(8, 4)):
    """A matte floor before a wall that emits the environment texture; the wall's texture
    coordinates run from lo to hi on both axes."""
    mats = [scenes.MaterialDesc(scenes.MATTE, {"albedo": (scenes.REC709, 0.6, 0.5, 0.4)}),
            scenes.MaterialDesc(scenes.ENVIRONMENT_EMITTER, {"emittance": (scenes.REC709, 1.0, 1.0, 1.0)},
                                {"scale": 1.0}, use_env_texture=True)]
    floor = scenes._quad((-2, 0, -2), (-2, 0, 2), (2, 0, 2), (2, 0, -2), (0, 1, 0), (1, 0, 0))
    wall = scenes._quad((-2, 0, -2), (2, 0, -2), (2, 3, -2), (-2, 3, -2), (0, 0, 1), (1, 0, 0))
    wall[:, 9:11] = lo + (hi - lo) * wall[:, 9:11]
    meshes = [scenes.MeshDesc("Floor", floor, [(scenes.quad_indices(1), 0)]),
              scenes.MeshDesc("Wall", wall, [(scenes.quad_indices(1), 1)])]
    tex = np.ones((env_size[1], env_size[0], 4), np.float16)
    tex[..., :3] = np.random.default_rng(5).uniform(0.1, 8.0, (env_size[1], env_size[0], 3))
    cam = scenes.CameraDesc((0.0, 1.2, 5.0), scenes.q_rotate_y(math.pi), 1.0, math.radians(45.0))
    return scenes.SceneDesc(mats, meshes, [scenes.InstanceDesc("Inst", scenes.identity4(), [0, 1])], cam,
                            scenes.EnvDesc(1, tex.view(np.uint16), 0.0), False, "emitter_wall")


@pytest.mark.parametrize("wavefront_depth", [0, 64])
@pytest.mark.parametrize("spectral", [False, True])
@pytest.mark.parametrize("lo,hi", [(-1.5, 2.5), (0.0, 1.0), (-40.0, -38.6)])
def test_texture_repeats_on_a_mesh(torch_gpu, lo, hi, spectral, wavefront_depth):
    W = H = 48
    frames = 4
    desc = emitter_wall(lo, hi)
    imgs, _, rng_gpu = render_gpu(desc, W, H, frames, 4, spectral, wavefront_depth=wavefront_depth)
    ref, _, rng_ref, _ = ob.Scene(desc, spectral=spectral).render(W, H, frames, max_path_length=4,
                                                                  rng_state=ob.seed_states(W, H))
    assert np.mean(rng_gpu == rng_ref) > 0.97
    assert_pixels_match_where_paths_match(imgs[-1][..., :3], ref, rng_gpu, rng_ref, W, H, 1e-3)
