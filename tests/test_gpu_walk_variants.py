"""The instantiations of the traversal and of the tail kernel, against each other and the oracle.

Two walks visit the same nodes in the same order with their stacks laid out differently; the tail
kernel takes one by the scene's size and node programs, with or without the radiance cache, and
the per-depth kernels always take the other.  An entry lost in one of them, or one variant's
shading, would show as a difference between schedules that must give the same bits."""
import numpy as np
import pytest

from oracle import binding as ob
from oracle import shader_nodes as osn
from tests.test_gpu_batch import run_batch, single
from tests.test_gpu_render import assert_pixels_match_where_paths_match, render_gpu
from tests.test_gpu_trace import degenerate_scene
from vlr_amd import api, scenes

pytestmark = pytest.mark.gpu


def lit_degenerate_scene(n):
    """The degenerate planes of test_gpu_trace seen from the side where a ray meets the deepest part
    of their tree first, over a floor and under an environment: the camera's rays stack up to 58
    entries, the floor's shadow rays up to 64, of which 16 (per-depth kernels: 12) lie in LDS."""
    desc = degenerate_scene("geometric", n)
    desc.materials.append(scenes.MaterialDesc(scenes.ENVIRONMENT_EMITTER, {"emittance": (scenes.REC709, 1.0, 1.0, 1.0)},
                                              {"scale": 1.0}, use_env_texture=True))
    floor = scenes._quad((-2, -0.6, -2), (-2, -0.6, 2), (2, -0.6, 2), (2, -0.6, -2), (0, 1, 0), (1, 0, 0))
    desc.meshes.append(scenes.MeshDesc("Floor", floor, [(scenes.quad_indices(1), 0)]))
    desc.instances.append(scenes.InstanceDesc("FloorInst", scenes.identity4(), [1]))
    pos = (-3.0, 0.4, 0.3)
    desc.camera = scenes.CameraDesc(pos, scenes.q_look_at(pos, (0.0, -0.1, 0.0)), 1.0, 0.8)
    desc.env = scenes.EnvDesc(1, scenes.value_noise_env(32, 16, 3), 0.0)
    return desc


@pytest.mark.parametrize("n", [4000, 5000])      # on both sides of the tail kernel's choice of walk
def test_deep_stacks_on_both_walks(torch_gpu, n):
    desc = lit_degenerate_scene(n)
    W = H = 64
    frames = 3
    runs = {d: render_gpu(desc, W, H, frames, 6, False, wavefront_depth=d, want_accum=True) for d in (0, 64)}
    imgs, st, rng, acc = runs[0]
    imgs1, st1, rng1, acc1 = runs[64]
    assert st["closestRays"] == st1["closestRays"] and st["shadowRays"] == st1["shadowRays"]
    assert np.array_equal(rng, rng1)
    assert np.array_equal(np.asarray(acc), np.asarray(acc1))
    ref, ost, orng, _ = ob.Scene(desc).render(W, H, frames, max_path_length=6, rng_state=ob.seed_states(W, H))
    print("rays", st["closestRays"], ost["closest_rays"], "identical RNG states", np.mean(rng == orng))
    assert np.mean(rng == orng) > 0.97
    assert_pixels_match_where_paths_match(imgs[-1][..., :3], ref, rng, orng, W, H, 1e-3)


def render_cached(desc, W, H, frames, spectral, wavefront_depth):
    with api.Context(spectral=spectral, max_path_length=6) as ctx:
        ctx.set_wavefront_depth(wavefront_depth)
        bs = api.build_scene(ctx, desc)
        ctx.bind_output(W, H)
        ctx.set_radiance_cache(True)
        ctx.set_cache_settings(trainingPaths=W * H // 4)
        for f in range(frames):
            ctx.render(bs.camera, f == 0, frames)
        return ctx.read_output(), ctx.read_rng(), ctx.stats(), ctx.cache_loss()


@pytest.mark.parametrize("triangles", [0, 6000])  # the Cornell box alone, and with blobs
@pytest.mark.parametrize("spectral", [False, True])
def test_cached_frames_on_both_walks(torch_gpu, triangles, spectral):
    """Cached frames are the same bits whether the tail kernel or the per-depth kernels trace them:
    the same paths end in the cache and the same samples train it, in the same order."""
    desc = scenes.tessellated_cornell(5, triangles) if triangles else scenes.cornell_box()
    W = H = 64
    img, rng, st, loss = render_cached(desc, W, H, 6, spectral, 0)
    img1, rng1, st1, loss1 = render_cached(desc, W, H, 6, spectral, 64)
    assert st["closestRays"] == st1["closestRays"] and st["shadowRays"] == st1["shadowRays"]
    assert loss == loss1 and loss[1] > 0
    assert np.array_equal(rng, rng1)
    assert np.array_equal(img.view(np.uint32), img1.view(np.uint32))


def textured(desc):
    """The scene with its first material's albedo read from a texture."""
    texels = np.random.default_rng(8).uniform(0.1, 0.9, (4, 4, 4)).astype(np.float32)
    image = scenes.ImageDesc(texels.view(np.uint8).reshape(4, 4, 16), 4, 4, "RGBA32Fx4", "Reflectance", scenes.REC709)
    desc.materials[0].plugs["albedo"] = (scenes.NodeDesc("Image2DTexture", image=image), osn.PLUG["Spectrum"], 0)
    return desc


@pytest.mark.parametrize("spectral", [False, True])
def test_batch_with_node_programs_equals_single_renders(torch_gpu, spectral):
    descs = [textured(scenes.cornell_box()), textured(scenes.tessellated_cornell(5, 6000)), scenes.cornell_box(seed=7)]
    specs = [(0, 48, 40, 9, 8), (1, 64, 33, 8, 6), (2, 17, 20, 10, 5)]
    outs, _, _, sched = run_batch(descs, specs, spectral)
    print("schedule", sched)
    for k, (s, W, H, spp, depth) in enumerate(specs):
        ref = single(descs[s], W, H, spp, depth, spectral)
        assert np.array_equal(outs[k].view(np.uint32), ref.view(np.uint32)), k
