"""Closest-hit and any-hit traversal at the edges of the box test, against the oracle's brute force.

The box test takes a plane's ray parameter as q * (step / d) + (origin - org) / d with a bound on
the rounding of those two terms (kernels.hip, NodeAxis).  The cases here are the ones the bound
is for: directions with zero, negative-zero and tiny components, unnormalised directions, origins
on box planes and in the plane of flat triangles, and scenes far from the origin of coordinates,
where the two terms cancel.  A culled box would lose a hit, so every hit must be the brute
force's, bit for bit."""
import numpy as np
import pytest

from oracle import binding as ob
from tests.helpers import gpu_trace
from vlr_amd import api, scenes

pytestmark = pytest.mark.gpu

INF = np.float32(3.4028235e38)


def moved(desc, offset):
    for inst in desc.instances:
        inst.transform = inst.transform.copy()
        inst.transform[12:15] += np.asarray(offset, np.float32)
    return desc


def vertex_coordinates(desc):
    """World-space vertex coordinates per axis, by the float32 transform of the library."""
    out = [[], [], []]
    for inst in desc.instances:
        m = inst.transform.reshape(4, 4, order="F").astype(np.float32)
        for k in inst.meshes:
            p = desc.meshes[k].vertices[:, 0:3]
            for a in range(3):
                out[a].append(m[a, 0] * p[:, 0] + m[a, 1] * p[:, 1] + m[a, 2] * p[:, 2] + m[a, 3])
    return [np.unique(np.concatenate(c)) for c in out]


def edge_rays(kind, n, lo, hi, seed, coords=None):
    rng = np.random.default_rng(seed)
    rays = np.zeros(n, api.RAY_DTYPE)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    o = rng.uniform(lo, hi, size=(n, 3))
    axis = rng.integers(0, 3, n)
    if kind == "parallel":            # along an axis, the other components 0 or -0
        s = rng.choice([-1.0, 1.0], n)
        d = np.where(rng.random((n, 3)) < 0.5, 0.0, -0.0)
        d[np.arange(n), axis] = s
    elif kind == "one zero":
        d[np.arange(n), axis] = rng.choice([0.0, -0.0], n)
    elif kind == "tiny":
        d[np.arange(n), axis] *= 10.0 ** -rng.uniform(6, 44, n)
    elif kind == "unnormalised":
        d *= 10.0 ** rng.uniform(-12, 12, (n, 1))
    elif kind == "on planes":         # origins on the planes of vertices, which the boxes' faces lie in
        for a in range(3):
            inside = coords[a][(coords[a] >= lo[a]) & (coords[a] <= hi[a])]
            o[axis == a, a] = rng.choice(inside, (axis == a).sum())
    rays["org"], rays["dir"], rays["tmax"] = o.astype(np.float32), d.astype(np.float32), INF
    return rays


@pytest.mark.parametrize("kind", ["parallel", "one zero", "tiny", "unnormalised", "on planes"])
@pytest.mark.parametrize("scene,offset", [("cornell", 0.0), ("cornell", 3000.0), ("blobs", 0.0), ("blobs", 1000.0)])
def test_edge_rays_hit_what_brute_force_hits(torch_gpu, kind, scene, offset):
    desc = scenes.cornell_box() if scene == "cornell" else scenes.tessellated_cornell(3, 6000)
    desc = moved(desc, (offset, -offset, 0.5 * offset))
    c = np.array([offset, -offset, 0.5 * offset])
    coords = vertex_coordinates(desc)
    rays = edge_rays(kind, 4096 + 17, c + [-1.6, -0.1, -1.6], c + [1.6, 3.1, 1.6], 11, coords)
    if kind == "on planes":
        assert np.all(np.any([np.isin(rays["org"][:, a], coords[a]) for a in range(3)], axis=0))
    with api.Context() as ctx:
        bs = api.build_scene(ctx, desc)
        hits = gpu_trace(torch_gpu, ctx, bs.scene, rays)
        blocked = gpu_trace(torch_gpu, ctx, bs.scene, rays, any_hit=True)["inst"] >= 0
    ref = ob.Scene(desc).trace_closest(rays, use_bvh=False)
    found = ref["inst"] >= 0
    print(kind, scene, offset, "hits", found.mean())
    assert found.mean() > 0.5
    np.testing.assert_array_equal(hits["inst"] >= 0, found)
    np.testing.assert_array_equal(hits["t"][found], ref["t"][found])
    np.testing.assert_array_equal(blocked, found)


@pytest.mark.parametrize("lo,hi", [(-122, -100), (-100, -60), (60, 100), (100, 127)])
@pytest.mark.parametrize("any_hit", [False, True])
def test_directions_of_extreme_length(torch_gpu, lo, hi, any_hit):
    """Scaling a direction by a power of two scales the hit's distance by its inverse and changes
    nothing else, down to directions whose smaller components are denormal and up to those whose
    reciprocals are.  The reference traces the directions scaled back, which is exact."""
    desc = scenes.tessellated_cornell(3, 6000)
    rays = edge_rays("", 4096 + 17, [-1.4, 0.1, -1.4], [1.4, 2.9, 1.4], 12)
    rng = np.random.default_rng(13)
    n = len(rays)
    axis = rng.integers(0, 3, n)
    d = rays["dir"].astype(np.float64)
    # half of the rays leave a plane only slowly: two of the components are 1 and 3 to 100 times smaller
    slow = rng.random(n) < 0.5
    d[slow, axis[slow]] *= 10.0 ** -rng.uniform(0.5, 2, slow.sum())
    exponent = rng.integers(lo, hi + 1, n)
    rays["dir"] = np.ldexp(d, exponent[:, None]).astype(np.float32)
    unit = rays.copy()
    unit["dir"] = np.ldexp(rays["dir"].astype(np.float64), -exponent[:, None]).astype(np.float32)
    with api.Context() as ctx:
        bs = api.build_scene(ctx, desc)
        hits = gpu_trace(torch_gpu, ctx, bs.scene, rays, any_hit=any_hit)
    ref = ob.Scene(desc).trace_closest(unit, use_bvh=False)
    found = ref["inst"] >= 0
    assert found.mean() > 0.5
    np.testing.assert_array_equal(hits["inst"] >= 0, found)
    if not any_hit:
        expected = np.ldexp(ref["t"].astype(np.float64), -exponent).astype(np.float32)
        np.testing.assert_array_equal(hits["t"][found], expected[found])
        same = found & (hits["prim"] == ref["prim"]) & (hits["geomInst"] == ref["geomInst"])
        assert same.sum() > 0.99 * found.sum()      # the others tie on an edge of two triangles
        np.testing.assert_array_equal(hits["b1"][same], ref["b1"][same])
        np.testing.assert_array_equal(hits["b2"][same], ref["b2"][same])
