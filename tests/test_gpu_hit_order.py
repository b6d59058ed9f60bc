"""Closest hits do not depend on how a launch visits the tree: every route against the ordered walk of the exact nodes
(a launch that counts tests), bit for bit, where two hits lie within a few roundings and a hit lies outside its own
box: meshes far from the origin, rays aimed at shared vertices and edges, nearly equal spheres, far origins."""
import numpy as np
import pytest

from raytracergpu_mastersproject_amd import layouts as L
from raytracergpu_mastersproject_amd import workloads as W

from helpers import gpu_trace

pytestmark = pytest.mark.gpu

MATS = W.make_materials([0.5, 0.5, 0.5], L.DIFFUSE)


def _mesh(freq, shift):
    tris = W.make_triangles(*W.icosphere(freq))
    for k in ("v0", "v1", "v2"):
        tris[k][:, :3] += np.float32(shift)
    return tris


def _shells(shift):
    """Spheres in pairs whose surfaces lie within a few roundings of each other."""
    rng = np.random.default_rng(5)
    sph = np.zeros(400, L.SPHERE)
    c = rng.uniform(-3, 3, (200, 3))
    sph["center"][:, :3] = np.repeat(c, 2, 0) + shift
    sph["radius"] = np.repeat(rng.uniform(0.2, 0.4, 200), 2) * (1 + 3e-7 * rng.integers(0, 3, 400))
    return sph


def _rays(n, tris, seed):
    """A third at random, a third at vertices and the middles of edges, a third from far outside."""
    r = np.random.default_rng(seed)
    lo, hi = W.scene_bounds(tris)
    rays = W.incoherent_rays(n, lo, hi, seed=seed, tmax=1e7)
    ext = float(np.max(np.asarray(hi) - lo))
    at = slice(1, n, 3)
    i = r.integers(0, len(tris), len(rays["o"][at]))
    w = r.choice([0.0, 0.5, 1.0], (len(i), 1))
    d = tris["v0"][i][:, :3] * (1 - w) + tris["v1"][i][:, :3] * w - rays["o"][at]
    rays["d"][at] = d / np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-30)
    out = slice(2, n, 3)
    d = rays["d"][out]
    rays["o"][out] -= d * (ext * 10.0 ** r.uniform(0, 2.9, (len(d), 1))).astype(np.float32)
    return rays


@pytest.mark.parametrize("shift", [0.0, 300.0, 1e5])  # the last over the exact nodes, which hold such a scene better
@pytest.mark.parametrize("scene", ["mesh", "shells"])
def test_every_route_finds_the_ordered_hit(ctx, native, scene, shift):
    tris = _mesh(48 if shift < 1e4 else 20, shift)
    sph = _shells(shift) if scene == "shells" else None
    sid = ctx.upload(tris, sph, MATS)
    # 64, 32, 16 and 8 lanes per ray; one, with and without teams at the end
    for n in (5_000, 30_000, 200_000, 380_000, 1_000_000) + ((4_300_000,) if shift == 300.0 else ()):
        rays = _rays(n, tris, n)
        dr = native.DeviceArray.from_numpy(rays)
        for fp32 in (True, False):
            want, _ = gpu_trace(ctx, sid, rays, counts=True, fp32=fp32)
            assert np.mean(want["prim"] != L.NO_HIT) > 0.2
            assert np.array_equal(gpu_trace(ctx, sid, rays, fp32=fp32).view(np.uint32), want.view(np.uint32))
            dh = native.DeviceArray(16 * n)
            half = n // 2 + 17
            ctx.trace_batch([(sid, half, dr.ptr, dh.ptr), (sid, n - half, dr.ptr + 32 * half, dh.ptr + 16 * half)], fp32=fp32)
            assert np.array_equal(dh.to_numpy(np.uint32), want.view(np.uint32))
        one = native.launch_config(persistent=0)
        assert np.array_equal(gpu_trace(ctx, sid, rays, cfg=one).view(np.uint32), want.view(np.uint32))
    ctx.release(sid)


@pytest.mark.parametrize("shift", [0.0, 300.0])
def test_every_schedule_renders_the_ordered_image(ctx, native, shift):
    """Against the same tree over the exact nodes: a caller's node buffer in which one leaf, behind the camera, has too
    small a box."""
    tris, n = _mesh(40, shift), 20 * 40 * 40
    tris = np.concatenate([tris, W.make_triangles(*[np.array([[0.0, y, 30.0]]) + shift + np.array(p) for y, p in
                                                    ((0, (0, 0, 0)), (0, (1, 0, 0)), (1, (0, 0, 1)))])])
    mats = np.concatenate([W.make_materials(np.full((3, 3), 0.9), k, 0.1) for k in (L.DIFFUSE, L.METALLIC)] +
                          [W.make_materials(np.ones((2, 3)), L.DIELECTRIC, 1.5), W.make_materials(np.ones((1, 3)), L.LIGHT)])
    tris["materialIndex"] = np.random.default_rng(1).integers(0, len(mats), n + 1)
    a = ctx.upload(tris, None, mats, flags=native.BUILD_KEEP_BINARY)
    nodes = ctx.nodes(a).copy()
    leaf = nodes[n:]
    last = np.nonzero(leaf["primitiveIndex"] == n)[0][0]
    leaf["maxX"][last] = leaf["minX"][last]
    b = ctx.upload(tris, None, mats, nodes=nodes)
    p = L.make_params(np.array((0.3, 0.6, -2.4)) + shift, (shift, shift, shift), (0.0, 1.0, 0.0), 50.0, n + 1, 0, len(mats), 8, 3)
    for w, h, spp in ((64, 64, 1), (256, 256, 1), (301, 203, 9), (640, 360, 20)):
        acc = native.DeviceArray(16 * w * h)

        def image(sid, flags):
            ctx.accum_clear(acc, w * h)
            ctx.render(sid, p, w, h, spp, acc, flags=flags)
            return acc.to_numpy(np.uint32, 4 * w * h)

        want = image(b, 0)
        for flags in (0, native.RENDER_PERSISTENT_PATHS, native.RENDER_NO_SPLIT, native.RENDER_WAVEFRONT):
            assert np.array_equal(image(a, flags), want), (w, h, spp, flags)
        ctx.accum_clear(acc, w * h)
        ctx.render_batch([(a, p, w, h, spp, acc)])
        assert np.array_equal(acc.to_numpy(np.uint32, 4 * w * h), want)
    ctx.release(a)
    ctx.release(b)


@pytest.mark.parametrize("far", [3, 512, 513, 5000, 0])  # rays from far outside; 0: all
@pytest.mark.parametrize("n", [5_000, 30_000, 200_001, 700_001])
def test_rays_from_far_outside(ctx, native, n, far):
    """They are left to a launch of their own: by a list of 512, or by the marks in the hit records."""
    tris = _mesh(48, 0.0)
    sid = ctx.upload(tris, None, MATS)
    rays = W.incoherent_rays(n, *W.scene_bounds(tris), seed=7, tmax=1e7)
    which = np.random.default_rng(n + far).permutation(n)[:far or n]
    rays["o"][which] -= rays["d"][which] * np.float32(4000.0)
    rays["d"][which[::50], 1] = np.float32(1e-30)  # no compressed nodes for these either
    dr, dh = native.DeviceArray.from_numpy(rays), native.DeviceArray(16 * n)
    for any_hit in (False, True):
        want, _ = gpu_trace(ctx, sid, rays, counts=True, any_hit=any_hit)
        assert np.array_equal(gpu_trace(ctx, sid, rays, any_hit=any_hit).view(np.uint32), want.view(np.uint32))
        third = n // 3
        ctx.trace_batch([(sid, third, dr.ptr, dh.ptr), (sid, 0, dr.ptr, dh.ptr),
                         (sid, n - third, dr.ptr + 32 * third, dh.ptr + 16 * third)], any_hit=any_hit)
        assert np.array_equal(dh.to_numpy(np.uint32), want.view(np.uint32))
    ctx.release(sid)


@pytest.mark.parametrize("n", [5_000, 30_000, 200_001, 700_001])
def test_bounds_that_are_not_numbers(ctx, native, n):
    """A NaN tmin bounds nothing, a NaN tmax lets no hit through, whichever route traces the ray."""
    tris = _mesh(24, 0.0)
    sid = ctx.upload(tris, None, MATS)
    rays = W.incoherent_rays(n, *W.scene_bounds(tris), seed=9, tmax=1e7)
    rays["tmin"][::3] = np.nan
    rays["tmax"][1::7] = np.nan
    rays["tmin"][2::5] = -np.inf
    rays["tmax"][3::11] = np.inf
    rays["tmin"][4::13], rays["tmax"][4::13] = 3.0, 1.0
    for any_hit in (False, True):
        want, _ = gpu_trace(ctx, sid, rays, counts=True, any_hit=any_hit, fp32=True)
        assert np.mean(want["prim"][::3] != L.NO_HIT) > 0.2
        got = gpu_trace(ctx, sid, rays, any_hit=any_hit, fp32=True)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    ctx.release(sid)
