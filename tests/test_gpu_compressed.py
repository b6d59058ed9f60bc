"""Width-4 launches over compressed nodes against the exact nodes, bit for bit.  A launch that counts tests per
ray reads the exact nodes, so its hits are the other side; the scenes and rays are those where a larger box
could let a hit through that the exact box does not: rays in box-face planes, zero and tiny direction
components, far origins, flat triangles, boxes of a caller's node buffer that hold more or less than they should."""
import numpy as np
import pytest

from raytracergpu_mastersproject_amd import layouts as L
from raytracergpu_mastersproject_amd import workloads as W

from helpers import gpu_trace, small_cluster_scene, with_spheres

pytestmark = pytest.mark.gpu


def _grid(k=24):
    """Axis-aligned unit cells of two triangles each in k x k floors at three heights: flat boxes, shared edges."""
    x, z = np.meshgrid(np.arange(k), np.arange(k), indexing="ij")
    parts = []
    for y in (0.0, 1.0, 2.5):
        a = np.stack([x.ravel(), np.full(k * k, y), z.ravel()], 1).astype(np.float64)
        b, c, d = a + [1, 0, 0], a + [1, 0, 1], a + [0, 0, 1]
        parts += [W.make_triangles(a, b, c), W.make_triangles(a, c, d)]
    return np.concatenate(parts)


def _rays(n, lo, hi, seed):
    rays = W.incoherent_rays(n, lo, hi, seed=seed)
    ctr, ext = (np.asarray(lo) + hi) / 2, float(np.max(np.asarray(hi) - lo)) + 1e-3
    r = np.random.default_rng(seed)
    rays["tmax"] = np.float32(1e7) * np.float32(max(ext, 1.0))
    far = slice(0, n, 5)  # from far away towards the scene
    d = rays["d"][far]
    rays["o"][far] = ctr - d * ext * np.exp(r.uniform(0, 11, len(d)))[:, None] + r.normal(size=d.shape) * 0.3 * ext
    axis = np.arange(1, n, 7)  # one or two zero components, both signs of zero
    rays["d"][axis, axis % 3] = 0.0
    rays["d"][axis[::2], (axis[::2] + 1) % 3] = -0.0
    rays["o"][axis[::3]] = np.round(rays["o"][axis[::3]])  # in the planes of cell faces
    tiny = np.arange(2, n, 31)
    rays["d"][tiny, tiny % 3] = np.resize(np.float32([1e-20, -1e-27, 3e-28, 1e-38, -1e-41]), len(tiny))
    rays["tmin"][3::11] = -0.25 * ext
    rays["tmax"][4::13] = 0.05 * ext
    rays["tmin"][5::97], rays["tmax"][5::97] = 2.0, 1.0
    rays["o"][6::211, 0] = np.inf
    rays["d"][7::211, 1] = np.nan
    rays["d"][8::211, 2] = np.inf
    return rays


def _check(ctx, native, sid, rays):
    for any_hit in (False, True):
        for fp32 in (False, True):
            exact, _ = gpu_trace(ctx, sid, rays, any_hit=any_hit, counts=True, fp32=fp32)
            for cfg in (None, native.launch_config(block=64, lds_stack=4, persistent=0)):
                got = gpu_trace(ctx, sid, rays, any_hit=any_hit, fp32=fp32, cfg=cfg)
                assert np.array_equal(got.view(np.uint32), exact.view(np.uint32))
            dr, dh = native.DeviceArray.from_numpy(rays), native.DeviceArray(16 * len(rays))
            ctx.trace_batch([(sid, len(rays), dr, dh)], any_hit=any_hit, fp32=fp32)
            assert np.array_equal(dh.to_numpy(np.uint32), exact.view(np.uint32))
    return float(np.mean(exact["prim"] != L.NO_HIT))


@pytest.mark.parametrize("leaf", [1, 4])
@pytest.mark.parametrize("scene,scale,shift", [("grid", 1.0, 0.0), ("grid", 1.0, 4096.0), ("grid", 1e-3, 0.0),
                                               ("cluster", 1.0, 0.0), ("cluster", 1000.0, 30000.0),
                                               ("cluster", 1e7, 0.0), ("cluster", 4e7, 0.0)])
def test_same_hits_as_exact_nodes(ctx, native, scene, scale, shift, leaf):
    tris, mats = (_grid(), W.make_materials([0.5, 0.5, 0.5], L.DIFFUSE)) if scene == "grid" else small_cluster_scene(6, 700, seed=41)
    sph = with_spheres(tris, mats, 6)
    for k in ("v0", "v1", "v2"):
        tris[k][:, :3] = tris[k][:, :3] * np.float32(scale) + np.float32(shift)
    sph["center"][:, :3] = sph["center"][:, :3] * np.float32(scale) + np.float32(shift)
    sph["radius"] *= np.float32(scale)
    sid = ctx.upload(tris, sph, mats, leaf_size=leaf)
    rays = _rays(900_001, *W.scene_bounds(tris), seed=42)  # above the sizes that use several lanes per ray
    assert _check(ctx, native, sid, rays) > 0.005
    ctx.release(sid)


@pytest.mark.parametrize("boxes", ["loose", "leaf too small", "parent too small", "inverted", "nan"])
def test_callers_node_boxes(ctx, native, boxes):
    tris, mats = small_cluster_scene(4, 300, seed=43)
    n = len(tris)
    sid = ctx.upload(tris, None, mats, flags=native.BUILD_KEEP_BINARY)
    nodes = ctx.nodes(sid).copy()
    ctx.release(sid)
    leaf = nodes[n - 1:]
    if boxes == "loose":
        nodes["minX"] -= 0.01
        nodes["maxZ"] += 0.02
    elif boxes == "leaf too small":
        leaf["maxX"][::3] = (leaf["minX"][::3] + leaf["maxX"][::3]) / 2
    elif boxes == "parent too small":
        mid = slice(n // 4, n // 2)
        nodes["minY"][mid] = (nodes["minY"][mid] + nodes["maxY"][mid]) / 2
    elif boxes == "inverted":
        leaf["minX"][::5], leaf["maxX"][::5] = leaf["maxX"][::5].copy(), leaf["minX"][::5].copy()
    else:
        leaf["minZ"][::50] = np.nan
    sid = ctx.upload(tris, None, mats, nodes=nodes)
    _check(ctx, native, sid, _rays(900_001, *W.scene_bounds(tris), seed=44))
    ctx.release(sid)
