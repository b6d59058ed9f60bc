"""Launches of few rays (several lanes per ray) against one lane per ray and the oracle, bit for bit: both
sides of every size at which the lanes per ray change, ties, spheres, multi-primitive leaves, odd rays, and
trees too deep for the shared stack."""
import numpy as np
import pytest

from raytracergpu_mastersproject_amd import layouts as L
from raytracergpu_mastersproject_amd import workloads as W

from helpers import compare_hits, gpu_trace, small_cluster_scene, upload_both, with_spheres

pytestmark = pytest.mark.gpu


def _same(a, b):
    return np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("n", [1, 63, 6144, 6145, 32768, 32769, 262144, 262145, 393216, 393217, 786432, 786433, 4194304,
                               4194305])
def test_sizes_agree_with_one_lane_per_ray(ctx, native, n, any_hit):
    tris, mats = small_cluster_scene(16, 4096, seed=31)
    sid = ctx.upload(tris, with_spheres(tris, mats, 7), mats)
    rays = W.incoherent_rays(n, *W.scene_bounds(tris), seed=32 + n)
    rays["tmax"][::3] = 0.4
    one = native.launch_config(block=64, lds_stack=8, persistent=0)
    for fp32 in (False, True):
        assert _same(gpu_trace(ctx, sid, rays, any_hit=any_hit, fp32=fp32),
                     gpu_trace(ctx, sid, rays, any_hit=any_hit, fp32=fp32, cfg=one))
    ctx.release(sid)


@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("n", [3000, 20000, 40000])
def test_ties_leaves_and_odd_rays(ctx, native, O, n, any_hit):
    """Every triangle three times (the smallest leaf slot wins), leaves of up to four, rays with a zero or
    NaN direction component, a negative tmin, an empty interval, an infinite origin."""
    tris, mats = small_cluster_scene(4, 500, seed=33)
    tris = np.concatenate([tris, tris, tris])
    sid, osc = upload_both(ctx, O, tris, with_spheres(tris, mats, 4), mats, leaf_size=4)
    rays = W.incoherent_rays(n, *W.scene_bounds(tris), seed=34)
    rays["d"][0::11, 1] = 0.0
    rays["d"][1::97, 0] = np.nan
    rays["tmin"][2::7] = -0.5
    rays["tmax"][3::13] = 0.0005
    rays["o"][4::101, 2] = np.inf
    rays["d"][5::17] = [0.0, 0.0, -1.0]
    g = gpu_trace(ctx, sid, rays, any_hit=any_hit)
    assert _same(g, gpu_trace(ctx, sid, rays, any_hit=any_hit,
                              cfg=native.launch_config(block=128, lds_stack=16, persistent=0)))
    assert compare_hits(g, osc.trace(rays, O.WIDE, any_hit=any_hit)) == 0
    ctx.release(sid)


def _chain(n, tris):
    """A builder output whose tree is a list: internal node i holds leaf i and internal node i + 1."""
    nodes = np.zeros(2 * n - 1, L.BVH_NODE)
    v = np.stack([tris[k][:, :3] for k in ("v0", "v1", "v2")])
    lo, hi = v.min(0) - 5e-4, v.max(0) + 5e-4
    for k, (a, b) in enumerate((("minX", "maxX"), ("minY", "maxY"), ("minZ", "maxZ"))):
        nodes[a][n - 1:], nodes[b][n - 1:] = lo[:, k], hi[:, k]
        nodes[a][:n - 1] = np.minimum.accumulate(lo[::-1, k])[::-1][:n - 1]
        nodes[b][:n - 1] = np.maximum.accumulate(hi[::-1, k])[::-1][:n - 1]
    i = np.arange(n - 1)
    nodes["left"][:n - 1] = n - 1 + i
    nodes["right"][:n - 1] = np.where(i == n - 2, 2 * n - 2, i + 1)
    nodes["primitiveIndex"][n - 1:] = np.arange(n)
    nodes["primitiveType"][n - 1:] = L.TRIANGLE_PRIMITIVE
    return nodes


@pytest.mark.parametrize("ntri,n", [(80, 40000), (95, 300000), (190, 20000), (190, 70000), (190, 300000)])
def test_deep_trees(ctx, native, ntri, n):
    """stack bounds from 82 (fits eight lanes' stack) to 190 (too deep for eight and sixteen)."""
    tris, mats = small_cluster_scene(2, 95, seed=35)
    tris = np.ascontiguousarray(tris[:ntri])
    sid = ctx.upload(tris, None, mats, nodes=_chain(ntri, tris))
    assert ctx.info(sid).stack_bound >= ntri - 2
    rays = W.incoherent_rays(n, *W.scene_bounds(tris), seed=36)
    for any_hit in (False, True):
        g = gpu_trace(ctx, sid, rays, any_hit=any_hit)
        assert _same(g, gpu_trace(ctx, sid, rays, any_hit=any_hit,
                                  cfg=native.launch_config(block=64, lds_stack=16, persistent=0)))
        assert np.mean(g["prim"] != L.NO_HIT) > 0.001
    ctx.release(sid)


def test_a_tuned_shape_leaves_small_launches_to_teams(ctx, native):
    """Tuned with more rays than teams are best at, where one lane per ray wins; a small query then takes as long as before."""
    s = W.soup_scene(1024)
    sid = ctx.upload(s["tris"], None, s["materials"])
    lo, hi = W.scene_bounds(s["tris"])
    n = 300_000
    many = native.DeviceArray.from_numpy(W.incoherent_rays(n, lo, hi, seed=38))
    few = native.DeviceArray.from_numpy(W.incoherent_rays(4096, lo, hi, seed=39))
    hits = native.DeviceArray(16 * n)

    def small_us():
        t = []
        for _ in range(40):
            a, b = native.Event(), native.Event()
            a.record()
            ctx.trace(sid, few, 4096, hits)
            b.record()
            t.append(a.elapsed_ms(b) * 1e3)
        return float(np.median(t))

    before = small_us()
    res = ctx.autotune(sid, many, n, hits)
    assert res.cfg.persistent == 0  # else this test says nothing
    assert small_us() < 1.8 * before
    want = gpu_trace(ctx, sid, W.incoherent_rays(4096, lo, hi, seed=39), cfg=native.launch_config(persistent=0))
    ctx.trace(sid, few, 4096, hits)
    assert np.array_equal(hits.to_numpy(np.uint32, 4 * 4096), want.view(np.uint32))
    ctx.release(sid)
