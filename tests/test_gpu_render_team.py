"""Small images, whose paths are traced by several lanes each, against the one-lane-per-path persistent launch:
both sides of every size at which the lanes per path change, with all materials and spheres, samples continued over
calls, depths 0 to 12, a camera far outside the scene, and no scratch allocation."""
import numpy as np
import pytest

from raytracergpu_mastersproject_amd import layouts as L
from raytracergpu_mastersproject_amd import workloads as W

from helpers import with_spheres

pytestmark = pytest.mark.gpu


def _image(ctx, native, sid, params, w, h, calls, flags=0, noalloc=False):
    acc, seg = native.DeviceArray(16 * w * h), native.DeviceArray(8)
    seg.zero()
    ctx.accum_clear(acc, w * h)
    for spp in calls:
        (ctx.render_noalloc if noalloc else ctx.render)(sid, params, w, h, spp, acc, flags=flags, segments=seg)
    return acc.to_numpy(np.uint32), int(seg.to_numpy(np.uint64, 1)[0])


def _scene(ctx, ntri=6000, leaf_size=1):
    s = W.served_scene(ntri, 51)
    return ctx.upload(s["tris"], with_spheres(s["tris"], s["materials"], 9), s["materials"], leaf_size=leaf_size), s["params"]


@pytest.mark.parametrize("w,h,calls", [(1, 1, (1,)), (64, 128, (1,)), (8193, 1, (1,)), (128, 64, (2, 2)),
                                       (181, 181, (1,)), (256, 128, (1,)), (32769, 1, (1,)), (200, 111, (3, 8)),
                                       (512, 512, (1,)), (262145, 1, (1,)), (600, 600, (1, 2)), (131073, 1, (1,)),
                                       (512, 512, (2,)), (524289, 1, (1,)), (2048, 256, (4,)), (2097153, 1, (1,))])
def test_sizes_agree_with_one_lane_per_path(ctx, native, w, h, calls):
    sid, params = _scene(ctx)
    a, segs = _image(ctx, native, sid, params, w, h, calls)
    b, _ = _image(ctx, native, sid, params, w, h, calls, flags=native.RENDER_PERSISTENT_PATHS)
    assert np.array_equal(a, b) and segs >= w * h
    c, _ = _image(ctx, native, sid, params, w, h, calls, noalloc=True)
    assert np.array_equal(a, c)
    ctx.release(sid)


@pytest.mark.parametrize("depth", [0, 1, 2, 12])
@pytest.mark.parametrize("flags", [0, 1, 2])  # RT_RENDER_REFERENCE_MATERIALS, RT_RENDER_NO_PRIMARY_CACHE
def test_depths_and_flags(ctx, native, depth, flags):
    sid, params = _scene(ctx, leaf_size=3)
    params = params.copy()
    params["maxRayTraceDepth"], params["randomState"] = depth, 77
    for w, h, calls in ((70, 50, (2,)), (200, 150, (1, 4)), (300, 300, (2,))):
        a, _ = _image(ctx, native, sid, params, w, h, calls, flags=flags)
        b, _ = _image(ctx, native, sid, params, w, h, calls, flags=flags | native.RENDER_PERSISTENT_PATHS)
        assert np.array_equal(a, b)
    ctx.release(sid)


def test_far_camera_and_empty_scene(ctx, native):
    sid, params = _scene(ctx)
    params = params.copy()
    params["camPos"][:3], params["verticalFOV"] = (0.0, 9e4, -9e4), 0.002
    a, _ = _image(ctx, native, sid, params, 96, 96, (2,))
    b, _ = _image(ctx, native, sid, params, 96, 96, (2,), flags=native.RENDER_PERSISTENT_PATHS)
    assert np.array_equal(a, b)
    ctx.release(sid)
    sid = ctx.upload(None, None, W.make_materials([0.5, 0.5, 0.5], L.DIFFUSE))
    a, _ = _image(ctx, native, sid, params, 40, 30, (2,))
    b, _ = _image(ctx, native, sid, params, 40, 30, (2,), flags=native.RENDER_PERSISTENT_PATHS)
    assert np.array_equal(a, b)
    ctx.release(sid)
