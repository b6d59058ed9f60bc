"""Calls captured into a graph: every replay gives the eager call's result, with other work of the context in between."""
import numpy as np
import pytest
import torch

from raytracergpu_mastersproject_amd import layouts as L
from raytracergpu_mastersproject_amd import workloads as W

from helpers import gpu_trace

pytestmark = pytest.mark.gpu


class _Handle:
    def __init__(self, stream):
        self.handle = stream.cuda_stream


def _capture(call):
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        call(_Handle(stream))
    return graph


@pytest.mark.parametrize("how,w,h,spp", [("render", 64, 64, 1), ("render", 501, 333, 1), ("render", 1920, 1080, 1),
                                         ("noalloc", 256, 256, 1), ("noalloc", 501, 333, 5)])
def test_renders(native, how, w, h, spp):
    """An image of one sample a pixel needs no path storage: rt_render takes none while its stream is captured."""
    ctx = native.Context(0)  # holds no storage from earlier renders
    s = W.soup_scene(1024)
    sid = ctx.upload(s["tris"], None, s["materials"])
    acc, ref = native.DeviceArray(16 * w * h), native.DeviceArray(16 * w * h)
    fn = ctx.render if how == "render" else ctx.render_noalloc

    def call(stream=None):
        ctx.accum_clear(acc, w * h, stream=stream)
        fn(sid, s["params"], w, h, spp, acc, stream=stream)

    graph = _capture(call)
    for k in range(4):
        ctx.accum_clear(ref, w * h)
        ctx.render(sid, s["params"], w, h, spp, ref)
        want = ref.to_numpy(np.uint32)
        acc.zero()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(acc.to_numpy(np.uint32), want), k
    ctx.release(sid)
    del graph
    ctx.close()


@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("n", [64, 30_000, 200_001, 1_000_000])
def test_queries(ctx, native, n, any_hit):
    tris, mats = W.cluster_scene(16, 4096, seed=81)
    sid = ctx.upload(tris, None, mats)
    rays = W.incoherent_rays(n, *W.scene_bounds(tris), seed=82)
    rays["o"][::100] -= rays["d"][::100] * np.float32(9000.0)  # traced by the launch over the marked rays
    dr, dh = native.DeviceArray.from_numpy(rays), native.DeviceArray(16 * n)
    graph = _capture(lambda st: ctx.trace(sid, dr, n, dh, any_hit=any_hit, stream=st))
    for k in range(4):
        want = gpu_trace(ctx, sid, rays, any_hit=any_hit)
        dh.zero()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(dh.to_numpy(L.HIT, n).view(np.uint32), want.view(np.uint32)), k
    ctx.release(sid)
