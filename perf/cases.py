"""Performance cases of the ray-tracing library: what its users run, through the public Python binding.

  listed()            the fixed cases
  draw(rng)           one more case of the same kinds, its sizes spread over the same ranges
  prepare(case, seed) what a program holds before the call: resident scenes, device rays, images, a server
  run(state)          one pass through the public entry points, and its outputs
  work(case)          bytes that a pass cannot avoid: rays and geometry read once, hits and pixels written once
  exact(case, seed)   the outputs in double precision by brute force, where that is defined and affordable

Kinds of case:
  query   one rt_trace call over resident geometry (picking, visibility, baking)
  batch   one rt_trace_batch call over many resident scenes
  render  clear an image, path trace it, resolve it for display
  frame   a frame of an animated scene: upload and build, render, resolve, release
  load    a scene arrives, is built, answers one query and leaves
  serve   a server with resident scenes answers a burst of ray queries and renders
"""
from __future__ import annotations

import math

import numpy as np
import torch

from raytracergpu_mastersproject_amd import layouts as L
from raytracergpu_mastersproject_amd import native as N
from raytracergpu_mastersproject_amd import workloads as W

DEV = "cuda:0"
TMIN, TMAX = 0.001, 16.0  # rays end a little beyond any scene used here

_context = None


def _ctx() -> N.Context:
    """The process's context (a program holds one per GPU)."""
    global _context
    if _context is None:
        _context = N.Context(0)
    return _context


def listed():
    return [
        # a handful of rays against a small model: picking under the cursor, a physics probe
        dict(name="pick_64", kind="query", tris=1024, spheres=0, rays=64, any=False, fp32=False),
        # the smallest batch of the served and fused workloads
        dict(name="query_4k", kind="query", tris=120_000, spheres=0, rays=4096, any=False, fp32=False),
        # the reference's own fp32 results, triangles and spheres together, an odd count
        dict(name="query_64k_fp32", kind="query", tris=20_000, spheres=64, rays=65_537, any=False, fp32=True),
        # shadow rays (any hit) for a half-megapixel image, two lights
        dict(name="shadow_1m", kind="query", tris=1_000_000, spheres=0, rays=1_000_003, any=True, fp32=False),
        # the headline ray query: 16.8 M incoherent rays, 4.2 M triangles, closest hit
        dict(name="query_16m", kind="query", tris=4_194_304, spheres=0, rays=16_777_216, any=False, fp32=False),
        # many scenes' ray batches in one launch
        dict(name="batch_32", kind="batch", scenes=32, tri_hi=300_000, ray_hi=262_144),
        # the reference's soup case: 256x256, one sample, depth 8
        dict(name="render_soup", kind="render", scene="soup", tris=1024, width=256, height=256, spp=1),
        # a preview image with a ragged width
        dict(name="render_preview", kind="render", scene="served", tris=200_000, width=501, height=333, spp=12),
        # the headline frame: 1 M-triangle displaced icosphere, 1080p, 16 samples
        dict(name="render_1080p", kind="render", scene="icosphere", tris=1_003_520, width=1920, height=1080, spp=16),
        # one frame as the reference runs it: every frame uploads its scene, builds the BVH, renders, shows
        dict(name="frame_small", kind="frame", tris=3000, spheres=8, width=256, height=256, spp=1),
        # a server brings a scene in and answers its first query
        dict(name="load_1m", kind="load", tris=1_000_000, rays=65_536),
        # a burst of ray queries and small renders over resident scenes, served together
        dict(name="serve_burst", kind="serve", scenes=8, tri_hi=300_000, queries=20, ray_hi=100_000, renders=6),
    ]


def _log(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["query", "query", "query", "render", "render", "batch", "frame", "load", "serve"])
    if kind == "query":
        return dict(kind=kind, tris=_log(rng, 1000, 4_000_000), spheres=rng.choice([0, 0, 17]), rays=_log(rng, 64, 12_000_000),
                    any=rng.random() < 0.3, fp32=rng.random() < 0.3)
    if kind == "render":
        w, h = _log(rng, 64, 1920), _log(rng, 64, 1080)
        return dict(kind=kind, scene=rng.choice(["soup", "served"]), tris=_log(rng, 1000, 600_000), width=w, height=h,
                    spp=min(_log(rng, 1, 32), max(1, 16_000_000 // (w * h))))
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(4, 32), tri_hi=_log(rng, 20_000, 300_000), ray_hi=_log(rng, 16_000, 262_144))
    if kind == "frame":
        return dict(kind=kind, tris=_log(rng, 200, 50_000), spheres=rng.randint(0, 32), width=_log(rng, 64, 512),
                    height=_log(rng, 64, 512), spp=rng.randint(1, 4))
    if kind == "load":
        return dict(kind=kind, tris=_log(rng, 20_000, 900_000), rays=_log(rng, 4096, 65_536))
    return dict(kind=kind, scenes=rng.randint(3, 8), tri_hi=_log(rng, 20_000, 300_000), queries=rng.randint(4, 20),
                ray_hi=_log(rng, 8_000, 100_000), renders=rng.randint(1, 6))


# ---------------- inputs ----------------

def _clusters(ntri: int, seed: int):
    """A clustered soup of `ntri` triangles; their size follows the count, so the share of rays that hit
    stays that of the 4.2 M-triangle workload."""
    k = max(1, min(64, ntri // 64))
    per = -(-ntri // k)
    tris, mats = W.cluster_scene(k, per, tri_radius=0.005 * (4_194_304 / ntri) ** (1.0 / 3.0), seed=seed)
    return tris[:ntri], mats


def _spheres(count: int, seed: int) -> np.ndarray:
    rng = W.SplitMix64(seed ^ 0x5F)
    s = np.zeros(count, L.SPHERE)
    s["center"][:, :3] = rng.uniform(3 * count, -0.9, 0.9).reshape(count, 3)
    s["center"][:, 3] = 1.0
    s["radius"] = rng.uniform(count, 0.03, 0.15)
    return s


def _rays(n: int, lo, hi, seed: int) -> torch.Tensor:
    """[n, 8] float32 on the GPU: origins uniform in the scene's box, directions uniform on the sphere."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    lo, hi = (torch.as_tensor(np.asarray(v), dtype=torch.float32, device=DEV) for v in (lo, hi))
    r = torch.empty(n, 8, device=DEV)
    r[:, 0:3] = lo + (hi - lo) * torch.rand(n, 3, generator=g, device=DEV)
    r[:, 3] = TMIN
    d = torch.randn(n, 3, generator=g, device=DEV)
    r[:, 4:7] = d / d.norm(dim=1, keepdim=True)
    r[:, 7] = TMAX
    return r


def _geometry(case, seed: int):
    tris, mats = _clusters(case["tris"], seed)
    return tris, _spheres(case.get("spheres", 0), seed), mats


def _log_sizes(count: int, lo: float, hi: float, stream: int):
    """Log-uniform sizes; they belong to the case, so that every seed's outputs have the same shapes."""
    return [int(v) for v in np.exp(W.SplitMix64(stream).uniform(count, math.log(lo), math.log(hi)))]


def _render_scene(case, seed: int):
    if case["scene"] == "icosphere":
        return W.icosphere_scene(int(round(math.sqrt(case["tris"] / 20.0))), seed=seed, random_state=seed & 0xFFFF)
    s = W.soup_scene(case["tris"], seed=seed) if case["scene"] == "soup" else W.served_scene(case["tris"], seed)
    s["params"]["randomState"] = seed & 0xFFFF
    return s


def _frame_scene(case, seed: int):
    """A model in model space with its transform, spheres, a floor and a light."""
    s = W.soup_scene(case["tris"], seed=seed)
    mats = np.concatenate([W.material_palette(seed), s["materials"]])
    tris = s["tris"].copy()
    soup = slice(0, case["tris"])
    tris["materialIndex"] += 41
    tris["materialIndex"][soup] = (W.SplitMix64(seed ^ 0xA5).u64(case["tris"]) % np.uint64(40)).astype(np.uint32)
    tris["modelIndex"][soup] = 1
    sph = _spheres(case["spheres"], seed)
    sph["materialIndex"] = np.arange(case["spheres"]) % 40
    a = 0.1 + 0.01 * (seed % 100)
    spin = np.eye(4, dtype=np.float32)
    spin[0, 0] = spin[2, 2] = math.cos(a)
    spin[2, 0], spin[0, 2] = math.sin(a), -math.sin(a)  # column-major storage below
    models = np.stack([np.eye(4, dtype=np.float32), spin.T.copy()]).reshape(-1, 16)
    p = L.make_params((0.0, 0.5, -3.5), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 40.0, len(tris), len(sph), len(mats), 8,
                      seed & 0xFFFF)
    return tris, sph, mats, models, p


class _State:
    """Scenes, buffers and perhaps a server; closed and released when the program drops them."""

    def __init__(self, kind):
        self.kind, self.scenes, self.server = kind, [], None

    def upload(self, *args, **kw) -> int:
        sid = _ctx().upload(*args, **kw)
        self.scenes.append(sid)
        return sid

    def __del__(self):
        try:
            if self.server is not None:
                self.server.close()
            for sid in self.scenes:
                _ctx().release(sid)
        except Exception:
            pass


def _image(width, height):
    return torch.empty(height, width, 4, device=DEV)


def _hits(n):
    return torch.empty(n, 4, dtype=torch.int32, device=DEV)


def prepare(case, seed):
    s = _State(case["kind"])
    kind = s.kind
    if kind == "query":
        tris, sph, mats = _geometry(case, seed)
        s.sid = s.upload(tris, sph, mats)
        lo, hi = W.scene_bounds(tris)
        s.n, s.any, s.fp32 = case["rays"], bool(case["any"]), bool(case["fp32"])
        s.rays, s.hits = _rays(s.n, lo, hi, seed), _hits(s.n)
    elif kind == "batch":
        ntris = _log_sizes(case["scenes"], 1000, case["tri_hi"], 1)
        s.counts = _log_sizes(case["scenes"], 4096, case["ray_hi"], 2)
        s.hits, s.items, s.rays, at = _hits(sum(s.counts)), [], [], 0
        for k, (nt, nr) in enumerate(zip(ntris, s.counts)):
            tris, mats = _clusters(nt, seed * 64 + k)
            lo, hi = W.scene_bounds(tris)
            s.rays.append(_rays(nr, lo, hi, seed * 64 + k))
            s.items.append((s.upload(tris, None, mats), nr, s.rays[-1].data_ptr(), s.hits.data_ptr() + 16 * at))
            at += nr
    elif kind == "render":
        sc = _render_scene(case, seed)
        s.sid = s.upload(sc["tris"], sc["spheres"], sc["materials"])
        s.params, s.width, s.height, s.spp = sc["params"], case["width"], case["height"], case["spp"]
        s.accum, s.shown = _image(s.width, s.height), _image(s.width, s.height)
    elif kind == "frame":
        s.tris, s.spheres, s.materials, s.models, s.params = _frame_scene(case, seed)
        s.width, s.height, s.spp = case["width"], case["height"], case["spp"]
        s.accum, s.shown = _image(s.width, s.height), _image(s.width, s.height)
    elif kind == "load":
        s.tris, _, s.materials = _geometry(case, seed)
        lo, hi = W.scene_bounds(s.tris)
        s.n = case["rays"]
        s.rays, s.hits = _rays(s.n, lo, hi, seed), _hits(s.n)
    else:
        bounds = []
        setups = [W.served_scene(nt, seed * 64 + k) for k, nt in enumerate(_log_sizes(case["scenes"], 10_000, case["tri_hi"], 3))]
        for sc in setups:
            s.upload(sc["tris"], None, sc["materials"])
            bounds.append(W.scene_bounds(sc["tris"][:-4]))  # the soup, without floor and light
        counts = _log_sizes(case["queries"], 4096, case["ray_hi"], 4)
        s.hits, s.images, s.reqs, s.rays, at = _hits(sum(counts)), [], [], [], 0
        for q, n in enumerate(counts):
            lo, hi = bounds[q % len(bounds)]
            s.rays.append(_rays(n, lo, hi, seed * 64 + q))
            r = N.Request()
            r.kind, r.scene_id, r.nrays, r.trace_flags = N.REQ_TRACE, s.scenes[q % len(bounds)], n, N.REQ_DEVICE_BUFFERS
            r.rays, r.out = s.rays[-1].data_ptr(), s.hits.data_ptr() + 16 * at
            s.reqs.append(r)
            at += n
        for k in range(case["renders"]):
            img = np.zeros((256, 256, 4), np.float32)
            p = setups[k % len(setups)]["params"].copy()
            p["randomState"] = (seed + k) & 0xFFFF
            s.images.append(img)
            s.reqs.append(N.render_request(s.scenes[k % len(setups)], p, 256, 256, 1 + k % 4, out=img))
        s.server = N.Server(_ctx(), arena_bytes=1 << 30)
    return s


# ---------------- one pass ----------------

def _records(hits: torch.Tensor):
    """The hit records as the library wrote them: ids, and t, u, v."""
    return {"prim": hits[:, 0], "tuv": hits.view(torch.float32)[:, 1:]}


def _show(s, sid):
    ctx, npix = _ctx(), s.width * s.height
    ctx.accum_clear(s.accum.data_ptr(), npix)
    ctx.render(sid, s.params, s.width, s.height, s.spp, s.accum.data_ptr())
    ctx.resolve(s.accum.data_ptr(), npix, s.spp, s.shown.data_ptr())
    return {"accum": s.accum, "shown": s.shown}


def run(s):
    ctx = _ctx()
    if s.kind == "query":
        ctx.trace(s.sid, s.rays.data_ptr(), s.n, s.hits.data_ptr(), any_hit=s.any, fp32=s.fp32)
        return _records(s.hits)
    if s.kind == "batch":
        ctx.trace_batch(s.items)
        return _records(s.hits)
    if s.kind == "render":
        return _show(s, s.sid)
    if s.kind == "frame":
        sid = ctx.upload(s.tris, s.spheres, s.materials, models=s.models)
        out = _show(s, sid)
        ctx.release(sid)
        return out
    if s.kind == "load":
        sid = ctx.upload(s.tris, None, s.materials)
        ctx.trace(sid, s.rays.data_ptr(), s.n, s.hits.data_ptr())
        ctx.release(sid)
        return _records(s.hits)
    for r in s.reqs:
        s.server.submit(r)
    s.server.drain()
    return {**_records(s.hits), "images": s.images}


def work(case):
    kind = case["kind"]

    def query(tris, rays):  # rays in, hits out, and the triangles' vertices (few rays need few of them)
        return 48.0 * rays + 36.0 * min(tris, 64.0 * rays)

    def image(tris, w, h, spp):  # image out and shown, and the triangles its paths can need
        return 32.0 * w * h + 36.0 * min(tris, 64.0 * w * h * spp)

    mean = lambda lo, hi: (hi - lo) / math.log(hi / lo)  # noqa: E731  of a log-uniform size
    if kind == "query":
        b = query(case["tris"], case["rays"])
    elif kind == "batch":
        b = case["scenes"] * query(mean(1000, case["tri_hi"]), mean(4096, case["ray_hi"]))
    elif kind == "render":
        b = image(case["tris"], case["width"], case["height"], case["spp"])
    elif kind == "frame":
        b = 64.0 * case["tris"] + image(case["tris"], case["width"], case["height"], case["spp"])
    elif kind == "load":
        b = 64.0 * case["tris"] + query(case["tris"], case["rays"])
    else:
        b = case["queries"] * query(mean(10_000, case["tri_hi"]), mean(4096, case["ray_hi"]))
        b += case["renders"] * image(mean(10_000, case["tri_hi"]), 256, 256, 2)
    return {"bytes": b, "flops": 0.0}


# ---------------- double precision ----------------

def _brute_triangles(o, d, v0, v1, v2):
    """Nearest hit of each ray in double precision: (t, u, v), t = TMAX on a miss.  u and v weigh v1 and
    v2; a triangle seen within 1e-4 of edge-on counts as missed, as the reference's triangleHit has it.
    The candidate is found with products of ray and triangle coefficients (Pluecker coordinates), its
    t, u, v by Moller-Trumbore."""
    e1, e2 = v1 - v0, v2 - v0
    nrm = torch.linalg.cross(e1, e2)
    length = nrm.norm(dim=1)
    cu = torch.cat([e2, -torch.linalg.cross(e2, v0)], 1)
    cv = torch.cat([-e1, torch.linalg.cross(e1, v0)], 1)
    ct = torch.cat([nrm, -(nrm * v0).sum(1, keepdim=True)], 1)
    rows = max(1, min(len(o), (1 << 27) // max(1, len(v0))))
    best_t, best_i = [], []
    for a in range(0, len(o), rows):
        oo, dd = o[a:a + rows], d[a:a + rows]
        det = -(dd @ nrm.T)
        md = torch.cat([torch.linalg.cross(oo, dd), dd], 1)
        u, v = (md @ cu.T) / det, (md @ cv.T) / det
        t = (torch.cat([oo, torch.ones_like(oo[:, :1])], 1) @ ct.T) / det
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= TMIN) & (t <= TMAX) & (det.abs() >= 1e-4 * length)
        t = torch.where(ok, t, torch.full_like(t, float("inf")))
        m = t.min(dim=1)
        best_t.append(m.values)
        best_i.append(m.indices)
    bt, bi = torch.cat(best_t), torch.cat(best_i)
    hit = torch.isfinite(bt)
    e1, e2, s = e1[bi], e2[bi], o - v0[bi]
    p, q = torch.linalg.cross(d, e2), torch.linalg.cross(s, e1)
    det = (e1 * p).sum(1)
    z = torch.zeros_like(bt)
    return (torch.where(hit, (e2 * q).sum(1) / det, z + TMAX32), torch.where(hit, (s * p).sum(1) / det, z),
            torch.where(hit, (d * q).sum(1) / det, z))


TMAX32 = float(np.float32(TMAX))


def _brute_spheres(o, d, c, r):
    """Nearest sphere hit: (t, u, v); u, v are the reference's coordinates of the sphere's centre."""
    oc = o[:, None, :] - c[None]
    a, hb = (d * d).sum(1)[:, None], (oc * d[:, None, :]).sum(2)
    disc = hb * hb - a * ((oc * oc).sum(2) - r * r)
    sq = disc.clamp(min=0).sqrt()
    near, far = (-hb - sq) / a, (-hb + sq) / a
    inside = lambda x: (x >= TMIN) & (x <= TMAX)  # noqa: E731
    t = torch.where(inside(near), near, torch.where(inside(far), far, torch.full_like(far, float("inf"))))
    t = torch.where(disc >= 0, t, torch.full_like(t, float("inf")))
    m = t.min(dim=1)
    u = ((torch.atan2(-c[:, 2], c[:, 0]) + math.pi) / (2 * math.pi))[m.indices]
    v = (torch.acos(-c[:, 1]) / math.pi)[m.indices]
    return m.values, u, v


def exact(case, seed):
    """Closest hits by brute force.  An any-hit query may return any of a ray's hits, and a path traced
    image follows a chain of 32-bit random states: neither has a value in double precision."""
    if case["kind"] not in ("query", "load") or case.get("any") or case["tris"] * case["rays"] > 1e11:
        return None
    tris, sph, _ = _geometry(case, seed)
    lo, hi = W.scene_bounds(tris)
    rays = _rays(case["rays"], lo, hi, seed).double()
    o, d = rays[:, 0:3].contiguous(), rays[:, 4:7].contiguous()
    v = [torch.from_numpy(np.ascontiguousarray(tris[k][:, :3])).to(DEV).double() for k in ("v0", "v1", "v2")]
    t, a, b = _brute_triangles(o, d, *v)
    if len(sph):
        c = torch.from_numpy(np.ascontiguousarray(sph["center"][:, :3])).to(DEV).double()
        st, su, sv = _brute_spheres(o, d, c, torch.from_numpy(sph["radius"].copy()).to(DEV).double())
        nearer = st < t
        t, a, b = torch.where(nearer, st, t), torch.where(nearer, su, a), torch.where(nearer, sv, b)
    return {"prim": None, "tuv": torch.stack([t, a, b], 1)}
