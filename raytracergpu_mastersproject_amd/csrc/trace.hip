// trace.hip -- ray-query kernels (closest-hit / any-hit) over the resident wide BVH.
//
// Two schedules of one lane per ray:
//   persistent: a grid sized to fill every CU once; each wave takes chunks of rays
//     from global counters (WorkLines), one atomic per chunk (ChunkSchedule: smaller chunks for
//     the last rays).  When at least `refill` lanes of a wave are idle they take the
//     next rays of the wave's chunk (ballot + popcount + lane prefix), so finished
//     lanes are refilled while long rays keep traversing.
//   direct: one lane per ray (a launch-tuner candidate; the camera rays of renders).
// A launch of few rays, and the last rays of each persistent wave, are traced by a team of lanes per ray (team.hpp).
// Closest-hit launches over compressed nodes or by few lanes per ray leave marked the rays that need the exact nodes' order; a launch
// behind them traces these (launch_marked, launch_team).
// The batched variants run many scenes' ray batches in one launch.
#include <algorithm>
#include <cstdlib>
#include <vector>

#include "rt_internal.hpp"
#include "team.hpp"

namespace rtgpu {
namespace {

struct SceneView {
    const uint32_t *nodes;  // of the launch's layout
    const uint32_t *wide, *slot_ref;
    const LeafRecord *rec;
    const uint32_t *slot_prim;
    const rt_triangle *tris;  // world-space primitives, for the refined results
    const rt_sphere *sph;
    uint32_t nwide;
    Reach reach;
    __device__ LeafBoxes operator()() const { return LeafBoxes{wide, slot_ref}; }
};

struct TraceArgs {
    SceneView sc;  // sc.slot_prim == nullptr: hits carry the leaf slot instead of the primitive id
    const rt_ray *rays;
    rt_hit *hits;
    uint32_t *counts;
    uint32_t n;
    uint32_t refill;
    unsigned int *work;
    uint32_t leaf_weight;
    const uint32_t *n_dev;  // when set, the ray count is min(*n_dev, n)
    uint32_t limit;         // of a team of kLastTeam lanes; 0: the last rays stay with their lanes
};

// A counter slot's words: per line, 0 and 1 the launch's work counter, 2 and 3 that of the launch over the marked rays
// (which must be traced in the exact nodes' order, kRedo); word kMarks of the first line counts the marked
// rays, and the words from kMarkList of every line hold the indices of the first kMarkCap of them.
constexpr uint32_t kMarks = 4, kMarkList = 16, kMarkPerLine = kCounterStride - kMarkList, kMarkCap = kMarkPerLine * kCounterLines;

template <typename T> __device__ __forceinline__ uint32_t *mark_count(T *work) { return reinterpret_cast<uint32_t *>(work) + kMarks; }
template <typename T> __device__ __forceinline__ uint32_t *mark_entry(T *work, uint32_t k) {
    return reinterpret_cast<uint32_t *>(work) + (k / kMarkPerLine) * kCounterStride + kMarkList + k % kMarkPerLine;
}
// Rays are read once and hits written once per launch: non-temporal accesses keep them from
// displacing the BVH nodes and leaf records in L2 and the MALL (refined closest-hit query on
// 4M triangles: 5.10 against 5.13 ms).
typedef float nt_f4 __attribute__((ext_vector_type(4)));
typedef unsigned int nt_u4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void store_hit_nt(rt_hit *hits, uint32_t i, uint4 h) {
    const nt_u4 v = {h.x, h.y, h.z, h.w};
    __builtin_nontemporal_store(v, reinterpret_cast<nt_u4 *>(hits) + i);
}

// The ray's hit record says that it is to be traced again; g: its index in the launch.  `full`: the lane has seen the list full,
// and the count no longer matters (one counter for all would hold up a launch that marks every ray).
template <typename T> __device__ __forceinline__ void mark_ray(T *work, rt_hit *hits, uint32_t i, uint64_t g, bool &full) {
    store_hit_nt(hits, i, make_uint4(kRedo, 0u, 0u, 0u));
    if (full) return;
    uint32_t *n = mark_count(work);
    full = __hip_atomic_load(n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) > kMarkCap;
    if (full) return;
    const uint32_t k = atomicAdd(n, g > 0xFFFFFFFFull ? kMarkCap + 1u : 1u);
    if (k < kMarkCap) *mark_entry(work, k) = (uint32_t)g;
}

__device__ __forceinline__ void load_ray(const rt_ray *rays, uint32_t i, v3 &o, float &tmin, v3 &d, float &tmax) {
    const nt_f4 *p = reinterpret_cast<const nt_f4 *>(rays + i);
    const nt_f4 a = __builtin_nontemporal_load(p), b = __builtin_nontemporal_load(p + 1);
    o = v3{a.x, a.y, a.z};
    tmin = a.w;
    d = v3{b.x, b.y, b.z};
    tmax = b.w;
}

__device__ __forceinline__ void store_hit(const SceneView &sc, const Trav &t, rt_hit *hits, uint32_t *counts,
                                          uint32_t i) {
    uint4 h;
    if (t.bslot == kEmpty) h = make_uint4(RT_NO_HIT, __float_as_uint(t.bt), 0u, 0u);
    else h = make_uint4(sc.slot_prim ? sc.slot_prim[t.bslot] : t.bslot, __float_as_uint(t.bt), __float_as_uint(t.bu),
                        __float_as_uint(t.bv));
    store_hit_nt(hits, i, h);
    if (counts) reinterpret_cast<uint2 *>(counts)[i] = make_uint2(t.nbox, t.ntri);
}

template <int W, int S, bool ANY, bool COUNT>
__global__ __launch_bounds__(256) void k_trace_direct(TraceArgs a) {
    extern __shared__ uint32_t lds[];
    uint2 spill[kSpillCap];
    const StackMem m = stack_mem<S>(lds, spill);
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (a.n_dev ? min(*a.n_dev, a.n) : a.n)) return;
    v3 o, d;
    float tmin, tmax;
    load_ray(a.rays, i, o, tmin, d, tmax);
    Trav t;
    trav_init<W, ANY>(t, o, d, tmin, tmax, a.sc.nwide, a.sc.reach);
    bool exact = false;
    if constexpr (W == kQ4) {
        exact = needs_exact_nodes<ANY>(o, d, a.sc.reach.far_limit);
        if (exact) t.have = false;
    }
    trav_run<W, S, ANY, COUNT>(t, m, a.sc.nodes, a.sc.rec, a.sc, a.leaf_weight);
    if constexpr (W == kQ4) {
        if (exact || t.bslot == kRedo)
            walk_exact<S, ANY>(t, m, o, d, tmin, tmax, a.sc.nwide, a.sc.wide, a.sc.rec, a.sc, a.leaf_weight);
    }
    store_hit(a.sc, t, a.hits, a.counts, i);
}

// The stored result of a finished ray, with t, u, v of a hit refined in double as k_refine_hits
// refines them (the same operations on the same fp32 inputs, so the same bits).
__device__ __forceinline__ void store_refined(const SceneView &sc, const Trav &t, rt_hit *hits, uint32_t *counts,
                                              uint32_t i) {
    uint4 h;
    if (t.bslot == kEmpty) {
        h = make_uint4(RT_NO_HIT, __float_as_uint(t.bt), 0u, 0u);
    } else {
        const uint32_t prim = sc.slot_prim[t.bslot];
        float tt = t.bt, u = t.bu, v = t.bv;
        if (prim & RT_SPHERE_BIT) {
            const float4 c = *reinterpret_cast<const float4 *>(sc.sph + (prim & ~RT_SPHERE_BIT));
            const float r = sc.sph[prim & ~RT_SPHERE_BIT].radius;
            refine_sphere(dvec(c.x, c.y, c.z), (double)r, dvec(t.o.x, t.o.y, t.o.z), dvec(t.d.x, t.d.y, t.d.z), tt);
        } else {
            const float4 *tp = reinterpret_cast<const float4 *>(sc.tris + prim);
            const float4 p0 = tp[0], p1 = tp[1], p2 = tp[2];
            refine_triangle(dvec(p0.x, p0.y, p0.z), dvec(p1.x, p1.y, p1.z), dvec(p2.x, p2.y, p2.z),
                            dvec(t.o.x, t.o.y, t.o.z), dvec(t.d.x, t.d.y, t.d.z), tt, u, v);
        }
        h = make_uint4(prim, __float_as_uint(tt), __float_as_uint(u), __float_as_uint(v));
    }
    store_hit_nt(hits, i, h);
    if (counts) reinterpret_cast<uint2 *>(counts)[i] = make_uint2(t.nbox, t.ntri);
}

// A team's result, by the lane that holds it.
template <int T, bool REFINE>
__device__ __forceinline__ void store_team(const SceneView &sc, const TeamHit &h, v3 o, v3 d, rt_hit *hits, uint32_t i) {
    if (!h.owner && !(h.slot == kEmpty && threadIdx.x % T == 0)) return;
    Trav t;
    t.o = o;
    t.d = d;
    t.bt = h.t;
    t.bslot = h.slot;
    t.bu = h.u;
    t.bv = h.v;
    if constexpr (REFINE) store_refined(sc, t, hits, nullptr, i);
    else store_hit(sc, t, hits, nullptr, i);
}

// The last rays of a wave, one per lane in `live`, from their start: ray i of that lane, g in the launch.
template <int S, bool ANY, bool REFINE, typename W>
__device__ __forceinline__ void trace_last(unsigned long long live, const SceneView &sc, const rt_ray *rays,
                                           rt_hit *hits, uint32_t i, uint64_t g, W *work, void *lds, uint32_t limit) {
    const bool on = (threadIdx.x & 63u) / kLastTeam < (uint32_t)__popcll(live);
    v3 o, d;
    float tmin, tmax;
    load_ray(rays, i, o, tmin, d, tmax);
    const TeamHit h = team_trace<kLastTeam, ANY>(on, o, d, tmin, tmax, sc.wide, sc.nwide, sc.rec,
                                                 reinterpret_cast<uint2 *>(wave_lds<S>(lds)), limit, sc.reach);
    if (on && h.redo) {
        bool full = false;
        if (threadIdx.x % kLastTeam == 0) mark_ray(work, hits, i, g, full);
    } else if (on) {
        store_team<kLastTeam, REFINE>(sc, h, o, d, hits, i);
    }
}

// Ray i by a team of T lanes; every lane of the wave calls it.  A closest-hit ray that must be traced in the exact nodes' order:
// by the team's first lane with 32 lanes or more, whose launches are short; else it is marked for k_trace_marked,
// in whose waves 64 such rays are traced at once (350,000 rays from far away over 1 M triangles: 1,830 us by first lanes, 8 of 64 at
// work; 890 us with one lane per ray and no teams).
constexpr bool team_marks(uint32_t t) { return t <= 16u; }

template <int T, bool ANY, bool REFINE>
__device__ __forceinline__ void trace_by_team(bool live, const SceneView &sc, const rt_ray *rays, rt_hit *hits, uint32_t i,
                                              uint2 *stacks, uint32_t limit) {
    v3 o{0.0f, 0.0f, 0.0f}, d{0.0f, 0.0f, 0.0f};
    float tmin = 0.0f, tmax = 0.0f;
    if (live) load_ray(rays, i, o, tmin, d, tmax);
    // any hit: the teams read the exact nodes, and no order changes its result
    // teams have time for larger boxes, up to 1,000 extents: 1 M triangles from 900 extents 4,096 rays 34 us, by first lanes 230; 100,000 rays
    // 209, by the launch over the marked rays 394
    const float far_limit = sc.reach.far_limit + 1.5f * (sc.reach.far_limit - sc.reach.coord);
    const bool exact = !ANY && live && needs_exact_nodes<ANY>(o, d, far_limit);
    TeamHit h = team_trace<T, ANY>(live && !exact, o, d, tmin, tmax, sc.wide, sc.nwide, sc.rec, stacks, limit, sc.reach);
    bool stored = !live;
    if constexpr (!ANY) {
        const bool ordered = live && (exact || h.redo);
        if constexpr (team_marks(T)) {
            if (ordered && threadIdx.x % T == 0) hits[i].prim = kRedo;
            stored = stored || ordered;
        } else if (__ballot(ordered) != 0ull) {
            uint2 spill[kSpillCap];
            const TeamHit again = team_ordered<T, 16, ANY>(ordered, o, d, tmin, tmax, sc.wide, sc.nwide, sc.rec,
                                                           stack_mem<16>(stacks, spill), sc);
            if (ordered) h = again;
        }
    }
    if (!stored) store_team<T, REFINE>(sc, h, o, d, hits, i);
}

// One team of T lanes per ray, one wave per block, every ray at once: no work counter, no refill.
template <int T, bool ANY, bool REFINE> __global__ __launch_bounds__(64) void k_trace_team(TraceArgs a, uint32_t limit) {
    __shared__ uint2 stacks[64 / T * team_stack(T)];
    const uint32_t i = blockIdx.x * (64u / T) + threadIdx.x / T;
    trace_by_team<T, ANY, REFINE>(i < a.n, a.sc, a.rays, a.hits, i, stacks, limit);
}

// The rays that a launch of teams has marked, a lane per ray.
template <bool REFINE>
__device__ __forceinline__ void trace_marked(const SceneView &sc, const rt_ray *rays, rt_hit *hits, uint32_t i, const StackMem &m,
                                             uint32_t leaf_weight) {
    if (hits[i].prim != kRedo) return;
    v3 o, d;
    float tmin, tmax;
    load_ray(rays, i, o, tmin, d, tmax);
    Trav t;
    walk_exact<16, false>(t, m, o, d, tmin, tmax, sc.nwide, sc.wide, sc.rec, sc, leaf_weight);
    if constexpr (REFINE) store_refined(sc, t, hits, nullptr, i);
    else store_hit(sc, t, hits, nullptr, i);
}

template <bool REFINE> __global__ __launch_bounds__(128) void k_trace_marked(TraceArgs a) {
    extern __shared__ uint32_t lds[];
    uint2 spill[kSpillCap];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < a.n) trace_marked<REFINE>(a.sc, a.rays, a.hits, i, stack_mem<16>(lds, spill), a.leaf_weight);
}

constexpr uint32_t kNoRay = ~0u;

// Whether fp32 results wait for the refill too.  16.8 M rays on compressed nodes: closest hit 3,777 -> 3,300 us, any hit
// 3,452 -> 3,090; exact width-4 nodes with counts, 4 M rays 947 -> 906.  Width 2 is slower with it (1,116 -> 1,180 us)
// and width 8's any hit too (1,052 -> 1,078).
template <int W> constexpr bool kDefer = W == kQ4 || W == 4;

// Work counters at most.  Width 2's kernel without the refinement has one (fixed here: as an argument it cost as much as 32): with 32,
// launches from 2 M rays are slower than they were before (fp32 closest hits over 1 M triangles, 32 counters | one: 1 M rays 736 | 808 us,
// 1.4 M 874 | 906, 2 M 1,090 | 1,005, 4 M 1,754 | 1,639, 12 M 4,568 | 3,738).
template <int W, bool REFINE> constexpr uint32_t kLines = W == 2 && !REFINE ? 1u : kCounterLines;

// REFINE: store each hit with t, u, v refined in double (store_refined) instead of the fp32 values.
// LAST: the wave's last rays go on with teams of lanes (trace_last).
// MARKED: only the rays that the launch before has marked (mark_ray).
template <int W, int S, bool ANY, bool COUNT, bool REFINE, bool LAST, bool MARKED>
__global__ __launch_bounds__(256, W == kQ4 ? 5 : 1) void k_trace_persistent(TraceArgs a) {
    extern __shared__ uint32_t lds[];
    uint2 spill[kSpillCap];
    const StackMem m = stack_mem<S>(lds, spill);
    const uint32_t lane = threadIdx.x & 63u;
    const unsigned long long lt = lane ? (~0ull >> (64u - lane)) : 0ull;
    uint32_t rid = kNoRay;  // a launch has fewer rays than this
    // A finished ray's result is stored at the wave's next refill (or at the end), with those of the lanes that finished
    // since the last one: storing, and refining in double, as each lane finishes would run that code on almost every
    // iteration.  See kDefer for fp32 results.
    uint32_t done = kNoRay;
    bool exhausted = false;
    uint32_t q_next = 0, q_end = 0;  // the wave's current chunk of ray indices (wave-uniform)
    uint32_t n = a.n_dev ? min(*a.n_dev, a.n) : a.n;
    bool listed = false;  // the marked rays' indices are in the list
    unsigned int *work = a.work;
    if constexpr (MARKED) {
        const uint32_t marks = *mark_count(a.work);
        if (marks == 0u) return;
        listed = marks <= kMarkCap;
        if (listed) n = marks;
        work += 2;
    }
    const uint32_t wpb = blockDim.x / 64u;
    const ChunkSchedule<uint32_t> sched(n, gridDim.x * wpb);
    WorkLines lines(blockIdx.x * wpb + __builtin_amdgcn_readfirstlane(threadIdx.x / 64u), gridDim.x * wpb,
                    kLines<W, REFINE>);
    Trav t;
    t.have = false;
    t.top = 0;
    bool full = false;  // mark_ray's
    const auto store = [&](uint32_t i) {
        if (W == kQ4 && !ANY && t.bslot == kRedo) mark_ray(a.work, a.hits, i, i, full);
        else if constexpr (REFINE) store_refined(a.sc, t, a.hits, a.counts, i);
        else store_hit(a.sc, t, a.hits, a.counts, i);
    };
    for (;;) {
        const unsigned long long idle = __ballot(rid == kNoRay);
        const uint32_t nidle = (uint32_t)__popcll(idle);
        if (!exhausted && nidle >= a.refill) {
            if (done != kNoRay) {
                store(done);
                done = kNoRay;
            }
            while (q_next == q_end && !exhausted) {  // one atomic per chunk
                const int leader = __ffsll((unsigned long long)idle) - 1;
                uint32_t base = 0;
                if ((int)lane == leader) base = atomicAdd(lines.counter(work), 1u);
                base = (uint32_t)__shfl((int)base, leader);
                uint64_t lo, hi;
                if (sched.range((uint32_t)lines.item(base), lo, hi)) { q_next = (uint32_t)lo; q_end = (uint32_t)hi; }
                else exhausted = !lines.next();
            }
            if (!exhausted) {
                const uint32_t take = min(nidle, q_end - q_next);
                const uint32_t r = (uint32_t)__popcll(idle & lt);
                if (rid == kNoRay && r < take) {
                    rid = q_next + r;
                    if constexpr (MARKED) {
                        if (listed) rid = *mark_entry(a.work, rid);
                        else if (a.hits[rid].prim != kRedo) rid = kNoRay;
                    }
                    if (!MARKED || rid != kNoRay) {
                        v3 o, d;
                        float tmin, tmax;
                        load_ray(a.rays, rid, o, tmin, d, tmax);
                        if (!walk_init<W, S, ANY>(t, m, o, d, tmin, tmax, a.sc.nwide, a.sc.reach, a.sc.rec, a.sc, a.leaf_weight)) {
                            mark_ray(a.work, a.hits, rid, rid, full);
                            rid = kNoRay;
                        }
                    }
                }
                q_next += take;
            }
        }
        const unsigned long long live = __ballot(rid != kNoRay);
        if (live == 0ull) {  // every lane idle
            if (exhausted) break;  // and the queue is drained
            continue;  // no ray of those taken was started
        }
        if (LAST && exhausted && a.limit && (uint32_t)__popcll(live) <= kLastRays) break;
        const bool on_node = rid != kNoRay && at_node(t), on_leaf = rid != kNoRay && at_leaf(t);
        if (choose_leaf_phase(on_node, on_leaf, a.leaf_weight)) {
            if (on_leaf) leaf_step<W, S, ANY, COUNT>(t, m, a.sc.rec, a.sc);
        } else {
            if (on_node) walk_node<W, S, ANY, COUNT>(t, m, a.sc.nodes);
        }
        walk_pop<W, S, ANY>(t, m);
        if (rid != kNoRay && trav_done(t)) {
            if constexpr (REFINE || kDefer<W>) done = rid;
            else store(rid);
            rid = kNoRay;
        }
    }
    if (done != kNoRay) store(done);
    if constexpr (LAST) {
        const unsigned long long live = __ballot(rid != kNoRay);
        if (live == 0ull) return;
        const uint32_t i = (uint32_t)__shfl((int)rid, (int)last_ray_lane<kLastTeam>(live));
        trace_last<S, ANY, REFINE>(live, a.sc, a.rays, a.hits, i, i, a.work, lds, a.limit);
    }
}

// ---------------------------------------------------------------------------
// Refined results: t, u, v of every hit recomputed in double precision from the hit
// primitive's stored fp32 geometry and the fp32 ray (refine_triangle / refine_sphere).
// The primitive id, decided by the fp32 traversal, is untouched; so is a result whose
// recomputation has no solution in double (a zero determinant, a negative discriminant).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void refine_one(const rt_triangle *tris, const rt_sphere *sph, const rt_ray *rays,
                                           rt_hit *hits, uint32_t i) {
    uint4 *hp = reinterpret_cast<uint4 *>(hits) + i;
    uint4 h = *hp;
    if (h.x == RT_NO_HIT) return;
    v3 o, d;
    float tmin, tmax;
    load_ray(rays, i, o, tmin, d, tmax);
    float t = __uint_as_float(h.y), u = __uint_as_float(h.z), v = __uint_as_float(h.w);
    bool ok;
    if (h.x & RT_SPHERE_BIT) {
        const float4 c = *reinterpret_cast<const float4 *>(sph + (h.x & ~RT_SPHERE_BIT));
        const float r = sph[h.x & ~RT_SPHERE_BIT].radius;
        ok = refine_sphere(dvec(c.x, c.y, c.z), (double)r, dvec(o.x, o.y, o.z), dvec(d.x, d.y, d.z), t);
    } else {
        const float4 *tp = reinterpret_cast<const float4 *>(tris + h.x);
        const float4 a = tp[0], b = tp[1], c = tp[2];
        ok = refine_triangle(dvec(a.x, a.y, a.z), dvec(b.x, b.y, b.z), dvec(c.x, c.y, c.z), dvec(o.x, o.y, o.z),
                             dvec(d.x, d.y, d.z), t, u, v);
    }
    if (ok) *hp = make_uint4(h.x, __float_as_uint(t), __float_as_uint(u), __float_as_uint(v));
}

__global__ __launch_bounds__(256) void k_refine_hits(const rt_ray *rays, rt_hit *hits, uint32_t n,
                                                     const rt_triangle *tris, const rt_sphere *sph) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) refine_one(tris, sph, rays, hits, i);
}

// ---------------------------------------------------------------------------
// batched: many (scene, rays) items in one persistent launch.  A global ray
// index runs over the concatenation of all items; item boundaries are found by
// binary search in an exclusive prefix of item sizes held in the argument block.
// ---------------------------------------------------------------------------
struct BatchItemDev {
    SceneView sc;
    const rt_ray *rays;
    rt_hit *hits;
    uint64_t first;  // global index of the item's first ray
};

struct BatchArgs {
    const BatchItemDev *items;
    uint32_t nitems;
    uint32_t refill;
    uint64_t total;
    unsigned long long *work;
    uint32_t leaf_weight;
    uint32_t limit;  // as in TraceArgs
};

// the last item in [lo, hi) whose first ray is at or before g
__device__ __forceinline__ uint32_t find_item(const BatchItemDev *items, uint32_t lo, uint32_t hi, uint64_t g) {
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (items[mid].first <= g) lo = mid;
        else hi = mid;
    }
    return lo;
}

// REFINE: store each hit with t, u, v refined in double (store_refined); LAST, MARKED: as in k_trace_persistent.
template <int W, int S, bool ANY, bool REFINE, bool LAST, bool MARKED>
__global__ __launch_bounds__(256, W == kQ4 ? 5 : 1) void k_trace_batch(BatchArgs a) {
    extern __shared__ uint32_t lds[];
    uint2 spill[kSpillCap];
    const StackMem m = stack_mem<S>(lds, spill);
    const uint32_t lane = threadIdx.x & 63u;
    const unsigned long long lt = lane ? (~0ull >> (64u - lane)) : 0ull;
    bool active = false, exhausted = false;
    bool pending = false;  // a finished ray (item, local) whose result waits for the wave's next refill
    uint32_t item = 0, local = 0;
    uint64_t q_next = 0, q_end = 0;  // the wave's current chunk of global ray indices
    uint32_t c_lo = 0, c_hi = 1;     // the items the chunk's rays belong to: [c_lo, c_hi)
    // the lane's scene, kept in registers: a table load per traversal step would add its
    // latency to every step
    const uint32_t *nodes = nullptr;
    const LeafRecord *rec = nullptr;
    uint64_t total = a.total;
    bool listed = false;
    unsigned long long *work = a.work;
    if constexpr (MARKED) {
        const uint32_t marks = *mark_count(a.work);
        if (marks == 0u) return;
        listed = marks <= kMarkCap;
        if (listed) total = marks;
        work += 1;
    }
    const uint32_t wpb = blockDim.x / 64u;
    const ChunkSchedule<uint64_t> sched(total, gridDim.x * wpb);
    WorkLines lines(blockIdx.x * wpb + __builtin_amdgcn_readfirstlane(threadIdx.x / 64u), gridDim.x * wpb);
    Trav t;
    t.have = false;
    t.top = 0;
    bool full = false;
    const auto store = [&]() {
        const BatchItemDev &it = a.items[item];
        if (W == kQ4 && !ANY && t.bslot == kRedo) mark_ray(a.work, it.hits, local, it.first + local, full);
        else if constexpr (REFINE) store_refined(it.sc, t, it.hits, nullptr, local);
        else store_hit(it.sc, t, it.hits, nullptr, local);
    };
    for (;;) {
        const unsigned long long idle = __ballot(!active);
        const uint32_t nidle = (uint32_t)__popcll(idle);
        if (!exhausted && nidle >= a.refill) {
            if (pending) {  // as in k_trace_persistent: the lanes that finished store together
                store();
                pending = false;
            }
            while (q_next == q_end && !exhausted) {
                const int leader = __ffsll((unsigned long long)idle) - 1;
                unsigned long long base = 0;
                if ((int)lane == leader) base = atomicAdd(lines.counter(work), 1ull);
                base = __shfl(base, leader);
                uint64_t lo, hi;
                if (!sched.range(lines.item(base), lo, hi)) {
                    exhausted = !lines.next();
                } else {  // chunks are short: usually one item, found once per chunk
                    q_next = lo;
                    q_end = hi;
                    c_lo = listed ? 0u : find_item(a.items, 0u, a.nitems, q_next);
                    c_hi = listed ? a.nitems : find_item(a.items, c_lo, a.nitems, q_end - 1u) + 1u;
                }
            }
            const uint32_t take = exhausted ? 0u : (uint32_t)min((uint64_t)nidle, q_end - q_next);
            const uint32_t r = (uint32_t)__popcll(idle & lt);
            uint64_t g = q_next + r;
            q_next += take;
            if (!active && r < take) {
                if (MARKED && listed) g = *mark_entry(a.work, (uint32_t)g);
                item = find_item(a.items, c_lo, c_hi, g);
                local = (uint32_t)(g - a.items[item].first);
                if (!MARKED || listed || a.items[item].hits[local].prim == kRedo) {
                    nodes = MARKED ? a.items[item].sc.wide : a.items[item].sc.nodes;
                    rec = a.items[item].sc.rec;
                    v3 o, d;
                    float tmin, tmax;
                    load_ray(a.items[item].rays, local, o, tmin, d, tmax);
                    active = walk_init<W, S, ANY>(t, m, o, d, tmin, tmax, a.items[item].sc.nwide, a.items[item].sc.reach, rec,
                                                  a.items[item].sc, a.leaf_weight);
                    if (!active) mark_ray(a.work, a.items[item].hits, local, g, full);
                }
            }
        }
        const unsigned long long live = __ballot(active);
        if (live == 0ull) {
            if (exhausted) break;
            continue;
        }
        if (LAST && exhausted && a.limit && (uint32_t)__popcll(live) <= kLastRays) break;
        const bool on_node = active && at_node(t), on_leaf = active && at_leaf(t);
        if (choose_leaf_phase(on_node, on_leaf, a.leaf_weight)) {
            if (on_leaf) leaf_step<W, S, ANY, false>(t, m, rec, a.items[item].sc);
        } else {
            if (on_node) walk_node<W, S, ANY, false>(t, m, nodes);
        }
        walk_pop<W, S, ANY>(t, m);
        if (active && trav_done(t)) {
            if constexpr (REFINE || kDefer<W>) pending = true;
            else store();
            active = false;
        }
    }
    if (pending) store();
    if constexpr (LAST) {
        const unsigned long long live = __ballot(active);
        if (live == 0ull) return;
        const int from = (int)last_ray_lane<kLastTeam>(live);
        const BatchItemDev &it = a.items[(uint32_t)__shfl((int)item, from)];
        const uint32_t i = (uint32_t)__shfl((int)local, from);
        trace_last<S, ANY, REFINE>(live, it.sc, it.rays, it.hits, i, it.first + i, a.work, lds, a.limit);
    }
}

// The same for few rays in all: a team of T lanes per ray, every ray at once.
template <int T, bool ANY, bool REFINE>
__global__ __launch_bounds__(64) void k_trace_team_batch(BatchArgs a, uint32_t limit) {
    __shared__ uint2 stacks[64 / T * team_stack(T)];
    const uint32_t g = blockIdx.x * (64u / T) + threadIdx.x / T;
    const BatchItemDev &it = a.items[find_item(a.items, 0u, a.nitems, min((uint64_t)g, a.total - 1u))];
    trace_by_team<T, ANY, REFINE>(g < a.total, it.sc, it.rays, it.hits, (uint32_t)(g - it.first), stacks, limit);
}

template <bool REFINE> __global__ __launch_bounds__(128) void k_trace_marked_batch(BatchArgs a) {
    extern __shared__ uint32_t lds[];
    uint2 spill[kSpillCap];
    const uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= a.total) return;
    const BatchItemDev &it = a.items[find_item(a.items, 0u, a.nitems, g)];
    trace_marked<REFINE>(it.sc, it.rays, it.hits, (uint32_t)(g - it.first), stack_mem<16>(lds, spill), a.leaf_weight);
}

template <int T, bool ANY, bool REFINE> void *team_kernel_t(bool batch) {
    return batch ? (void *)k_trace_team_batch<T, ANY, REFINE> : (void *)k_trace_team<T, ANY, REFINE>;
}
template <int T> void *team_kernel_t(bool any, bool refine, bool batch) {
    if (any) return refine ? team_kernel_t<T, true, true>(batch) : team_kernel_t<T, true, false>(batch);
    return refine ? team_kernel_t<T, false, true>(batch) : team_kernel_t<T, false, false>(batch);
}
void *team_kernel(uint32_t t, bool any, bool refine, bool batch) {
    switch (t) {
        case 8: return team_kernel_t<8>(any, refine, batch);
        case 16: return team_kernel_t<16>(any, refine, batch);
        case 32: return team_kernel_t<32>(any, refine, batch);
        default: return team_kernel_t<64>(any, refine, batch);
    }
}

__global__ void k_zero_counter(unsigned int *c) {
    if (threadIdx.x < kCounterLines) reinterpret_cast<uint4 *>(c + threadIdx.x * kCounterStride)[0] = make_uint4(0u, 0u, 0u, 0u);
    if (threadIdx.x == 0) c[kMarks] = 0u;
}

SceneView view_of(const Scene &sc) {
    return SceneView{sc.nodes(), sc.wide.as<uint32_t>(), sc.slot_ref.as<uint32_t>(), sc.records.as<LeafRecord>(), sc.slot_prim.as<uint32_t>(),
                     sc.tris.as<rt_triangle>(), sc.spheres.as<rt_sphere>(), sc.nwide, sc.reach};
}

template <int W, int S> struct Kernels {
    template <bool ANY> static void *direct(bool count) {
        if constexpr (W == kQ4) return (void *)k_trace_direct<W, S, ANY, false>;
        else return count ? (void *)k_trace_direct<W, S, ANY, true> : (void *)k_trace_direct<W, S, ANY, false>;
    }
    template <bool ANY, bool REFINE> static void *persistent(bool count, bool last) {
        if constexpr (W == kQ4)
            return last ? (void *)k_trace_persistent<W, S, ANY, false, REFINE, true, false>
                        : (void *)k_trace_persistent<W, S, ANY, false, REFINE, false, false>;
        else return count ? (void *)k_trace_persistent<W, S, ANY, true, REFINE, false, false>
                     : (void *)k_trace_persistent<W, S, ANY, false, REFINE, false, false>;
    }
    template <bool ANY, bool REFINE> static void *batch(bool last) {
        if constexpr (W == kQ4)
            if (last) return (void *)k_trace_batch<W, S, ANY, REFINE, true, false>;
        return (void *)k_trace_batch<W, S, ANY, REFINE, false, false>;
    }
    static void *get(int which, bool any, bool count, bool last) {
        if (which == 0) return any ? direct<true>(count) : direct<false>(count);
        if (which == 1) return any ? persistent<true, false>(count, last) : persistent<false, false>(count, last);
        if (which == 3) return any ? persistent<true, true>(count, last) : persistent<false, true>(count, last);
        if (which == 2) return any ? batch<true, false>(last) : batch<false, false>(last);
        return any ? batch<true, true>(last) : batch<false, true>(last);
    }
};

template <int W> void *pick(uint32_t s, int which, bool any, bool count, bool last) {
    switch (s) {
        case 4: return Kernels<W, 4>::get(which, any, count, last);
        case 16: return Kernels<W, 16>::get(which, any, count, last);
        default: return Kernels<W, 8>::get(which, any, count, last);
    }
}

// layout: Scene::layout (compressed nodes never count); which: 0 one lane per ray, 1 persistent, 2 persistent over many
// scenes (never counts), 3 persistent storing refined hits, 4 persistent over many scenes storing refined hits; last:
// the waves' last rays by teams (compressed nodes only)
void *pick_kernel(uint32_t layout, uint32_t s, int which, bool any, bool count, bool last) {
    switch (layout) {
        case kQ4: return pick<kQ4>(s, which, any, count, last);
        case 2: return pick<2>(s, which, any, count, last);
        case 8: return pick<8>(s, which, any, count, last);
        default: return pick<4>(s, which, any, count, last);
    }
}

// Whether a persistent launch of n rays ends with teams.  Up to 16,384 rays per CU: 2 M rays on 1 M triangles 530 us and
// 549 without, 4 M 865 and 874.  Beyond, the share of the end is small and the larger kernel's main loop costs about
// 1 %: 8 M rays 1,482 and 1,467, 16 M on 4 M triangles 3,444 and 3,387.
bool ends_with_teams(const rt_context *ctx, uint64_t n) { return n <= 16384ull * (uint64_t)ctx->num_cus; }

uint32_t persistent_grid(rt_context *ctx, const void *kernel, uint32_t block, size_t lds) {
    int per_cu = 0;
    RT_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, (int)block, lds));
    return (uint32_t)std::max(1, per_cu) * (uint32_t)ctx->num_cus;
}

// After a launch for closest hits: the rays that it has marked, if any, over the exact nodes.  An empty launch takes 3 us.
template <class A> void launch_marked(rt_context *ctx, A &a, void *k, uint64_t n, hipStream_t stream) {
    constexpr uint32_t block = 128, lds_stack = 16;  // holds any stack that the launch before could
    const size_t lds = stack_lds_bytes(lds_stack, block);
    const uint32_t grid = (uint32_t)std::min<uint64_t>(persistent_grid(ctx, k, block, lds), (n + block - 1) / block);
    void *args[] = {&a};
    RT_HIP(hipLaunchKernel(k, dim3(grid), dim3(block), args, lds, stream));
}
void launch_marked(rt_context *ctx, TraceArgs a, bool refine, hipStream_t stream) {
    a.sc.nodes = a.sc.wide;
    launch_marked(ctx, a, refine ? (void *)k_trace_persistent<4, 16, false, false, true, false, true>
                                 : (void *)k_trace_persistent<4, 16, false, false, false, false, true>, a.n, stream);
}
void launch_marked(rt_context *ctx, BatchArgs a, bool refine, hipStream_t stream) {
    launch_marked(ctx, a, refine ? (void *)k_trace_batch<4, 16, false, true, false, true>
                                 : (void *)k_trace_batch<4, 16, false, false, false, true>, a.total, stream);
}


// A launch of a team per ray, and one over the rays that it has marked.
template <class A>
void launch_team(uint32_t team, bool any, bool refine, bool batch, A &a, uint64_t n, uint32_t stack_bound, hipStream_t stream) {
    uint32_t limit = team_limit(team, stack_bound);
    void *args[] = {&a, &limit};
    RT_HIP(hipLaunchKernel(team_kernel(team, any, refine, batch), dim3(((uint32_t)n + 64u / team - 1) / (64u / team)), dim3(64), args, 0,
                           stream));
    if (any || !team_marks(team)) return;
    void *k = batch ? (refine ? (void *)k_trace_marked_batch<true> : (void *)k_trace_marked_batch<false>)
                    : (refine ? (void *)k_trace_marked<true> : (void *)k_trace_marked<false>);
    RT_HIP(hipLaunchKernel(k, dim3(((uint32_t)n + 127u) / 128u), dim3(128), args, stack_lds_bytes(16, 128), stream));
}

}  // namespace

void check_stack(const Scene &sc, const LaunchCfg &c) {
    if (sc.stack_bound > c.lds_stack + kSpillCap)
        throw Error(RT_ERR_OVERFLOW, "traversal stack bound " + std::to_string(sc.stack_bound) +
                                         " exceeds the kernel's capacity " + std::to_string(c.lds_stack + kSpillCap));
}

LaunchCfg resolve_cfg(const rt_context *ctx, const Scene &sc, const rt_launch_config *cfg, bool any) {
    (void)ctx;
    LaunchCfg c = sc.has_tuned ? (any ? sc.tuned_any : sc.tuned_closest) : LaunchCfg{};
    if (cfg) {
        if (cfg->block) c.block = cfg->block;
        if (cfg->lds_stack) c.lds_stack = cfg->lds_stack;
        c.persistent = cfg->persistent;
        c.teams = cfg->persistent != 0u;
        if (cfg->refill) c.refill = cfg->refill;
    }
    RT_REQUIRE(c.block == 64 || c.block == 128 || c.block == 256, "block must be 64, 128 or 256");
    RT_REQUIRE(c.lds_stack == 4 || c.lds_stack == 8 || c.lds_stack == 16, "lds_stack must be 4, 8 or 16");
    c.refill = std::min<uint32_t>(std::max<uint32_t>(c.refill, 1u), 64u);
    if (const char *lw = std::getenv("RTGPU_LEAF_WEIGHT")) c.leaf_weight = (uint32_t)std::max(1, std::atoi(lw));
    if (const char *sm = std::getenv("RTGPU_SHADE_MIN")) c.shade_min = (uint32_t)std::min(64, std::max(1, std::atoi(sm)));
    return c;
}

// Lanes per ray of a plain launch of n rays; 0: one lane per ray.  The lines lie where the times
// cross (us; 256 CUs; closest hit, 1 M triangles unless stated):
//   24 rays per CU     a wave per ray, every wave resident: 4,096 rays 21.4 with 64 lanes, 22.6 with 32
//   128 rays per CU    16,384 rays 33.0 with 32 lanes, 42.5 with 16; 65,536 rays 80.1 and 75.0
//   1,024 rays per CU  131,072 rays 118 with 16 lanes, 128 with 8; 400,000 rays 287 and 281
//   1,536 rays per CU  400,000 rays 281 with 8 lanes, 296 with one; 524,288 rays 348 and 304
//                      (4 M triangles 333 and 376, 427 and 392; 1,024 triangles 82 and 89, 102 and 93)
// Four lanes per ray were slower than eight at every size.  A launch that counts tests per ray keeps
// one lane per ray (its counts are those of the ordered traversal), as do the widths 2 and 8, a
// caller's one-lane-per-ray configuration, and a tree too deep for the team's stack.  A tuned configuration says
// how the larger launches run: that one lane per ray was the best shape at the tuner's size says nothing about small ones.
static uint32_t team_size(const rt_context *ctx, uint32_t layout, uint32_t stack_bound, uint64_t n, const LaunchCfg &c) {
    if (layout != kQ4 || !c.teams) return 0;
    const uint64_t cus = (uint64_t)ctx->num_cus;
    if (n > 1536u * cus) return 0;
    const uint32_t t = n <= 24u * cus ? 64u : n <= 128u * cus ? 32u : n <= 1024u * cus ? 16u : 8u;
    return team_limit(t, stack_bound) ? t : 0u;
}

void launch_trace(rt_context *ctx, const Scene &sc, const rt_ray *rays, uint32_t n, rt_hit *hits, uint32_t *counts,
                  uint32_t flags, const LaunchCfg &c, hipStream_t stream) {
    if (n == 0) return;
    RT_REQUIRE(rays && hits, "rays/hits must be device pointers");
    check_stack(sc, c);
    const bool any = (flags & RT_TRACE_ANY) != 0, refine = (flags & RT_TRACE_FP32) == 0;
    // Persistent launches refine in the kernel, at each wave's refills: a separate pass reads every ray and hit again
    // (16.8 M any-hit rays 3,390 us with it, 3,295 without; 1 M on 1,024 triangles 106 and 100).  Width 8's any hit, with
    // its larger kernel, keeps the pass (4 M rays 1,093 us, 1,118 in the kernel).
    // So do large any-hit launches of width 2 (12 M rays over 1 M triangles 4,382 us, 3,868 with the pass and the kernel without
    // the refinement; 1.4 M 797 and 913).
    const bool pass = any && (sc.width == 8 || (sc.width == 2 && n > 6144ull * (uint64_t)ctx->num_cus));
    const bool refine_in_kernel = refine && c.persistent && !pass;
    TraceArgs a{view_of(sc), rays, hits, counts, n, c.refill, nullptr, c.leaf_weight, nullptr, team_limit(kLastTeam, sc.stack_bound)};
    uint32_t layout = sc.layout();
    if (counts) {  // the counts are those of the exact boxes
        layout = sc.width;
        a.sc.nodes = a.sc.wide;
    }
    const size_t lds = stack_lds_bytes(c.lds_stack, c.block);
    if (const uint32_t team = counts ? 0u : team_size(ctx, layout, sc.stack_bound, n, c)) {
        launch_team(team, any, refine, false, a, n, sc.stack_bound, stream);
        RT_HIP(hipGetLastError());
        return;
    }
    if (!c.persistent) {
        void *k = pick_kernel(layout, c.lds_stack, 0, any, counts != nullptr, false);
        const uint32_t grid = (uint32_t)(((uint64_t)n + c.block - 1) / c.block);
        void *args[] = {&a};
        RT_HIP(hipLaunchKernel(k, dim3(grid), dim3(c.block), args, lds, stream));
    } else {
        a.work = ctx->counter_slot();
        k_zero_counter<<<1, 64, 0, stream>>>(a.work);
        void *k = pick_kernel(layout, c.lds_stack, refine_in_kernel ? 3 : 1, any, counts != nullptr, ends_with_teams(ctx, n));
        // no more lanes than rays: a small batch would otherwise launch the whole device's worth of
        // waves, nearly all of which find no chunk and exit
        const uint32_t grid = (uint32_t)std::min<uint64_t>(persistent_grid(ctx, k, c.block, lds),
                                                           ((uint64_t)n + c.block - 1) / c.block);
        void *args[] = {&a};
        RT_HIP(hipLaunchKernel(k, dim3(grid), dim3(c.block), args, lds, stream));
        if (layout == kQ4 && !any) launch_marked(ctx, a, refine, stream);
    }
    if (refine && !refine_in_kernel)
        k_refine_hits<<<(uint32_t)(((uint64_t)n + 255u) / 256u), 256, 0, stream>>>(rays, hits, n, a.sc.tris, a.sc.sph);
    RT_HIP(hipGetLastError());
}

void launch_trace_queue(rt_context *ctx, const Scene &sc, const rt_ray *rays, uint32_t n_max, const uint32_t *n_dev,
                        rt_hit *hits, const LaunchCfg &c, hipStream_t stream) {
    if (n_max == 0) return;
    check_stack(sc, c);
    SceneView v = view_of(sc);
    v.slot_prim = nullptr;  // hits carry leaf slots
    TraceArgs a{v, rays, hits, nullptr, n_max, c.refill, ctx->counter_slot(), c.leaf_weight, n_dev,
                team_limit(kLastTeam, sc.stack_bound)};
    const size_t lds = stack_lds_bytes(c.lds_stack, c.block);
    // camera rays of a small image: a team per ray (65,536 pixels on 200 k triangles: 130 us less per frame)
    if (const uint32_t team = n_dev || n_max > 1024u * (uint64_t)ctx->num_cus ? 0u : team_size(ctx, sc.layout(), sc.stack_bound, n_max, c)) {
        launch_team(team, false, false, false, a, n_max, sc.stack_bound, stream);
        RT_HIP(hipGetLastError());
        return;
    }
    if (!n_dev) {
        // A count known on the host means camera rays: neighbouring lanes trace neighbouring
        // pixels, and about two thirds of them leave the scene at once.  One thread per ray lets
        // such waves retire and new ones start (0.45 vs 0.69 ms for the 1080p frame's primaries);
        // refilling lanes in a persistent wave mixes rays at different depths instead.
        void *k = pick_kernel(sc.layout(), c.lds_stack, 0, false, false, false);
        void *args[] = {&a};
        RT_HIP(hipLaunchKernel(k, dim3((uint32_t)(((uint64_t)n_max + c.block - 1) / c.block)), dim3(c.block), args, lds, stream));
        RT_HIP(hipGetLastError());
        return;
    }
    k_zero_counter<<<1, 64, 0, stream>>>(a.work);
    void *k = pick_kernel(sc.layout(), c.lds_stack, 1, false, false, ends_with_teams(ctx, n_max));
    const uint32_t grid = persistent_grid(ctx, k, c.block, lds);
    void *args[] = {&a};
    RT_HIP(hipLaunchKernel(k, dim3(grid), dim3(c.block), args, lds, stream));
    if (sc.layout() == kQ4) launch_marked(ctx, a, false, stream);
    RT_HIP(hipGetLastError());
}

void launch_trace_items(rt_context *ctx, const std::vector<TraceItem> &items, uint32_t flags, const LaunchCfg &c,
                        hipStream_t stream) {
    for (const TraceItem &it : items) {  // before the first launch: a bad item leaves every hit buffer as it was
        RT_REQUIRE(it.n == 0 || (it.rays && it.hits), "batch item with NULL rays/hits");
        check_stack(*it.sc, c);
    }
    // one launch per node layout present, each over that layout's items in order
    for (uint32_t layout : {2u, 4u, 8u, (uint32_t)kQ4}) {
        std::vector<BatchItemDev> hv;
        uint64_t total = 0;
        uint32_t bound = 0;
        for (const TraceItem &it : items) {
            if (it.sc->layout() != layout) continue;
            hv.push_back(BatchItemDev{view_of(*it.sc), it.rays, it.hits, total});
            total += it.n;
            bound = std::max(bound, it.sc->stack_bound);
        }
        if (total == 0) continue;
        int slot = 0;
        void *table = ctx->tables.stage(hv.data(), sizeof(BatchItemDev) * hv.size(), stream, slot);
        BatchArgs a{static_cast<const BatchItemDev *>(table), (uint32_t)hv.size(), c.refill, total, nullptr,
                    c.leaf_weight, team_limit(kLastTeam, bound)};
        const bool any = (flags & RT_TRACE_ANY) != 0, refine = (flags & RT_TRACE_FP32) == 0;
        if (const uint32_t team = team_size(ctx, layout, bound, total, c)) {  // as for one scene
            launch_team(team, any, refine, true, a, total, bound, stream);
        } else {
            a.work = reinterpret_cast<unsigned long long *>(ctx->counter_slot());
            k_zero_counter<<<1, 64, 0, stream>>>(reinterpret_cast<unsigned int *>(a.work));
            const size_t lds = stack_lds_bytes(c.lds_stack, c.block);
            void *k = pick_kernel(layout, c.lds_stack, refine ? 4 : 2, any, false, ends_with_teams(ctx, total));
            const uint32_t grid = (uint32_t)std::min<uint64_t>(persistent_grid(ctx, k, c.block, lds),
                                                               (total + c.block - 1) / c.block);
            void *args[] = {&a};
            RT_HIP(hipLaunchKernel(k, dim3(grid), dim3(c.block), args, lds, stream));
            if (layout == kQ4 && !any) launch_marked(ctx, a, refine, stream);
        }
        RT_HIP(hipGetLastError());
        ctx->tables.commit(slot, stream);
    }
}

void launch_trace_batch(rt_context *ctx, const rt_batch_item *items, uint32_t nitems, uint32_t flags,
                        const LaunchCfg &c, hipStream_t stream) {
    if (nitems == 0) return;
    RT_REQUIRE(items, "items is NULL");
    std::vector<TraceItem> v(nitems);
    for (uint32_t i = 0; i < nitems; ++i)
        v[i] = TraceItem{&ctx->scene(items[i].scene_id), items[i].rays, items[i].hits, items[i].nrays};
    launch_trace_items(ctx, v, flags, c, stream);
}

}  // namespace rtgpu
