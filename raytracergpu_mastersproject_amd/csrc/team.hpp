// team.hpp -- one ray traced by a team of T lanes (8, 16, 32 or 64) over the width-4 BVH.
//
// With one lane per ray, a launch of few rays lasts as long as its longest ray's chain of dependent
// node and leaf loads (0.2-0.4 ms on 0.1-4 M triangles), most of it with the device nearly idle.
// Here the lanes that would stay idle shorten that chain: each iteration takes up to T/4 entries
// from the team's stack, one per quad of lanes; a quad's lane c tests child c, and a leaf child is
// tested by the lane that found it, at once.  Node children go back on the stack.
//   Closest hit: the nearest quad's children on top, each quad's nearest first.  More nodes are
//   visited than one after the other would (a hit culls only what has not been started).  The result is
//   that of the ordered traversal, or the team says that it must be traced in that order
//   (traverse.hpp: closest hits out of another order).
//   Any hit: the stack keeps depth-first child order, first entry on top, and lanes follow it.  A
//   hit discards everything later in that order and the search goes on with what is earlier, so the
//   result is the hit that the depth-first traversal finds first.
// Measured, closest hit, us per call, before -> now:
//   64 rays / 1,024 triangles 45 -> 11;  4,096 rays / 120 k 142 -> 17;  65,536 / 1 M 322 -> 75;
//   262,144 / 1 M 396 -> 195.
// Bound now: a launch of up to ~32 k rays by the chain's latency (depth of the tree plus the visits
// that do not fit the quads), a larger one by the extra node visits.
#pragma once

#include "traverse.hpp"

namespace rtgpu {

template <int CTRL> __device__ __forceinline__ uint32_t dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}
constexpr int quad_perm(int a, int b, int c, int d) { return a | (b << 2) | (c << 4) | (d << 6); }
constexpr int kRowMirror = 0x140, kRowHalfMirror = 0x141;

// minimum over the team's lanes, in all of them (every lane of the wave active)
template <int T> __device__ __forceinline__ uint32_t team_min(uint32_t v) {
    v = min(v, dpp<quad_perm(1, 0, 3, 2)>(v));
    v = min(v, dpp<quad_perm(2, 3, 0, 1)>(v));
    if constexpr (T >= 8) v = min(v, dpp<kRowHalfMirror>(v));
    if constexpr (T >= 16) v = min(v, dpp<kRowMirror>(v));
    if constexpr (T >= 32) v = min(v, (uint32_t)__shfl_xor((int)v, 16));
    if constexpr (T >= 64) v = min(v, (uint32_t)__shfl_xor((int)v, 32));
    return v;
}

// Orders the wave's LDS accesses: a lane reads what another lane of its wave wrote.
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr uint32_t team_stack(uint32_t t) { return kTeamStackWave / 64u * t; }

// The stack holds at most 3 entries more per entry taken than before it.  While it holds more than
// `limit` entries a team takes one at a time, which is a depth-first walk and adds at most the tree's
// stack bound.  0: the tree is too deep for a team stack of this size.
inline uint32_t team_limit(uint32_t t, uint32_t stack_bound) {
    const uint32_t q = t / 4u, need = 3u * q + stack_bound;
    return team_stack(t) >= need + q ? team_stack(t) - need : 0u;
}

struct TeamHit {
    float t;        // closest hit: in every lane; any hit: in the owner (a miss: tmax)
    uint32_t slot;  // in every lane; kEmpty: a miss
    float u, v;     // in the owner
    bool owner;     // the lane that found the hit
    bool redo;      // closest hit, in every lane: the ray must be traced in the exact nodes' order (team_ordered)
};

// Every lane of the wave calls it; `live` teams trace, all lanes of a team with the same ray.
template <int T, bool ANY>
__device__ __forceinline__ TeamHit team_trace(bool live, v3 o, v3 d, float tmin, float tmax, const uint32_t *wide,
                                              uint32_t nwide, const LeafRecord *__restrict__ rec, uint2 *stacks,
                                              uint32_t limit, const Reach &reach) {
    constexpr uint32_t Q = T / 4;
    const uint32_t lane = threadIdx.x & 63u, c = lane & 3u;
    const uint32_t quad = (lane % T) >> 2, team0 = lane & ~(uint32_t)(T - 1);
    uint2 *st = stacks + (lane / T) * team_stack(T);
    v3 idir, nlo, nhi;
    slab_axis(d.x, o.x, idir.x, nlo.x, nhi.x);
    slab_axis(d.y, o.y, idir.y, nlo.y, nhi.y);
    slab_axis(d.z, o.z, idir.z, nlo.z, nhi.z);
    const float pad = ANY ? 0.0f : ray_pad(o, reach);
    float bt = tmax, cull = tmax;           // closest hit: the team's best t, and the end of its window (hit_window)
    float lt = tmax, lw = tmax, lu = 0.0f, lv = 0.0f;  // this lane's best (any hit: last) hit
    uint32_t ls = kEmpty;
    bool redo = false;                      // closest hit: this lane saw two hits in one window
    bool owner = false;                     // any hit: this lane holds the team's hit
    // the root (the same from every lane), entered as node_step enters it: a NaN tmin bounds nothing
    uint32_t top = live && nwide > 0 && !has_nan(d) && (ANY || !(tmin > tmax * kRobust)) ? 1u : 0u;
    if (top) st[0] = make_uint2(0u, 0xFF800000u);
    wave_fence();
    while (__ballot(top > 0) != 0ull) {
        const uint32_t take = top > limit ? 1u : min(Q, top);
        bool alive = quad < take;
        uint2 e = make_uint2(0u, 0u);
        if (alive) e = st[top - 1u - quad];
        if constexpr (!ANY) alive = alive && __uint_as_float(e.y) <= cull * kRobust;
        wave_fence();
        bool push = false, found = false;
        float tn = 0.0f;
        uint32_t child = kEmpty;
        if (alive) {
            const uint32_t *p = wide + (size_t)e.x * 32u + c;
            const float lox = __uint_as_float(p[0]), hix = __uint_as_float(p[4]), loy = __uint_as_float(p[8]);
            const float hiy = __uint_as_float(p[12]), loz = __uint_as_float(p[16]), hiz = __uint_as_float(p[20]);
            child = p[24];
            const float x0 = fmaf(lox, idir.x, nlo.x), x1 = fmaf(hix, idir.x, nhi.x);
            const float y0 = fmaf(loy, idir.y, nlo.y), y1 = fmaf(hiy, idir.y, nhi.y);
            const float z0 = fmaf(loz, idir.z, nlo.z), z1 = fmaf(hiz, idir.z, nhi.z);
            const float nx = fminf(x0, x1), ny = fminf(y0, y1), nz = fminf(z0, z1);
            const float fx = fmaxf(x0, x1), fy = fmaxf(y0, y1), fz = fmaxf(z0, z1);
            float tf, entry = 0.0f;
            if constexpr (ANY) {
                tn = fmaxf(fmaxf(nx, ny), fmaxf(nz, tmin));
                tf = fminf(fminf(fx, fy), fminf(fz, bt));
            } else {  // the box larger by the ray's pad
                tn = fmaxf(fmaxf(fmaf(-pad, fabsf(idir.x), nx), fmaf(-pad, fabsf(idir.y), ny)),
                           fmaxf(fmaf(-pad, fabsf(idir.z), nz), tmin));
                tf = fminf(fminf(fmaf(pad, fabsf(idir.x), fx), fmaf(pad, fabsf(idir.y), fy)),
                           fminf(fmaf(pad, fabsf(idir.z), fz), cull));
            }
            const bool hit = child != kEmpty && tn <= tf * kRobust;
            push = hit && !(child & kLeafBit);
            bool leaf = hit && (child & kLeafBit);
            if constexpr (!ANY) {  // leaves by their exact boxes
                entry = fmaxf(fmaxf(nx, ny), fmaxf(nz, tmin));
                leaf = leaf && entry <= fminf(fminf(fx, fy), fz) * kRobust;
            }
            if (leaf) {
                const uint32_t first = leaf_first(child), end = first + leaf_count(child);
                for (uint32_t s = first; s < end; ++s) {
                    const LeafRecord r = rec[s];
                    float th = 0.0f, u = 0.0f, v = 0.0f;
                    bool h;
                    if (is_sphere_record(r)) {
                        h = sphere_test(r, o, d, tmin, cull, th);
                        u = r.r1.y;
                        v = r.r1.z;
                    } else {
                        h = triangle_test(r, o, d, tmin, cull, th, u, v);
                    }
                    if constexpr (!ANY) {
                        const float window = hit_window(th, entry);
                        const bool best = th < lt || (th == lt && s < ls);
                        if (h && (best ? window > th && lt <= window : lw > lt && th <= lw)) redo = true;
                        h = h && best;
                        if (h) lw = window;
                    }
                    if (h && (!ANY || th <= bt)) {
                        lt = th;
                        ls = s;
                        lu = u;
                        lv = v;
                        found = true;
                        if (ANY) break;
                    }
                }
            }
        }
        unsigned long long pushing = (__ballot(push) >> team0) & (~0ull >> (64 - T));
        uint32_t base = top - take;
        if constexpr (ANY) {
            // The entries taken are the first ones in depth-first order and lanes follow that order, so a
            // hit leaves only the pushes of earlier lanes worth visiting.
            const unsigned long long fm = (__ballot(found) >> team0) & (~0ull >> (64 - T));
            if (fm != 0ull) {
                const uint32_t first = (uint32_t)__ffsll(fm) - 1u;
                owner = lane - team0 == first;
                pushing &= (1ull << first) - 1ull;
                push = push && lane - team0 < first;
                base = 0u;
            }
            if (push) st[base + (uint32_t)__popcll((pushing >> (lane - team0)) >> 1)] = make_uint2(child, 0u);
        } else {
            if (__ballot(found) != 0ull) {
                cull = bt = ord_dec(team_min<T>(ord_key(lt)));
                if (__ballot(lw > lt) != 0ull)  // rare
                    cull = ord_dec(~team_min<T>(~ord_key(lt == bt ? fmaxf(lw, bt) : bt)));
            }
            const uint32_t k = push ? ((__float_as_uint(tn) & ~3u) | c) : 0u;
            const uint32_t farther = (dpp<quad_perm(1, 2, 3, 0)>(k) > k ? 1u : 0u) +
                                     (dpp<quad_perm(2, 3, 0, 1)>(k) > k ? 1u : 0u) +
                                     (dpp<quad_perm(3, 0, 1, 2)>(k) > k ? 1u : 0u);
            if (push) st[base + (uint32_t)__popcll((pushing >> (4u * quad)) >> 4) + farther] = make_uint2(child, __float_as_uint(tn));
        }
        top = base + (uint32_t)__popcll(pushing);
        wave_fence();
    }
    if constexpr (ANY) {
        const uint32_t slot = team_min<T>(owner ? ls : kEmpty);
        return TeamHit{owner ? lt : tmax, slot, lu, lv, owner, false};
    }
    // the smallest (t, slot); a slot is tested by one lane only
    const uint32_t slot = team_min<T>(lt == bt ? ls : kEmpty);
    redo = redo || (cull > bt && ls != kEmpty && ls != slot && lt <= cull);  // another lane's hit in the window
    const unsigned long long rm = (__ballot(redo) >> team0) & (~0ull >> (64 - T));
    return TeamHit{bt, slot, lu, lv, slot != kEmpty && ls == slot && lt == bt, rm != 0ull};
}

// The rays of the `on` teams in the exact nodes' order, by their first lanes (rare).  Every lane of the wave calls it; `m` takes
// the team stacks' place.
template <int T, int S, bool ANY, class B>
__device__ __forceinline__ TeamHit team_ordered(bool on, v3 o, v3 d, float tmin, float tmax, const uint32_t *wide, uint32_t nwide,
                                                const LeafRecord *rec, const StackMem &m, const B &boxes) {
    Trav t;
    t.bt = tmax;
    t.bslot = kEmpty;
    t.bu = t.bv = 0.0f;
    const bool first = threadIdx.x % T == 0;
    if (on && first) walk_exact<S, ANY>(t, m, o, d, tmin, tmax, nwide, wide, rec, boxes, 2u);
    wave_fence();
    const int from = (int)(threadIdx.x & 63u & ~(uint32_t)(T - 1));
    return TeamHit{__shfl(t.bt, from), (uint32_t)__shfl((int)t.bslot, from), t.bu, t.bv, first && t.bslot != kEmpty, false};
}

// The closest hit of each live team's ray, in the ordered traversal's terms.
template <int T, int S, class B>
__device__ __forceinline__ TeamHit team_closest(bool live, v3 o, v3 d, float tmin, float tmax, const uint32_t *wide, uint32_t nwide,
                                                const LeafRecord *rec, uint2 *stacks, uint32_t limit, const Reach &reach,
                                                const StackMem &m, const B &boxes) {
    TeamHit h = team_trace<T, false>(live, o, d, tmin, tmax, wide, nwide, rec, stacks, limit, reach);
    if (__ballot(live && h.redo) != 0ull) {
        const TeamHit again = team_ordered<T, S, false>(live && h.redo, o, d, tmin, tmax, wide, nwide, rec, m, boxes);
        if (h.redo) h = again;
    }
    return h;
}

// The end of a launch whose waves trace a ray (path) per lane: once a wave finds no more work and at most kLastRays of its
// lanes are live, each of these rays goes on with a team of kLastTeam lanes.  A lane alone would take as long as
// its ray's chain of loads, while the device empties: 1 M any-hit rays on 1 M triangles
// 432 -> 375 us.  Rays start over; fewer rays (6: 386 us) or more in two rounds (12: 404) are slower.
constexpr uint32_t kLastTeam = 8, kLastRays = 64 / kLastTeam;

// The lane whose ray this lane's team of T takes over; `live`: at most 64 / T lanes, and not none.
template <int T> __device__ __forceinline__ uint32_t last_ray_lane(unsigned long long live) {
    for (uint32_t k = (threadIdx.x & 63u) / T; k > 0u && (live & (live - 1ull)) != 0ull; --k) live &= live - 1ull;
    return (uint32_t)__ffsll(live) - 1u;
}

// team_limit of T lanes, from that of kLastTeam
template <int T> __device__ __forceinline__ uint32_t last_limit(uint32_t limit) {
    return limit + (team_stack(T) - 3u * (T / 4u)) - (team_stack(kLastTeam) - 3u * (kLastTeam / 4u));
}

}  // namespace rtgpu
