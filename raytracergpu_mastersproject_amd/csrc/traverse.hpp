// traverse.hpp -- wide-BVH traversal shared by the ray-query and path-tracing kernels.
//
// One lane owns one ray.  A ray's current entry is either a wide node or a leaf:
//   node_step(): W slab tests; hit children are ordered by (entry distance, entry)
//                -- one 64-bit key each, sorted by a network -- the nearest becomes
//                the current entry and the rest are pushed far-to-near;
//   leaf_step(): the leaf's primitives are tested (triangleHit / sphereHit).
// Each ray's sequence of visited entries depends only on the ray and the tree, so
// its counts of AABB and primitive tests are reproducible.  The kernels choose, per
// wave and per iteration, whether lanes sitting on nodes or lanes sitting on leaves
// advance (a ballot); lanes of the other kind simply wait, which changes when a ray
// advances but never the order of its own steps.  This keeps the ~80-instruction
// triangle test from being executed by the whole wave on almost every iteration.
//
// The stack keeps its newest S entries in LDS columns private to the lane and spills
// older ones to a private array, so deep trees never fault.  A slot is 6 bytes: the
// 32-bit entry and the upper half of its distance's order key (see push()).
//
// Closest-hit semantics are those of hitBVH (raytraceBVH.comp:195-265) for any
// traversal order: the smallest t wins and, among equal t, the smallest leaf slot
// wins -- exactly the primitive the reference's right-first traversal tests last,
// because it accepts equal t (`t > tMax` rejects, :130).
#pragma once

#include "rt_device.hpp"

namespace rtgpu {

constexpr uint32_t kSpillCap = 184;  // private spill entries per lane (beyond the LDS part)
constexpr uint32_t kChunk = 512;     // work items a wave takes from the global counter per atomic

// Which rays a wave takes per atomic.  The counter counts chunks, not rays: the first rays go in
// chunks of `chunk`, the last 10 per resident lane in chunks of 128 and then 64.  When the
// counter runs out, a wave is then left with at most one or two rays per lane instead of a
// whole chunk (8 rays per lane at 512), and the launch drains sooner; the few thousand extra
// atomics cost less than that drain.
// T is the ray-index type: uint32_t for one batch of rays, uint64_t for the fused many-scene
// launch.
template <typename T> struct ChunkSchedule {
    T n, nA, nB, KA, KB;
    uint32_t chunk;

    // Fewer rays per chunk when there are too few for every wave to take two chunks
    // (a small launch then ends with its longest ray, not with a wave's run of rays)
    __device__ __forceinline__ ChunkSchedule(T n_, uint32_t waves) {
        n = n_;
        chunk = (uint32_t)max((T)64u, min((T)kChunk, (T)(n / (2u * waves)) & ~(T)63u));
        const T lanes = (T)waves * 64u;
        const T nC = chunk > 64u ? min(n, (T)(2u * lanes)) : (T)0u;
        nB = chunk > 128u ? min((T)(n - nC), (T)(8u * lanes)) : (T)0u;
        nA = n - nB - nC;
        KA = (nA + chunk - 1u) / chunk;
        KB = (nB + 127u) / 128u;
    }
    // rays [lo, hi) of chunk c; false when c is past the end
    __device__ __forceinline__ bool range(T c, uint64_t &lo, uint64_t &hi) const {
        if (c < KA) {
            lo = (uint64_t)c * chunk;
            hi = min(lo + chunk, (uint64_t)nA);
        } else if (c - KA < KB) {
            lo = (uint64_t)nA + (uint64_t)(c - KA) * 128u;
            hi = min(lo + 128u, (uint64_t)nA + nB);
        } else {
            lo = (uint64_t)nA + nB + (uint64_t)(c - KA - KB) * 64u;
            hi = min(lo + 64u, (uint64_t)n);
        }
        return lo < (uint64_t)n;
    }
};

// A wave's place among a launch's work counters.  Wave w of `waves` takes from counter w % lines; value v of counter k
// stands for item v * lines + k, so the items are taken nearly in order.  When its counter has run out, a wave
// helps one other before it stops.  A counter per 32 waves or more: a few waves share one.
struct WorkLines {
    uint32_t lines, home;
    bool helping;
    __device__ __forceinline__ WorkLines(uint32_t wave, uint32_t waves, uint32_t max_lines = kCounterLines) {
        lines = 1u;
        while (lines < max_lines && lines * 64u <= waves) lines *= 2u;
        home = wave & (lines - 1u);
        helping = lines == 1u;
    }
    template <typename T> __device__ __forceinline__ T *counter(T *work) const {
        return work + home * (kCounterStride * 4u / (uint32_t)sizeof(T));
    }
    __device__ __forceinline__ uint64_t item(uint64_t value) const { return value * lines + home; }
    // the counter has run out: false when there is no other to try
    __device__ __forceinline__ bool next() {
        if (helping) return false;
        helping = true;
        home ^= lines / 2u;
        return true;
    }
};

template <int W> struct WideNode {
    float lo[3][W], hi[3][W];
    uint32_t child[W];
};

template <int W> __device__ __forceinline__ void load_node(const uint32_t *wide, uint32_t idx, WideNode<W> &nd);

template <> __device__ __forceinline__ void load_node<2>(const uint32_t *wide, uint32_t idx, WideNode<2> &nd) {
    const float4 *p = reinterpret_cast<const float4 *>(wide) + (size_t)idx * 4u;
    float4 x = p[0], y = p[1], z = p[2];
    uint4 c = reinterpret_cast<const uint4 *>(p)[3];
    nd.lo[0][0] = x.x; nd.lo[0][1] = x.y; nd.hi[0][0] = x.z; nd.hi[0][1] = x.w;
    nd.lo[1][0] = y.x; nd.lo[1][1] = y.y; nd.hi[1][0] = y.z; nd.hi[1][1] = y.w;
    nd.lo[2][0] = z.x; nd.lo[2][1] = z.y; nd.hi[2][0] = z.z; nd.hi[2][1] = z.w;
    nd.child[0] = c.x; nd.child[1] = c.y;
}

__device__ __forceinline__ void unpack4(float4 v, float *o) { o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w; }

template <> __device__ __forceinline__ void load_node<4>(const uint32_t *wide, uint32_t idx, WideNode<4> &nd) {
    const float4 *p = reinterpret_cast<const float4 *>(wide) + (size_t)idx * 8u;
    unpack4(p[0], nd.lo[0]); unpack4(p[1], nd.hi[0]);
    unpack4(p[2], nd.lo[1]); unpack4(p[3], nd.hi[1]);
    unpack4(p[4], nd.lo[2]); unpack4(p[5], nd.hi[2]);
    uint4 c = reinterpret_cast<const uint4 *>(p)[6];
    nd.child[0] = c.x; nd.child[1] = c.y; nd.child[2] = c.z; nd.child[3] = c.w;
}

template <> __device__ __forceinline__ void load_node<8>(const uint32_t *wide, uint32_t idx, WideNode<8> &nd) {
    const float4 *p = reinterpret_cast<const float4 *>(wide) + (size_t)idx * 16u;
    unpack4(p[0], nd.lo[0]); unpack4(p[1], nd.lo[0] + 4);
    unpack4(p[2], nd.hi[0]); unpack4(p[3], nd.hi[0] + 4);
    unpack4(p[4], nd.lo[1]); unpack4(p[5], nd.lo[1] + 4);
    unpack4(p[6], nd.hi[1]); unpack4(p[7], nd.hi[1] + 4);
    unpack4(p[8], nd.lo[2]); unpack4(p[9], nd.lo[2] + 4);
    unpack4(p[10], nd.hi[2]); unpack4(p[11], nd.hi[2] + 4);
    uint4 c0 = reinterpret_cast<const uint4 *>(p)[12], c1 = reinterpret_cast<const uint4 *>(p)[13];
    nd.child[0] = c0.x; nd.child[1] = c0.y; nd.child[2] = c0.z; nd.child[3] = c0.w;
    nd.child[4] = c1.x; nd.child[5] = c1.y; nd.child[6] = c1.z; nd.child[7] = c1.w;
}

// order-preserving map float -> uint32 (total order, -0 < +0) and back
__device__ __forceinline__ uint32_t ord_key(float f) {
    const uint32_t b = __float_as_uint(f);
    return b ^ ((uint32_t)((int32_t)b >> 31) | 0x80000000u);  // negative: ~b; otherwise b | sign bit
}
__device__ __forceinline__ float ord_dec(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

constexpr uint32_t kOrdLowest = 0x00800000u;  // ord_key(-FLT_MAX): never culled, and exact in 16 bits

// per-lane traversal state
struct Trav {
    v3 o, d, idir;
    v3 nlo, nhi;        // per-axis slab offsets of the low and high planes (see slab_axis); of the planes a
                        // ray enters and leaves through on compressed nodes
    float tmin, bt;     // ray start; best t so far (initially tmax)
    float cull;         // compressed nodes, closest hit: what lies beyond is skipped; bt, or more (test_leaf)
    uint32_t bslot;     // leaf slot of the best hit (kEmpty = none, kRedo = the ray must be traced in the exact nodes' order)
    float bu, bv;       // barycentrics of the best hit
    uint32_t cur;       // current entry (node index or leaf entry)
    bool have;          // cur is valid
    float cur_tn;       // its entry distance (not beside cur: a compressed node step stores both from one
                        // 64-bit key, which the compiler would then do through scratch memory)
    uint32_t top, nspill;
    uint32_t nbox, ntri;
};

// A stack slot holds an entry and the upper 16 bits of ord_key(entry distance).  The
// truncated key decodes to a distance no larger than the true one, so culling a popped
// entry against the best hit stays conservative; it may only keep an entry that the full
// key would have culled.  Six bytes per slot instead of eight let more waves share a
// CU's LDS.
constexpr uint32_t kStackSlotBytes = 6;

struct StackMem {
    uint32_t *ent;    // this lane's LDS entry column: slot k at ent[k * 64]
    uint16_t *key;    // this lane's LDS key column, same indexing
    uint2 *spill;     // private spill array (kSpillCap entries of (entry, key << 16))
};

// A wave's LDS: S x 64 entries, then S x 64 keys; at least what the team stacks of its last rays need, which take
// the same place (team.hpp).  6 KB a wave: 26 waves fit a CU, more than the registers let in.
constexpr uint32_t kTeamStackWave = 768;  // team stack entries of 8 bytes per wave
__host__ __device__ constexpr uint32_t wave_lds_bytes(uint32_t lds_stack) {
    return lds_stack * 64u * kStackSlotBytes > kTeamStackWave * 8u ? lds_stack * 64u * kStackSlotBytes : kTeamStackWave * 8u;
}
template <int S> __device__ __forceinline__ uint32_t *wave_lds(void *lds) {
    return static_cast<uint32_t *>(lds) + (threadIdx.x / 64u) * (wave_lds_bytes(S) / 4u);
}
template <int S> __device__ __forceinline__ StackMem stack_mem(void *lds, uint2 *spill) {
    uint32_t *ent = wave_lds<S>(lds);
    uint16_t *key = reinterpret_cast<uint16_t *>(ent + (size_t)S * 64u);
    return StackMem{ent + threadIdx.x % 64u, key + threadIdx.x % 64u, spill};
}

inline size_t stack_lds_bytes(uint32_t lds_stack, uint32_t block) {
    return (size_t)wave_lds_bytes(lds_stack) * (block / 64u);
}

template <int S> __device__ __forceinline__ void push(Trav &t, const StackMem &m, uint32_t e, uint32_t tnkey) {
    if (t.top - t.nspill == (uint32_t)S) {  // LDS part full: move its oldest entry out
        const uint32_t o = (t.nspill & (S - 1)) * 64u;
        if (t.nspill < kSpillCap) m.spill[t.nspill] = make_uint2(m.ent[o], (uint32_t)m.key[o] << 16);
        t.nspill++;
    }
    const uint32_t o = (t.top & (S - 1)) * 64u;
    m.ent[o] = e;
    m.key[o] = (uint16_t)(tnkey >> 16);
    t.top++;
}

template <int S> __device__ __forceinline__ void pop(Trav &t, const StackMem &m) {
    uint2 v;
    if (t.top > t.nspill) {
        t.top--;
        const uint32_t o = (t.top & (S - 1)) * 64u;
        v = make_uint2(m.ent[o], (uint32_t)m.key[o] << 16);
    } else {
        t.nspill--;
        t.top--;
        v = (t.nspill < kSpillCap) ? m.spill[t.nspill] : make_uint2(kEmpty, 0u);
    }
    t.cur = v.x;
    t.cur_tn = ord_dec(v.y);
    t.have = v.x != kEmpty;
}

// Slab distances take one FMA per plane: fma(plane, idir, n) with n = -(o * idir) rounded once
// per ray.  That rounding is an absolute error of up to u|n| (u = 2^-24) in every distance of the
// axis, which the relative widening kRobust does not cover, so each axis carries two offsets:
// nlo for the planes it enters through and nhi for those it leaves through, n lowered and raised
// by e = 4u|n| (which also covers the rounding of n -+ e).  Near distances come out no larger and
// far distances no smaller than with the exact offset, and a box the exact test enters is never
// culled.  The bound widens an axis only where that axis decides the entry or exit distance: a
// per-ray widening by max e over the axes would be huge for a ray almost parallel to an axis
// plane (|d_i| of 1e-7 gives |n| of 1e7) and would send it through most of the tree.
// A zero direction component gets idir = +-2^100 instead of infinity, with e = 0: the products
// with a power of two are exact, so that axis's distances are (plane - o) * 2^100 rounded once
// (coordinates below 2^27 in magnitude), the slab of a direction component of 2^-100 with the
// zero's sign.  A ray lying exactly in the plane of a box face on such an axis enters the box where
// that nudged ray moves into it (low face with +0, high face with -0) and is culled on the other
// face; the reference's AABBhitCheck (raytraceBVH.comp:184-193) culls it on both through 0 * inf =
// NaN, and brute force finds what a cull misses.
__device__ __forceinline__ void slab_axis(float d, float o, float &idir, float &nlo, float &nhi) {
    idir = d != 0.0f ? 1.0f / d : copysignf(0x1p100f, d);
    const float n = -(o * idir);
    const float e = d != 0.0f ? copysignf(0x1p-22f * fabsf(n), idir) : 0.0f;
    nlo = n - e;
    nhi = n + e;
}

constexpr int kQ4 = 44;  // layout code of width 4 with compressed nodes (see node_step_q); 2, 4, 8: exact nodes

// ---------------------------------------------------------------------------
// Closest hits out of another order than the exact nodes'.
//
// A hit's t is rounded, so it can lie a little before the box of its own leaf.  The ordered traversal of the exact nodes
// (node_step<4>) then finds it or not, depending on what it has found before: it skips boxes behind the best hit.  Traversals in
// other orders (compressed nodes, teams of lanes) give the same result all the same:
//   - Let H be the hits whose leaf's exact box the ray enters, M the smallest (t, slot) of them, and E the
//     distance at which the ray enters M's leaf.  The ordered traversal finds M unless another hit's t lies before
//     E: every box around M is entered no later than E, and nothing but such a hit skips it.
//   - These traversals see every hit of H up to their best one's E: they skip what lies beyond it, and their boxes are larger by
//     the most that rounding takes a hit out of its box (ray_pad).  Hits outside H are dropped (leaf_span).
//   - When there is no other hit before E, their result is M.  When there is, the ray is traced
//     again over the exact nodes in their order (kRedo).  That takes two hits a few roundings apart, at a corner
//     that both triangles share: about one ray in 10^7 into a mesh, one in 10^6 aimed at its vertices.
// It costs closest hits 4 to 10 % (4,096 rays / 120 k triangles 17.7 -> 19.2 us, 65,537 / 20 k 47 -> 53, 16.8 M / 4.2 M 3,505 -> 3,635;
// 1080p x 16 frame 5,294 -> 5,558, 501x333x12 817 -> 892), as much on either side of the lines between routes: times given beside those
// lines that were taken before are lower by as much.
// ---------------------------------------------------------------------------
constexpr uint32_t kRedo = 0xFFFFFFFEu;  // Trav::bslot

// How far outside its box a hit of this ray can lie, by the roundings of triangle_test and sphere_test.  u = 2^-24, S the sum of
// the scene's and the origin's largest coordinates.  Triangle: 14 u S off its plane (the numerator's two products
// 7, the denominator's 5, the division 2), 2 u S in the point, and 25 u L^3 / |e1 x e2| in the
// plane (L its longest side): in all below 32 u S, but for needles with L^3 / |e1 x e2| > S / 2.  Sphere of radius r: the discriminant is off by
// 21 u times the squared distance to its centre (at most 3 S^2), so the point by at most 32 u S^2 / r, and
// along the ray by 14 u S.
__device__ __forceinline__ float ray_pad(v3 o, const Reach &reach) {
    const float s = reach.coord + fmaxf(fmaxf(fabsf(o.x), fabsf(o.y)), fabsf(o.z));
    return 0x1p-19f * s * (1.0f + s * reach.inv_radius);
}

// The end of the window before the leaf of a hit at `t`, entered at `entry`: another hit there makes the result
// depend on the order.  None (t itself) when the box is entered before the hit.
__device__ __forceinline__ float hit_window(float t, float entry) {
    return entry <= t * kRobust ? t : fmaxf(t, fmaf(fabsf(entry), 0x1p-21f, entry));
}

// slab_axis for compressed nodes: offsets of the planes the ray enters and leaves through, boxes larger by `pad`
__device__ __forceinline__ void slab_axis_q(float d, float o, float pad, float &idir, float &near, float &far) {
    float lo, hi;
    slab_axis(d, o, idir, lo, hi);
    const float g = pad * fabsf(idir);
    near = (idir < 0.0f ? hi : lo) - g;
    far = (idir < 0.0f ? lo : hi) + g;
}

// A ray that compressed nodes are not made for: a direction component so small, and not zero, that plane
// distances overflow; and for a closest hit an origin beyond the scene's limit (Scene::reach).
template <bool ANY> __device__ __forceinline__ bool needs_exact_nodes(v3 o, v3 d, float far_limit) {
    return (!ANY && fmaxf(fmaxf(fabsf(o.x), fabsf(o.y)), fabsf(o.z)) > far_limit) || (d.x != 0.0f && fabsf(d.x) < 0x1p-90f) ||
           (d.y != 0.0f && fabsf(d.y) < 0x1p-90f) || (d.z != 0.0f && fabsf(d.z) < 0x1p-90f);
}

template <int W, bool ANY>
__device__ __forceinline__ void trav_init(Trav &t, v3 o, v3 d, float tmin, float tmax, uint32_t nwide, const Reach &reach) {
    t.o = o;
    t.d = d;
    if constexpr (W == kQ4) {  // any hit: the first one in the order of the children, whatever boxes were entered before
        const float pad = ANY ? 0.0f : ray_pad(o, reach);
        slab_axis_q(d.x, o.x, pad, t.idir.x, t.nlo.x, t.nhi.x);
        slab_axis_q(d.y, o.y, pad, t.idir.y, t.nlo.y, t.nhi.y);
        slab_axis_q(d.z, o.z, pad, t.idir.z, t.nlo.z, t.nhi.z);
    } else {
        slab_axis(d.x, o.x, t.idir.x, t.nlo.x, t.nhi.x);
        slab_axis(d.y, o.y, t.idir.y, t.nlo.y, t.nhi.y);
        slab_axis(d.z, o.z, t.idir.z, t.nlo.z, t.nhi.z);
    }
    t.tmin = tmin;
    t.bt = t.cull = tmax;
    t.bslot = kEmpty;
    t.bu = 0.0f;
    t.bv = 0.0f;
    t.cur = 0u;  // root
    t.cur_tn = tmin;
    t.have = nwide > 0 && !has_nan(d);  // a NaN direction misses (the reference's root slab test fails)
    t.top = 0;
    t.nspill = 0;
    t.nbox = 0;
    t.ntri = 0;
}

__device__ __forceinline__ bool trav_done(const Trav &t) { return !t.have && t.top == 0; }
__device__ __forceinline__ bool at_leaf(const Trav &t) { return t.have && (t.cur & kLeafBit); }
__device__ __forceinline__ bool at_node(const Trav &t) { return t.have && !(t.cur & kLeafBit); }

__device__ __forceinline__ void cswap64(uint64_t *k, int i, int j) {
    const uint64_t a = k[i], b = k[j];
    const bool sw = a > b;
    k[i] = sw ? b : a;
    k[j] = sw ? a : b;
}

template <int W> __device__ __forceinline__ void sort_keys(uint64_t *k) {
    if constexpr (W == 2) {
        cswap64(k, 0, 1);
    } else if constexpr (W == 4) {
        cswap64(k, 0, 1); cswap64(k, 2, 3);
        cswap64(k, 0, 2); cswap64(k, 1, 3);
        cswap64(k, 1, 2);
    } else {  // Batcher odd-even merge sort, 19 comparators
        cswap64(k, 0, 1); cswap64(k, 2, 3); cswap64(k, 4, 5); cswap64(k, 6, 7);
        cswap64(k, 0, 2); cswap64(k, 1, 3); cswap64(k, 4, 6); cswap64(k, 5, 7);
        cswap64(k, 1, 2); cswap64(k, 5, 6);
        cswap64(k, 0, 4); cswap64(k, 1, 5); cswap64(k, 2, 6); cswap64(k, 3, 7);
        cswap64(k, 2, 4); cswap64(k, 3, 5);
        cswap64(k, 1, 2); cswap64(k, 3, 4); cswap64(k, 5, 6);
    }
}

// Process the current wide node.  Precondition: at_node(t).
//   closest: hit children in increasing (ord_key(tn), entry); ANY: in child order.
//   COUNT: keep t.nbox / t.ntri (only launches that report per-ray counts need them).
template <int W, int S, bool ANY, bool COUNT = true>
__device__ __forceinline__ void node_step(Trav &t, const StackMem &m, const uint32_t *__restrict__ wide) {
    if (t.cur_tn > t.bt * kRobust) {
        t.have = false;  // culled by a closer hit found since it was pushed
    } else {
        WideNode<W> nd;
        load_node<W>(wide, t.cur, nd);
        uint64_t key[W];
        int nh = 0;
#pragma unroll
        for (int c = 0; c < W; ++c) {
            const bool valid = nd.child[c] != kEmpty;
            if constexpr (COUNT) t.nbox += valid ? 1u : 0u;
            float x0 = fmaf(nd.lo[0][c], t.idir.x, t.nlo.x), x1 = fmaf(nd.hi[0][c], t.idir.x, t.nhi.x);
            float y0 = fmaf(nd.lo[1][c], t.idir.y, t.nlo.y), y1 = fmaf(nd.hi[1][c], t.idir.y, t.nhi.y);
            float z0 = fmaf(nd.lo[2][c], t.idir.z, t.nlo.z), z1 = fmaf(nd.hi[2][c], t.idir.z, t.nhi.z);
            float tn = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), t.tmin));
            float tf = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fminf(fmaxf(z0, z1), t.bt));
            const bool hit = valid && tn <= tf * kRobust;
            nh += hit ? 1 : 0;
            const uint32_t hi = ANY ? (uint32_t)c : ord_key(tn);
            // a missed child's key sorts after every hit child's (ord_key of a distance is below ~0u)
            key[c] = ((uint64_t)(hit ? hi : ~0u) << 32) | nd.child[c];
        }
        sort_keys<W>(key);
        if (nh == 0) {
            t.have = false;
        } else {
#pragma unroll
            for (int k = W - 1; k >= 1; --k)
                if (k < nh) push<S>(t, m, (uint32_t)key[k], ANY ? kOrdLowest : (uint32_t)(key[k] >> 32));
            t.cur = (uint32_t)key[0];
            t.cur_tn = ANY ? -__uint_as_float(0x7F800000u) : ord_dec((uint32_t)(key[0] >> 32));
        }
    }
    if (!t.have && t.top > 0) pop<S>(t, m);
}

// ---------------------------------------------------------------------------
// Compressed width-4 nodes (layout code kQ4; rt_device.hpp describes them).
//
// On exact nodes the L1's address pipe is the busiest unit of the per-lane traversal: a 16-byte load takes one
// tag lookup per lane, and a 128-byte node takes seven of them (measured on the 16.8 M-ray / 4.2 M-triangle
// query: 2.58e9 lookups, address unit busy 84 % of the launch, VALU issue 66 %).  A 64-byte node takes four,
// and moves half the bytes.
// Decoding costs less than it seems: the planes of four children lie in one word, so the near and far
// planes of a ray are chosen per axis and not per child; a pair of children's planes becomes two half
// floats with one byte permute, which a mixed-precision FMA reads directly.  Children are sorted as
// doubles {distance, child} by v_min_f64 / v_max_f64, two instructions per comparator.
//
// The boxes are only ever larger than the exact ones, so every box that the exact test enters is
// entered: with N the ray's plane offset and A = 1/d, the exact distance is fl(P*A + N) and this one
// fl((1024+q)*fl(scale*A) + fl(origin*A + N)); the plane lies kPlaneMargin steps outside and the
// roundings are below 4e-4 steps plus 1u of the distance, for which kSlackQ leaves room (4u more than
// kRobust; applied to |tf|, so that it widens negative distances too).  A hit in a leaf that only the larger
// boxes reach must not count, or results would depend on the node format: a hit is taken only if the ray enters
// the leaf's exact box (leaf_entered, evaluated once per hit).
//
// Measured, exact -> compressed: 16.8 M rays / 4.2 M triangles 5.65 -> 3.68 ms (lookups 1.56e9, address unit
// busy 62 %, VALU issue 95 % with 32 of 64 lanes active; 19.4 GB beyond L2 where exact nodes read 23.1, of which
// the memory-side cache, which holds all 127 MB of nodes, serves an unknown part); 1080p x 16 spp frame 6.12 ->
// 5.31 ms; 1.0 M any-hit rays / 1 M triangles 612 -> 556 us.
// ---------------------------------------------------------------------------
constexpr float kSlackQ = 0x1.4p-21f;  // 10 * 2^-24

// where a leaf's exact box is found
struct LeafBoxes {
    const uint32_t *wide;      // the exact width-4 nodes
    const uint32_t *slot_ref;  // leaf slot -> 4 * node + child
};

// Entry and exit distances of one axis of a box lo <= hi, as slab_axis and node_step compute them.
__device__ __forceinline__ void axis_span(float lo, float hi, float d, float o, float idir, float &tn, float &tf) {
    const float n = -(o * idir), e = d != 0.0f ? 0x1p-22f * fabsf(n) : 0.0f;
    tn = fmaf(idir < 0.0f ? hi : lo, idir, n - e);
    tf = fmaf(idir < 0.0f ? lo : hi, idir, n + e);
}

// the entry and exit distances of child box `p` of an exact width-4 node, as node_step has them without a best hit
__device__ __forceinline__ void box_span(const float *p, v3 o, v3 d, v3 idir, float tmin, float &entry, float &exit) {
    float nx, fx, ny, fy, nz, fz;
    axis_span(p[0], p[4], d.x, o.x, idir.x, nx, fx);
    axis_span(p[8], p[12], d.y, o.y, idir.y, ny, fy);
    axis_span(p[16], p[20], d.z, o.z, idir.z, nz, fz);
    entry = fmaxf(fmaxf(nx, ny), fmaxf(nz, tmin));
    exit = fminf(fminf(fx, fy), fz);
}

// those of the leaf that holds `slot`
__device__ __forceinline__ void leaf_span(const LeafBoxes &b, const Trav &t, uint32_t slot, float &entry, float &exit) {
    const uint32_t ref = b.slot_ref[slot];
    box_span(reinterpret_cast<const float *>(b.wide) + (size_t)(ref >> 2) * 32u + (ref & 3u), t.o, t.d, t.idir, t.tmin, entry, exit);
}

// True when the ray enters the primitive's own box, from its record and drawn in by the record's
// rounding, so that it lies inside the leaf's box, and does so by `bound`: then the leaf is entered by then too.  Nearly every hit
// passes; the others (a hit near the box's corner, a triangle in an axis plane) look the leaf's box up.
__device__ __forceinline__ bool primitive_entered(const LeafRecord &r, const Trav &t, float bound) {
    const bool sphere = is_sphere_record(r);
    const auto axis = [&](float v0, float a, float b, float d, float o, float idir, float &tn,
                          float &tf) __attribute__((always_inline)) {
        const float v1 = sphere ? v0 - r.r0.w : v0 + a, v2 = sphere ? v0 + r.r0.w : v0 + b;
        const float lo = fminf(fminf(v0, v1), v2), hi = fmaxf(fmaxf(v0, v1), v2);
        const float in = 0x1p-21f * fmaxf(fabsf(lo), fabsf(hi));
        axis_span(lo + in, hi - in, d, o, idir, tn, tf);
    };
    float nx, fx, ny, fy, nz, fz;
    axis(r.r0.x, r.r1.x, r.r2.x, t.d.x, t.o.x, t.idir.x, nx, fx);
    axis(r.r0.y, r.r1.y, r.r2.y, t.d.y, t.o.y, t.idir.y, ny, fy);
    axis(r.r0.z, r.r1.z, r.r2.z, t.d.z, t.o.z, t.idir.z, nz, fz);
    return fmaxf(fmaxf(nx, ny), fmaxf(nz, t.tmin)) <= fminf(fminf(fx, fy), fminf(fz, bound)) * kRobust;
}

__device__ __forceinline__ double sort_min(double a, double b) {  // no canonicalisation: the bits are a key
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double sort_max(double a, double b) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ void cswap(double *k, int i, int j) {
    const double a = k[i], b = k[j];
    k[i] = sort_min(a, b);
    k[j] = sort_max(a, b);
}

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
// the planes 1024 + q of children 0 and 1 (PAIR 0) or 2 and 3 (PAIR 1) of a plane word
template <int PAIR> __device__ __forceinline__ half2_t plane_pair(uint32_t w) {
    return __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, w, PAIR ? 0x07030602u : 0x05010400u));
}

constexpr uint32_t kMissKey = 0x7FE00000u;  // high word of a missed child's key: above every distance, a finite double

template <int S, bool ANY>
__device__ __forceinline__ void node_step_q(Trav &t, const StackMem &m, const uint32_t *__restrict__ nodes) {
    const uint4 *p = reinterpret_cast<const uint4 *>(nodes) + (size_t)t.cur * 4u;
    const uint4 r0 = p[0], r1 = p[1], r2 = p[2], r3 = p[3];
    const v3 org{__uint_as_float(r0.x), __uint_as_float(r0.y), __uint_as_float(r0.z)};
    const float sx = __uint_as_float(r0.w) * t.idir.x, sy = __uint_as_float(r3.z) * t.idir.y,
                sz = __uint_as_float(r3.w) * t.idir.z;
    const float nx = fmaf(org.x, t.idir.x, t.nlo.x), fx = fmaf(org.x, t.idir.x, t.nhi.x);
    const float ny = fmaf(org.y, t.idir.y, t.nlo.y), fy = fmaf(org.y, t.idir.y, t.nhi.y);
    const float nz = fmaf(org.z, t.idir.z, t.nlo.z), fz = fmaf(org.z, t.idir.z, t.nhi.z);
    const bool gx = t.idir.x < 0.0f, gy = t.idir.y < 0.0f, gz = t.idir.z < 0.0f;
    const uint32_t wnx = gx ? r1.w : r1.y, wfx = gx ? r1.y : r1.w;
    const uint32_t wny = gy ? r2.w : r2.y, wfy = gy ? r2.y : r2.w;
    const uint32_t wnz = gz ? r3.y : r3.x, wfz = gz ? r3.x : r3.y;
    double key[4];
    const auto child = [&](int c, uint32_t e, _Float16 hnx, _Float16 hny, _Float16 hnz, _Float16 hfx, _Float16 hfy,
                           _Float16 hfz) __attribute__((always_inline)) {
        const float tn = fmaxf(fmaxf(fmaxf(fmaf((float)hnx, sx, nx), fmaf((float)hny, sy, ny)),
                                     fmaf((float)hnz, sz, nz)), t.tmin);
        const float tf = fminf(fminf(fminf(fmaf((float)hfx, sx, fx), fmaf((float)hfy, sy, fy)),
                                     fmaf((float)hfz, sz, fz)), ANY ? t.bt : t.cull);
        const bool hit = tn <= fmaf(fabsf(tf), kSlackQ, tf);
        key[c] = __hiloint2double((int)(hit ? (ANY ? (uint32_t)c : __float_as_uint(tn)) : kMissKey), (int)e);
    };
    {
        const half2_t a = plane_pair<0>(wnx), b = plane_pair<0>(wny), c = plane_pair<0>(wnz);
        const half2_t d = plane_pair<0>(wfx), e = plane_pair<0>(wfy), f = plane_pair<0>(wfz);
        child(0, r1.x, a.x, b.x, c.x, d.x, e.x, f.x);
        child(1, r1.z, a.y, b.y, c.y, d.y, e.y, f.y);
    }
    {
        const half2_t a = plane_pair<1>(wnx), b = plane_pair<1>(wny), c = plane_pair<1>(wnz);
        const half2_t d = plane_pair<1>(wfx), e = plane_pair<1>(wfy), f = plane_pair<1>(wfz);
        child(2, r2.x, a.x, b.x, c.x, d.x, e.x, f.x);
        child(3, r2.z, a.y, b.y, c.y, d.y, e.y, f.y);
    }
    cswap(key, 0, 1); cswap(key, 2, 3);
    cswap(key, 0, 2); cswap(key, 1, 3);
    cswap(key, 1, 2);
    t.have = __double2hiint(key[0]) < (int)kMissKey;
    if (t.have) {
        while (t.top + 3u - t.nspill > (uint32_t)S) {  // room for three in the LDS part: move its oldest entries out
            const uint32_t o = (t.nspill & (S - 1)) * 64u;
            if (t.nspill < kSpillCap) m.spill[t.nspill] = make_uint2(m.ent[o], (uint32_t)m.key[o] << 16);
            t.nspill++;
        }
#pragma unroll
        for (int k = 3; k >= 1; --k) {
            const uint32_t hi = (uint32_t)__double2hiint(key[k]);
            if ((int)hi < (int)kMissKey) {
                const uint32_t o = (t.top & (S - 1)) * 64u;
                m.ent[o] = (uint32_t)__double2loint(key[k]);
                m.key[o] = (uint16_t)(hi >> 16);
                t.top++;
            }
        }
        t.cur = (uint32_t)__double2loint(key[0]);
    }
}

// Takes the next entry of a lane that has none, unless the best hit culls it: one entry per wave step (a
// loop until an entry holds runs for the whole wave: 3.86 against 3.70 ms for the 16.8 M-ray query).  An
// entry's distance is its upper 16 bits, no larger than the true one if that is positive; one that is not
// positive is never culled.
template <int S, bool ANY> __device__ __forceinline__ void pop_q(Trav &t, const StackMem &m) {
    if (t.have || t.top == 0) return;
    t.top--;
    uint32_t e;
    float tn;
    if (t.top >= t.nspill) {
        const uint32_t o = (t.top & (S - 1)) * 64u;
        e = m.ent[o];
        asm("" : "+v"(e));  // else this load and the other become one through a generic pointer
        tn = __uint_as_float((uint32_t)m.key[o] << 16);
    } else {
        t.nspill--;
        const uint2 v = m.spill[min(t.nspill, kSpillCap - 1u)];
        e = v.x;
        tn = __uint_as_float(v.y);
    }
    t.cur = e;
    t.have = ANY || !(tn > fmaxf(t.cull * kRobust, 0.0f));
}

// Test the primitives of one leaf entry; true when the ray's traversal is over: an any-hit query has its hit, or the closest
// hit depends on the order (kRedo).
// boxes(): the LeafBoxes of compressed layouts (W == kQ4), not called for the others.
template <int W, bool ANY, bool COUNT, class B>
__device__ __forceinline__ bool test_leaf(Trav &t, uint32_t entry, const LeafRecord *__restrict__ rec, const B &boxes) {
    const uint32_t first = leaf_first(entry), cnt = leaf_count(entry);
    constexpr bool WINDOW = W == kQ4 && !ANY;
    for (uint32_t s = first; s < first + cnt; ++s) {
        if constexpr (COUNT) t.ntri++;
        const LeafRecord r = rec[s];
        const float last = WINDOW ? t.cull : t.bt;
        float th = 0.0f, a = 0.0f, b = 0.0f;
        bool hit;
        if (is_sphere_record(r)) {
            hit = sphere_test(r, t.o, t.d, t.tmin, last, th);
            a = r.r1.y;  // the sphere's centre-based u, v
            b = r.r1.z;
        } else {
            hit = triangle_test(r, t.o, t.d, t.tmin, last, th, a, b);
        }
        if constexpr (WINDOW) {
            if (!hit) continue;
            float window = th;
            if (!primitive_entered(r, t, th)) {
                float in, out;
                leaf_span(boxes(), t, s, in, out);
                if (!(in <= out * kRobust)) continue;
                window = hit_window(th, in);
            }
            const bool best = th < t.bt || (th == t.bt && s < t.bslot);
            // another hit (or the ray's end) in the window of the nearer one
            if (best ? window > th && t.bt <= window : t.cull > t.bt && th <= t.cull) {
                t.bslot = kRedo;
                return true;
            }
            if (!best) continue;
            t.bt = th;
            t.cull = window;
            t.bslot = s;
            t.bu = a;
            t.bv = b;
        } else if (hit && (th < t.bt || (th == t.bt && s < t.bslot))) {
            if constexpr (W == kQ4) {
                if (!primitive_entered(r, t, t.bt)) {
                    float in, out;
                    leaf_span(boxes(), t, s, in, out);
                    if (!(in <= fminf(out, t.bt) * kRobust)) continue;
                }
            }
            t.bt = th;
            t.bslot = s;
            t.bu = a;
            t.bv = b;
            if (ANY) return true;
        }
    }
    return false;
}

// Test the primitives of the current leaf, unless a closer hit found since it was pushed culls it.
// Precondition: at_leaf(t).
template <int W, int S, bool ANY, bool COUNT = true, class B>
__device__ __forceinline__ void leaf_step(Trav &t, const StackMem &m, const LeafRecord *__restrict__ rec, const B &boxes) {
    if constexpr (W == kQ4) {  // culled when popped; an empty child's inverted box can be entered from very far away
        if (t.cur != kEmpty && test_leaf<W, ANY, COUNT>(t, t.cur, rec, boxes)) t.top = t.nspill = 0;
        t.have = false;
    } else {
        if (t.cur_tn <= t.bt * kRobust && test_leaf<W, ANY, COUNT>(t, t.cur, rec, boxes)) {
            t.top = 0;  // any hit: done
            t.nspill = 0;
        }
        t.have = false;
        if (t.top > 0) pop<S>(t, m);
    }
}

// Wave-level choice of which lanes advance this iteration: leaves when enough lanes
// wait on a leaf (or no lane is on a node), nodes otherwise.
__device__ __forceinline__ bool choose_leaf_phase(bool on_node, bool on_leaf, uint32_t leaf_weight) {
    const unsigned long long mn = __ballot(on_node), ml = __ballot(on_leaf);
    if (ml == 0ull) return false;
    if (mn == 0ull) return true;
    return (uint32_t)__popcll(ml) * leaf_weight >= (uint32_t)__popcll(mn);
}

// One step of a lane whose ray is on a node.
template <int W, int S, bool ANY, bool COUNT>
__device__ __forceinline__ void walk_node(Trav &t, const StackMem &m, const uint32_t *nodes) {
    if constexpr (W == kQ4) node_step_q<S, ANY>(t, m, nodes);
    else node_step<W, S, ANY, COUNT>(t, m, nodes);
}

// After the wave's step, whatever its phase.
template <int W, int S, bool ANY> __device__ __forceinline__ void walk_pop(Trav &t, const StackMem &m) {
    if constexpr (W == kQ4) pop_q<S, ANY>(t, m);
}

// Run one ray to completion (used where lanes are not refilled).
template <int W, int S, bool ANY, bool COUNT, class B>
__device__ __forceinline__ void trav_run(Trav &t, const StackMem &m, const uint32_t *nodes, const LeafRecord *rec,
                                         const B &boxes, uint32_t leaf_weight) {
    for (;;) {
        const bool on_node = at_node(t), on_leaf = at_leaf(t);
        if (__ballot(!trav_done(t)) == 0ull) break;
        if (choose_leaf_phase(on_node, on_leaf, leaf_weight)) {
            if (on_leaf) leaf_step<W, S, ANY, COUNT>(t, m, rec, boxes);
        } else {
            if (on_node) walk_node<W, S, ANY, COUNT>(t, m, nodes);
        }
        walk_pop<W, S, ANY>(t, m);
    }
}

// A ray over the exact nodes in their own order, to its end.
template <int S, bool ANY, class B>
__device__ __forceinline__ void walk_exact(Trav &t, const StackMem &m, v3 o, v3 d, float tmin, float tmax, uint32_t nwide,
                                           const uint32_t *wide, const LeafRecord *rec, const B &boxes, uint32_t leaf_weight) {
    trav_init<4, ANY>(t, o, d, tmin, tmax, nwide, Reach{});
    trav_run<4, S, ANY, false>(t, m, wide, rec, boxes, leaf_weight);
}

// Starts a ray.  On compressed nodes one that needs the exact ones: for a closest hit false (it is left to the launch over the
// marked rays), an any hit is run to its end here (rare: the other lanes of its wave wait).
template <int W, int S, bool ANY, class B>
__device__ __forceinline__ bool walk_init(Trav &t, const StackMem &m, v3 o, v3 d, float tmin, float tmax,
                                          uint32_t nwide, const Reach &reach, const LeafRecord *rec, const B &boxes,
                                          uint32_t leaf_weight) {
    if (W == kQ4 && needs_exact_nodes<ANY>(o, d, reach.far_limit)) {
        if constexpr (!ANY) return false;
        walk_exact<S, ANY>(t, m, o, d, tmin, tmax, nwide, boxes().wide, rec, boxes, leaf_weight);
    } else {
        trav_init<W, ANY>(t, o, d, tmin, tmax, nwide, reach);
    }
    return true;
}

}  // namespace rtgpu
