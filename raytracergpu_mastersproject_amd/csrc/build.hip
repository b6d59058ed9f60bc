// build.hip -- device BVH construction for a resident scene.
//
// Replaces compute stage S1 of the reference (RaytracerGPU_MastersProject/
// RaytracerBVH.cpp:734-997): model->world transform, centroid bounds, Morton
// codes, a stable radix sort, Karras 2012 topology and a bottom-up refit,
// producing the reference's binary HLBVHNode buffer (the RaytracerBVH builder
// output).  That tree is then collapsed, level by level, into the wide SoA node
// layout the traversal kernels read, with the triangle data re-laid out per
// leaf slot (LeafRecord).  The reference's single-workgroup reduction and sort
// are replaced by device-wide kernels.
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstring>
#include <limits>
#include <vector>

#include "box_levels.hpp"
#include "rt_internal.hpp"

namespace rtgpu {
namespace {

constexpr int kB = 256;  // build kernels' block size

__device__ inline uint32_t fkey(float f) {
    uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ inline float fkey_dec(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

inline uint32_t grid_for(uint64_t n, int block = kB) {
    uint64_t g = (n + block - 1) / block;
    return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(g, 1u << 30));
}

// ModelSpaceToWorldSpace.comp:32-48: v' = M * vec4(v, 1) evaluated left to right
__host__ __device__ inline void mat_vec1(const float *m, float *v) {
    float x = v[0], y = v[1], z = v[2];
    float r[4];
    for (int i = 0; i < 4; ++i) r[i] = m[0 + i] * x + m[4 + i] * y + m[8 + i] * z + m[12 + i] * 1.0f;
    v[0] = r[0]; v[1] = r[1]; v[2] = r[2]; v[3] = r[3];
}
// (a primitive with a model index out of range stays as it is; the build reports it)
__global__ void k_model_to_world(rt_triangle *tris, uint32_t ntri, rt_sphere *sph, uint32_t nsph,
                                 const float *models, uint32_t nmodels) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < ntri) {
        rt_triangle t = tris[i];
        if (t.modelIndex >= nmodels) return;
        const float *m = models + 16u * t.modelIndex;
        mat_vec1(m, t.v0);
        mat_vec1(m, t.v1);
        mat_vec1(m, t.v2);
        tris[i] = t;
    } else if (i < ntri + nsph) {
        rt_sphere s = sph[i - ntri];
        if (s.modelIndex >= nmodels) return;
        float c[4] = {s.center[0], s.center[1], s.center[2], s.center[3]};
        mat_vec1(models + 16u * s.modelIndex, c);  // radius stays unscaled
        s.center[0] = c[0]; s.center[1] = c[1]; s.center[2] = c[2]; s.center[3] = c[3];
        sph[i - ntri] = s;
    }
}

// centroid of primitive i (GetEnclosingAABB.comp:26-28, GenerateMortonCodesOfPrimitives.comp:62-64)
__device__ inline v3 centroid(const rt_triangle *tris, uint32_t ntri, const rt_sphere *sph, uint32_t i) {
    if (i < ntri) {
        const rt_triangle &t = tris[i];
        v3 s = (v3{t.v0[0], t.v0[1], t.v0[2]} + v3{t.v1[0], t.v1[1], t.v1[2]}) + v3{t.v2[0], t.v2[1], t.v2[2]};
        return s / 3.0f;
    }
    const rt_sphere &s = sph[i - ntri];
    return v3{s.center[0], s.center[1], s.center[2]};
}

// Centroid bounds (GetEnclosingAABB.comp): min and max in a total order (-0 < +0), so the result does not depend
// on the order.  One partial result per block; the Morton kernel's blocks reduce the few partials
// themselves.  Atomics on six shared words from every block took 272 us of 1 M triangles' build, this takes 20.
constexpr uint32_t kBoundsBlocks = 256;

__device__ inline void bounds_reduce(uint32_t (&mn)[3], uint32_t (&mx)[3]) {  // block-wide, valid in every thread
    __shared__ uint32_t red[6][kB / 64];
    for (int a = 0; a < 3; ++a) {
        for (int off = 32; off > 0; off >>= 1) {
            mn[a] = min(mn[a], (uint32_t)__shfl_xor((int)mn[a], off));
            mx[a] = max(mx[a], (uint32_t)__shfl_xor((int)mx[a], off));
        }
    }
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    if (lane == 0)
        for (int a = 0; a < 3; ++a) { red[a][wave] = mn[a]; red[3 + a][wave] = mx[a]; }
    __syncthreads();
    for (int w = 0; w < kB / 64; ++w)
        for (int a = 0; a < 3; ++a) {
            mn[a] = min(mn[a], red[a][w]);
            mx[a] = max(mx[a], red[3 + a][w]);
        }
}

__global__ __launch_bounds__(kB) void k_centroid_bounds(const rt_triangle *tris, uint32_t ntri, const rt_sphere *sph,
                                                        uint32_t n, uint32_t *partial) {
    uint32_t mn[3], mx[3];
    for (int a = 0; a < 3; ++a) {  // GetEnclosingAABB.comp starts from +-1e9
        mn[a] = fkey(1000000000.0f);
        mx[a] = fkey(-1000000000.0f);
    }
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        v3 c = centroid(tris, ntri, sph, i);
        uint32_t k[3] = {fkey(c.x), fkey(c.y), fkey(c.z)};
        for (int a = 0; a < 3; ++a) {
            mn[a] = min(mn[a], k[a]);
            mx[a] = max(mx[a], k[a]);
        }
    }
    bounds_reduce(mn, mx);
    if (threadIdx.x == 0)
        for (int a = 0; a < 3; ++a) {
            partial[6u * blockIdx.x + a] = mn[a];
            partial[6u * blockIdx.x + 3 + a] = mx[a];
        }
}

__device__ inline uint32_t sep3(uint32_t v) {  // GenerateMortonCodesOfPrimitives.comp:20-28
    if (v == 1024u) v--;
    v = (v | (v << 16)) & 50331903u;
    v = (v | (v << 8)) & 50393103u;
    v = (v | (v << 4)) & 51130563u;
    v = (v | (v << 2)) & 153391689u;
    return v;
}

__global__ __launch_bounds__(kB) void k_morton(const rt_triangle *tris, uint32_t ntri, const rt_sphere *sph, uint32_t n,
                                               const uint32_t *partial, uint32_t nparts, uint32_t ref_morton,
                                               uint32_t *keys, uint32_t *vals) {
    uint32_t mn[3], mx[3];
    for (int a = 0; a < 3; ++a) {  // nparts <= kB
        mn[a] = threadIdx.x < nparts ? partial[6u * threadIdx.x + a] : 0xFFFFFFFFu;
        mx[a] = threadIdx.x < nparts ? partial[6u * threadIdx.x + 3 + a] : 0u;
    }
    bounds_reduce(mn, mx);
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float lo[3], span[3];
    const float delta = 0.001f, pad = 0.001f / 2.0f;
    for (int a = 0; a < 3; ++a) {  // padAABB (GetEnclosingAABB.comp:33-46)
        float l = fkey_dec(mn[a]), h = fkey_dec(mx[a]);
        if (h - l < delta) { l -= pad; h += pad; }
        lo[a] = l;
        span[a] = h - l;
    }
    v3 c = centroid(tris, ntri, sph, i);
    float cc[3] = {c.x, c.y, c.z};
    uint32_t q[3];
    for (int a = 0; a < 3; ++a) {
        float off = ref_morton ? cc[a] / span[a] : (cc[a] - lo[a]) / span[a];
        q[a] = f2u_sat(off * 1024.0f);
    }
    keys[i] = (sep3(q[2]) << 2) | (sep3(q[1]) << 1) | sep3(q[0]);
    vals[i] = i;
}

// exclusive sum of v over the block's threads, and the block's total
template <int THREADS> __device__ inline uint32_t block_exclusive_scan(uint32_t v, uint32_t *total) {
    __shared__ uint32_t wsum[THREADS / 64];
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    uint32_t x = v;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    uint32_t base = 0, all = 0;
    for (int w = 0; w < THREADS / 64; ++w) {
        if (w < wave) base += wsum[w];
        all += wsum[w];
    }
    __syncthreads();
    *total = all;
    return base + x - v;
}

// Temporaries of one build, carved from one block of the context's scratch cache.  Every
// launch of a build is on one stream, so a range can be handed out again as soon as the
// launches using it have been enqueued (mark / release); the block itself returns to the
// cache with an event after the build's last launch.
class Temps {
  public:
    Temps(rt_context *ctx, uint64_t bytes, hipStream_t st) : lease_(ctx->scratch, bytes, st), cap_(bytes) {}
    template <class T> T *take(uint64_t count) {
        const uint64_t b = (sizeof(T) * count + 255u) & ~uint64_t(255);
        RT_REQUIRE(used_ + b <= cap_, "internal: build temporaries exceed their bound");
        T *p = reinterpret_cast<T *>(lease_.ptr() + used_);
        used_ += b;
        return p;
    }
    uint64_t mark() const { return used_; }
    void release(uint64_t m) { used_ = m; }

  private:
    ScratchLease lease_;
    uint64_t cap_, used_ = 0;
};

uint64_t round256(uint64_t b) { return (b + 255u) & ~uint64_t(255); }

// ---------------------------------------------------------------------------
// Stable LSD radix sort, 4 passes x 8 bits (RadixSortSimple.comp's intent, A14):
// per-tile digit histograms -> exclusive scan of each digit's row of tiles -> stable
// scatter in which each round ranks 256 keys with wave ballots (keys keep tile order).
// ---------------------------------------------------------------------------
constexpr int kSortItems = 8;
constexpr int kSortTile = kB * kSortItems;

__global__ void k_radix_hist(const uint32_t *keys, uint32_t n, uint32_t shift, uint32_t *ghist, uint32_t nblocks) {
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    uint64_t base = (uint64_t)blockIdx.x * kSortTile;
    for (int r = 0; r < kSortItems; ++r) {
        uint64_t p = base + (uint64_t)r * kB + threadIdx.x;
        if (p < n) atomicAdd(&h[(keys[p] >> shift) & 255u], 1u);
    }
    __syncthreads();
    ghist[(uint64_t)threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

// One block per digit: its tiles' counts -> the sums of the tiles before, and the digit's total.  The scatter adds
// the smaller digits' totals itself.  A block's row is read in tiles of 2,048, so 1 M keys (489 tiles of keys) take
// 5 us; one block over all 125,000 counts took 117 us, most of a 1 M-key sort.
__global__ __launch_bounds__(kB) void k_radix_scan(const uint32_t *hist, uint32_t nblocks, uint32_t *before, uint32_t *totals) {
    const uint32_t *in = hist + (uint64_t)blockIdx.x * nblocks;
    uint32_t *out = before + (uint64_t)blockIdx.x * nblocks;
    uint32_t run = 0;
    for (uint32_t t0 = 0; t0 < nblocks; t0 += kB * 8u) {
        const uint32_t base = t0 + threadIdx.x * 8u;
        uint32_t v[8], s = 0, total;
        for (int k = 0; k < 8; ++k) {
            v[k] = base + k < nblocks ? in[base + k] : 0u;
            s += v[k];
        }
        uint32_t pre = run + block_exclusive_scan<kB>(s, &total);
        for (int k = 0; k < 8; ++k) {
            if (base + k < nblocks) out[base + k] = pre;
            pre += v[k];
        }
        run += total;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = run;
}

__global__ __launch_bounds__(kB) void k_radix_scatter(const uint32_t *keys_in, const uint32_t *vals_in, uint32_t *keys_out,
                                                      uint32_t *vals_out, uint32_t n, uint32_t shift,
                                                      const uint32_t *before, const uint32_t *totals, uint32_t nblocks) {
    static_assert(kB == 256, "a thread per digit");
    __shared__ uint32_t off[256];
    __shared__ uint32_t cnt[kB / 64][256];
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    uint32_t all;
    off[tid] = block_exclusive_scan<kB>(totals[tid], &all) + before[(uint64_t)tid * nblocks + blockIdx.x];
    const unsigned long long lt = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
    uint64_t base = (uint64_t)blockIdx.x * kSortTile;
    for (int r = 0; r < kSortItems; ++r) {
        for (int w = 0; w < kB / 64; ++w) cnt[w][tid] = 0;
        __syncthreads();
        uint64_t p = base + (uint64_t)r * kB + tid;
        bool valid = p < n;
        uint32_t key = valid ? keys_in[p] : 0u, val = valid ? vals_in[p] : 0u;
        uint32_t digit = (key >> shift) & 255u;
        unsigned long long peers = __ballot(valid);
        for (int b = 0; b < 8; ++b) {
            unsigned long long bb = __ballot((digit >> b) & 1u);
            peers &= ((digit >> b) & 1u) ? bb : ~bb;
        }
        uint32_t rank = (uint32_t)__popcll(peers & lt);
        if (valid && rank == 0) cnt[wave][digit] = (uint32_t)__popcll(peers);
        __syncthreads();
        if (valid) {
            uint32_t before = 0;
            for (int w = 0; w < wave; ++w) before += cnt[w][digit];
            uint32_t dst = off[digit] + before + rank;
            keys_out[dst] = key;
            vals_out[dst] = val;
        }
        __syncthreads();
        uint32_t add = 0;
        for (int w = 0; w < kB / 64; ++w) add += cnt[w][tid];
        off[tid] += add;
        __syncthreads();
    }
}

uint64_t sort_temp_bytes(uint64_t n) {
    const uint64_t nblocks = (n + kSortTile - 1) / kSortTile;
    return 2 * round256(4 * n) + 2 * round256(4 * 256 * nblocks) + round256(4 * 256);
}

// Few keys: each finds its place in the sorted order by counting the keys before it, the smaller ones and
// the equal ones of smaller index.  A block ranks 64 keys, one per lane; each of its 16 waves counts over a sixteenth of
// the keys, which it reads as scalars.  n^2 comparisons at two instructions each, but one launch and no
// dependent passes.  A build of 4,096 triangles takes 90 us with it and 140 with the passes, of 16,384 131 and 164, of
// 32,768 183 and 169: the line lies between.
constexpr uint32_t kRankSort = 16384;

__global__ __launch_bounds__(1024) void k_rank_sort(const uint32_t *__restrict__ keys, const uint32_t *__restrict__ vals,
                                                    uint32_t n, uint32_t *__restrict__ keys_out,
                                                    uint32_t *__restrict__ vals_out) {
    __shared__ uint32_t part[16][64];
    const uint32_t lane = threadIdx.x % 64u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64u);
    const uint32_t first = blockIdx.x * 64u, i = first + lane;
    const uint32_t key = i < n ? keys[i] : 0u;  // Morton codes have 30 bits: key + 1 does not wrap
    const uint32_t chunk = (n + 15u) / 16u, lo = min(wave * chunk, n), hi = min(lo + chunk, n);
    // keys before this block's: also the equal ones are before; keys after it: only the smaller ones
    const uint32_t a = min(max(first, lo), hi), b = min(max(first + 64u, lo), hi);
    uint32_t rank = 0;
#pragma unroll 8
    for (uint32_t j = lo; j < a; ++j) rank += keys[j] <= key ? 1u : 0u;
    for (uint32_t j = a; j < b; ++j) rank += keys[j] < key + (j < i ? 1u : 0u) ? 1u : 0u;
#pragma unroll 8
    for (uint32_t j = b; j < hi; ++j) rank += keys[j] < key ? 1u : 0u;
    part[wave][lane] = rank;
    __syncthreads();
    if (wave == 0u && i < n) {
        for (uint32_t w = 1; w < 16u; ++w) rank += part[w][lane];
        keys_out[rank] = key;
        vals_out[rank] = vals[i];
    }
}

// Sorts keys, and vals with them; the two pointers are then the result's, in the given arrays or in `tmp`.
void sort_pairs(uint32_t *&keys, uint32_t *&vals, uint32_t n, hipStream_t st, Temps &tmp) {
    if (n <= 1) return;
    uint32_t *k2 = tmp.take<uint32_t>(n), *v2 = tmp.take<uint32_t>(n);
    if (n <= kRankSort) {
        k_rank_sort<<<(n + 63u) / 64u, 1024, 0, st>>>(keys, vals, n, k2, v2);
        keys = k2;
        vals = v2;
        return;
    }
    const uint32_t nblocks = (n + kSortTile - 1) / kSortTile;
    uint32_t *hist = tmp.take<uint32_t>(256ull * nblocks), *before = tmp.take<uint32_t>(256ull * nblocks);
    uint32_t *totals = tmp.take<uint32_t>(256);
    for (uint32_t shift = 0; shift < 32u; shift += 8u) {
        k_radix_hist<<<nblocks, kB, 0, st>>>(keys, n, shift, hist, nblocks);
        k_radix_scan<<<256, kB, 0, st>>>(hist, nblocks, before, totals);
        k_radix_scatter<<<nblocks, kB, 0, st>>>(keys, vals, k2, v2, n, shift, before, totals, nblocks);
        std::swap(keys, k2);
        std::swap(vals, v2);
    }
}

// ---------------------------------------------------------------------------
// Karras topology (ConstructHLBVH.comp:58-106, 171-214)
// ---------------------------------------------------------------------------
__device__ inline int kdelta(const uint32_t *codes, int n, int i, int j) {
    if (j < 0 || j > n - 1) return -1;
    uint32_t ci = codes[i], cj = codes[j];
    if (ci == cj) return 32 + __clz((int)((uint32_t)i ^ (uint32_t)j));
    return __clz((int)(ci ^ cj));
}

__global__ void k_karras(const uint32_t *codes, int n, rt_bvh_node *nodes, uint2 *range) {
    int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n - 1) return;
    int dl = kdelta(codes, n, id, id - 1), dr = kdelta(codes, n, id, id + 1);
    int dir = (dr >= dl) ? 1 : -1;
    int dmin = min(dl, dr);
    int lmax = 2;
    while (kdelta(codes, n, id, id + lmax * dir) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t > 0; t >>= 1)
        if (kdelta(codes, n, id, id + (l + t) * dir) > dmin) l += t;
    int e = id + l * dir;
    int first = min(id, e), last = max(id, e);
    int common = kdelta(codes, n, first, last);
    int split = first, stride = last - first;
    do {
        stride = (stride + 1) >> 1;
        int ns = split + stride;
        if (ns < last && kdelta(codes, n, first, ns) > common) split = ns;
    } while (stride > 1);
    const int leaf0 = n - 1;
    int left = (split == first) ? leaf0 + split : split;
    int right = (split + 1 == last) ? leaf0 + split + 1 : split + 1;
    rt_bvh_node nd;
    nd.minX = nd.maxX = nd.minY = nd.maxY = nd.minZ = nd.maxZ = 0.0f;
    nd.left = (uint32_t)left;
    nd.right = (uint32_t)right;
    nd.primitiveIndex = 0;
    nd.primitiveType = 0;
    nodes[id] = nd;
    range[id] = make_uint2((uint32_t)first, (uint32_t)last);
}

__device__ inline bool has_nan3(const rt_bvh_node &b) {
    return has_nan(v3{b.minX, b.minY, b.minZ}) || has_nan(v3{b.maxX, b.maxY, b.maxZ});
}

// leaf boxes (ConstructHLBVH.comp:33-56, 134-169), leaf records and material table
__device__ inline void leaf_body(const rt_triangle *tris, const rt_sphere *sph, const float2 *sph_uv,
                                 const uint32_t *slot_prim, uint32_t i, rt_bvh_node *leaf_nodes, LeafRecord *records,
                                 uint32_t *slot_mat) {
    uint32_t p = slot_prim[i];
    rt_bvh_node nd;
    LeafRecord rec;
    if (p & RT_SPHERE_BIT) {
        const rt_sphere &s = sph[p & ~RT_SPHERE_BIT];
        float l[3], r[3];
        for (int a = 0; a < 3; ++a) { l[a] = s.center[a] - s.radius; r[a] = s.center[a] + s.radius; }
        nd.minX = gmin(l[0], r[0]); nd.maxX = gmax(l[0], r[0]);
        nd.minY = gmin(l[1], r[1]); nd.maxY = gmax(l[1], r[1]);
        nd.minZ = gmin(l[2], r[2]); nd.maxZ = gmax(l[2], r[2]);
        nd.primitiveIndex = p & ~RT_SPHERE_BIT;
        nd.primitiveType = RT_SPHERE_PRIMITIVE;
        rec.r0 = make_float4(s.center[0], s.center[1], s.center[2], s.radius);
        const float2 uv = sph_uv[p & ~RT_SPHERE_BIT];
        rec.r1 = make_float4(__uint_as_float(kSphereTag), uv.x, uv.y, 0.0f);
        rec.r2 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        rec.r3 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        slot_mat[i] = s.materialIndex;
    } else {
        const rt_triangle &t = tris[p];
        nd.minX = gmin(t.v0[0], gmin(t.v1[0], t.v2[0]));
        nd.maxX = gmax(t.v0[0], gmax(t.v1[0], t.v2[0]));
        nd.minY = gmin(t.v0[1], gmin(t.v1[1], t.v2[1]));
        nd.maxY = gmax(t.v0[1], gmax(t.v1[1], t.v2[1]));
        nd.minZ = gmin(t.v0[2], gmin(t.v1[2], t.v2[2]));
        nd.maxZ = gmax(t.v0[2], gmax(t.v1[2], t.v2[2]));
        nd.primitiveIndex = p;
        nd.primitiveType = RT_TRIANGLE_PRIMITIVE;
        rec = make_triangle_record(v3{t.v0[0], t.v0[1], t.v0[2]}, v3{t.v1[0], t.v1[1], t.v1[2]},
                                   v3{t.v2[0], t.v2[1], t.v2[2]});
        slot_mat[i] = t.materialIndex;
    }
    const float delta = 0.001f, pad = 0.001f / 2.0f;
    if (nd.maxX - nd.minX < delta) { nd.minX -= pad; nd.maxX += pad; }
    if (nd.maxY - nd.minY < delta) { nd.minY -= pad; nd.maxY += pad; }
    if (nd.maxZ - nd.minZ < delta) { nd.minZ -= pad; nd.maxZ += pad; }
    nd.left = 0;
    nd.right = 0;
    if (leaf_nodes) leaf_nodes[i] = nd;
    records[i] = rec;
}
// Also the leaf slot -> primitive table (sorted_vals, or the reference's unsorted placement), and *has_nan = 1
// when some box has a NaN plane (one store per wave; box_union needs to know).
__global__ void k_leaves(const rt_triangle *tris, uint32_t ntri, const rt_sphere *sph, const float2 *sph_uv,
                         const uint32_t *sorted_vals, uint32_t ref_leaves, uint32_t n, uint32_t *slot_prim,
                         rt_bvh_node *leaf_nodes, LeafRecord *records, uint32_t *slot_mat, uint32_t *has_nan) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t p = ref_leaves ? i : sorted_vals[i];
    slot_prim[i] = p < ntri ? p : (RT_SPHERE_BIT | (p - ntri));
    leaf_body(tris, sph, sph_uv, slot_prim, i, leaf_nodes, records, slot_mat);
    const rt_bvh_node nd = leaf_nodes[i];
    const bool nan = has_nan3(nd);
    const unsigned long long m = __ballot(nan);
    if (m != 0ull && __lane_id() == (uint32_t)__ffsll((long long)m) - 1u) *has_nan = 1u;
}
// leaf records only (caller-supplied node buffer: boxes come from that buffer)
__global__ void k_records(const rt_triangle *tris, const rt_sphere *sph, const float2 *sph_uv, const uint32_t *slot_prim,
                          uint32_t n, LeafRecord *records, uint32_t *slot_mat) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) leaf_body(tris, sph, sph_uv, slot_prim, i, nullptr, records, slot_mat);
}

// ConstructAABBsOfInternalNodes.comp:27-65 computes each internal box as the union of its children's,
// bottom-up, with an atomic visit counter per node.  On this device the eight XCDs keep separate L2 caches,
// so each of that scheme's release/acquire pairs writes back and invalidates a whole L2; one launch per
// level needs every node's depth first and ~60 launches and 6 host waits in all.  Here no node waits
// for another: an internal node's box is the union of the leaf boxes of its slot range, taken from a
// table of the unions of 2^k aligned slots (k = 1, 2, ...), 8 levels of it per launch, in at most 2 loads per level.
// The reference's min and max keep their left operand on ties and both trees keep the slots' order, so the
// bits are the same, -0 and +0 included.  With a NaN plane they are not associative: see k_refit_pass.
// 1 M triangles: 0.05 ms in 4 launches (before: 0.25 ms of kernels in 39 launches).
struct Box {
    float v[6];  // minX maxX minY maxY minZ maxZ
};
__device__ inline Box box_union(const Box &a, const Box &b) {
    Box r;
    for (int k = 0; k < 6; k += 2) {
        r.v[k] = gmin(a.v[k], b.v[k]);
        r.v[k + 1] = gmax(a.v[k + 1], b.v[k + 1]);
    }
    return r;
}
__device__ inline Box node_box(const rt_bvh_node &n) { return Box{{n.minX, n.maxX, n.minY, n.maxY, n.minZ, n.maxZ}}; }

struct BoxTable {  // its levels: box_levels.hpp
    const rt_bvh_node *leaves;
    Box *boxes;
    uint32_t n;
};

// Levels level+1 .. level+8 from level `level` (0: the leaves).  A block takes 256 of its boxes.
__global__ __launch_bounds__(kB) void k_box_table(BoxTable t, uint32_t level) {
    __shared__ Box sh[kB];
    const uint32_t have = box_count(t.n, level), i = blockIdx.x * kB + threadIdx.x;
    if (i < have) {
        if (level == 0) sh[threadIdx.x] = node_box(t.leaves[i]);
        else sh[threadIdx.x] = t.boxes[boxes_before(t.n, level) + i];
    }
    uint64_t at = boxes_before(t.n, level + 1u);
    for (uint32_t k = 1; k <= 8u; ++k) {
        const uint32_t count = box_count(t.n, level + k), j = blockIdx.x * (kB >> k) + threadIdx.x;
        const bool mine = threadIdx.x < (kB >> k) && j < count;
        Box b;
        __syncthreads();
        if (mine) b = box_union(sh[2u * threadIdx.x], sh[2u * threadIdx.x + 1u]);
        __syncthreads();
        if (mine) {
            sh[threadIdx.x] = b;
            t.boxes[at + j] = b;
        }
        at += count;
    }
}

__global__ void k_refit(rt_bvh_node *nodes, const uint2 *range, BoxTable t) {
    const uint32_t id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id + 1u >= t.n) return;
    uint32_t l = range[id].x, r = range[id].y + 1u, level = 0;
    uint64_t at = 0;  // of level `level` in the table
    Box left, right;
    bool hl = false, hr = false;
    while (l < r) {
        if (l & 1u) {
            const Box b = level ? t.boxes[at + l] : node_box(t.leaves[l]);
            left = hl ? box_union(left, b) : b;
            hl = true;
            ++l;
        }
        if (r & 1u) {
            --r;
            const Box b = level ? t.boxes[at + r] : node_box(t.leaves[r]);
            right = hr ? box_union(b, right) : b;
            hr = true;
        }
        l >>= 1;
        r >>= 1;
        at += level ? box_count(t.n, level) : 0u;
        ++level;
    }
    const Box b = hl && hr ? box_union(left, right) : hl ? left : right;
    rt_bvh_node &nd = nodes[id];
    nd.minX = b.v[0]; nd.maxX = b.v[1]; nd.minY = b.v[2]; nd.maxY = b.v[3]; nd.minZ = b.v[4]; nd.maxZ = b.v[5];
}

// Every node's union of its children's present boxes, from `in` to `out`.  As many passes as the tree is deep make
// every box final whatever the union's rules for NaN; an LBVH is at most 64 deep (each child's range shares a
// strictly longer prefix of the 64-bit (code, index) key than its parent's).  Scenes with NaN vertices only.
__global__ void k_refit_pass(const rt_bvh_node *in, rt_bvh_node *out, uint32_t n) {
    const uint32_t id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= 2u * n - 1u) return;
    rt_bvh_node nd = in[id];
    if (id < n - 1u) {
        const Box b = box_union(node_box(in[nd.left]), node_box(in[nd.right]));
        nd.minX = b.v[0]; nd.maxX = b.v[1]; nd.minY = b.v[2]; nd.maxY = b.v[3]; nd.minZ = b.v[4]; nd.maxZ = b.v[5];
    }
    out[id] = nd;
}

uint64_t refit_temp_bytes(uint64_t n) { return round256(sizeof(Box) * n); }

// Internal boxes of the n-1 internal nodes (leaf boxes are already written).
void refit(rt_bvh_node *nodes, const uint2 *range, uint32_t n, hipStream_t st, Temps &tmp) {
    const uint64_t mk = tmp.mark();
    BoxTable t{nodes + (n - 1), tmp.take<Box>(n), n};
    for (uint32_t level = 0; box_count(n, level) > 1u; level += 8) k_box_table<<<grid_for(box_count(n, level)), kB, 0, st>>>(t, level);
    k_refit<<<grid_for(n - 1), kB, 0, st>>>(nodes, range, t);
    tmp.release(mk);
}

// ---------------------------------------------------------------------------
// Collapse binary -> wide, breadth first.  A wide node made
// from binary node b takes b's children and repeatedly opens the child with the
// largest surface area until W children exist; a child whose subtree holds at
// most leaf_size primitives becomes a leaf over its contiguous slot range.
//
// Three steps: every binary node's choice of children (k_collapse_choose, all at once), the numbering of the wide
// nodes level by level (k_collapse_levels), which then only follows the choices, and the wide nodes themselves
// with their compressed copies (k_collapse_emit, all at once).  Wide nodes are numbered in queue order: queue[i] is the
// binary node of wide node i, a level's nodes are consecutive, and first[i] is the number of node i's first node child.
struct CollapseArgs {
    const rt_bvh_node *nodes;
    const uint2 *range;  // internal nodes: leaf-slot range of the subtree
    uint32_t n;          // primitives
    uint32_t width, leaf_size;
};

__device__ inline uint32_t subtree_count(const CollapseArgs &a, uint32_t b) {
    if (b >= a.n - 1 || (a.nodes[b].left == 0 && a.nodes[b].right == 0)) return 1u;
    uint2 r = a.range[b];
    return r.y - r.x + 1u;
}
__device__ inline bool is_internal(const CollapseArgs &a, uint32_t b) {
    return a.n > 1 && b < a.n - 1;
}
__device__ inline float box_area(const rt_bvh_node &nd) {
    float dx = nd.maxX - nd.minX, dy = nd.maxY - nd.minY, dz = nd.maxZ - nd.minZ;
    return dx * dy + dy * dz + dz * dx;
}

__device__ inline bool becomes_node(const CollapseArgs &a, uint32_t c) {
    return is_internal(a, c) && subtree_count(a, c) > a.leaf_size;
}

// chosen[W * b + k]: binary node b's children in a wide node (kEmpty behind the last); mask[b]: bit k is set when child k
// becomes a node itself.  Nodes that never become one (subtrees of at most leaf_size) are left out.
template <int W>
__global__ __launch_bounds__(kB) void k_collapse_choose(CollapseArgs a, uint32_t *chosen, uint8_t *mask) {
    const uint32_t b = blockIdx.x * kB + threadIdx.x;
    if (b >= max(a.n - 1u, 1u) || (b != 0u && !becomes_node(a, b))) return;
    uint32_t cand[W], l[W], r[W];  // child, its own children
    float area[W];                 // -1 when it cannot be opened
    int nc = 1;
    const auto load = [&](uint32_t c, uint32_t &id, uint32_t &left, uint32_t &right, float &ar) {
        const rt_bvh_node nd = a.nodes[c];
        id = c;
        left = nd.left;
        right = nd.right;
        ar = becomes_node(a, c) ? box_area(nd) : -1.0f;
    };
#pragma unroll
    for (int k = 0; k < W; ++k) cand[k] = kEmpty, l[k] = r[k] = 0u, area[k] = -1.0f;
    if (!is_internal(a, b)) {
        cand[0] = b;
    } else {
        const uint32_t bl = a.nodes[b].left, br = a.nodes[b].right;
        load(bl, cand[0], l[0], r[0], area[0]);
        load(br, cand[1], l[1], r[1], area[1]);
        for (nc = 2; nc < W; ++nc) {
            int best = -1;
            float best_area = -1.0f;
            uint32_t ol = 0, orr = 0;
#pragma unroll
            for (int k = 0; k < W; ++k)
                if (area[k] > best_area) best_area = area[k], best = k, ol = l[k], orr = r[k];
            if (best < 0) break;
            // the two children take the opened one's place
#pragma unroll
            for (int k = W - 1; k > 0; --k)
                if (k > best + 1) cand[k] = cand[k - 1], l[k] = l[k - 1], r[k] = r[k - 1], area[k] = area[k - 1];
            uint32_t c0, l0, r0, c1, l1, r1;
            float a0, a1;
            load(ol, c0, l0, r0, a0);
            load(orr, c1, l1, r1, a1);
#pragma unroll
            for (int k = 0; k < W; ++k) {
                if (k == best) cand[k] = c0, l[k] = l0, r[k] = r0, area[k] = a0;
                if (k == best + 1) cand[k] = c1, l[k] = l1, r[k] = r1, area[k] = a1;
            }
        }
    }
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < W; ++k) {
        if (cand[k] != kEmpty && becomes_node(a, cand[k])) m |= 1u << k;
        chosen[(size_t)b * W + k] = cand[k];
    }
    mask[b] = (uint8_t)m;
}

// [launch & 1]: the first wide node and the size of the level that the launch begins with; the other entry receives the
// next launch's.
struct CollapseState {
    uint32_t base[2], count[2];
    uint32_t depth, bad;  // levels with nodes so far; 1 when a level would not fit
};

constexpr uint32_t kLevelThreads = 1024;
constexpr uint32_t kLevelBlocks = 1024;  // at most, per launch

// A level is split into equal chunks, one per block; chunk sums are kept in three sets of kLevelBlocks words, by
// launch % 3: of the node children of this level's chunks (complete), of the next level's (added up here), and the
// one that the next launch adds to (cleared here).
__device__ inline uint32_t collapse_chunk(uint32_t count) {
    return ((count + kLevelBlocks - 1u) / kLevelBlocks + kLevelThreads - 1u) / kLevelThreads * kLevelThreads;
}

// The numbering of one level, or of as many as fit one block each (block 0 then goes through them in one
// launch, a microsecond or two for each).  Levels are launched ahead without the host reading their sizes; a
// launch past the last finds an empty one.  What bounds a level is its chain of dependent loads: queue entry ->
// choice -> the children's masks.  1 M triangles: 0.10 ms in 11 launches, and 0.05 ms for the choices (before, with
// the choices and the nodes inside the level launches: 0.47 ms in 42).
template <int W>
__global__ __launch_bounds__(kLevelThreads) void k_collapse_levels(uint32_t launch, CollapseState *st, uint32_t *queue,
                                                                   uint32_t *first, const uint32_t *chosen,
                                                                   const uint8_t *mask, uint32_t *sums,
                                                                   uint32_t max_nodes) {
    uint32_t base = st->base[launch & 1u], count = st->count[launch & 1u];
    const uint32_t *now = sums + (launch % 3u) * kLevelBlocks;
    uint32_t *next = sums + ((launch + 1u) % 3u) * kLevelBlocks, *later = sums + ((launch + 2u) % 3u) * kLevelBlocks;
    if (blockIdx.x == 0) later[threadIdx.x] = 0u;
    static_assert(kLevelBlocks == kLevelThreads, "a thread per chunk");
    const auto number = [&](uint32_t lo, uint32_t hi, uint32_t j, uint32_t next_base, uint32_t next_chunk) {
        for (uint32_t e0 = lo; e0 < hi; e0 += kLevelThreads) {
            const uint32_t e = e0 + threadIdx.x;
            uint32_t m = 0, c[W];
            if (e < hi) {
                const uint32_t b = queue[base + e];
                m = mask[b];
                for (int k = 0; k < W; ++k) c[k] = chosen[(size_t)b * W + k];
            }
            uint32_t tile, at = j + block_exclusive_scan<kLevelThreads>((uint32_t)__popc(m), &tile);
            j += tile;
            if (j > max_nodes) return j;  // cannot happen: a wide node is made from its own binary node
            // a wave's children lie in at most two chunks: their sums take two atomics instead of one a child, which
            // would go to few addresses (175 us on a level of 70,000 nodes, against 11)
            const uint32_t chunk0 = next_chunk ? (__builtin_amdgcn_readfirstlane(at) - next_base) / next_chunk : 0u;
            const uint32_t split = next_base + (chunk0 + 1u) * next_chunk;
            uint32_t below0 = 0, below1 = 0;
            if (e < hi) {
                first[base + e] = at;
                for (int k = 0; k < W; ++k)
                    if (m >> k & 1u) {
                        queue[at] = c[k];
                        if (next_chunk) (at < split ? below0 : below1) += (uint32_t)__popc((uint32_t)mask[c[k]]);
                        ++at;
                    }
            }
            if (next_chunk) {
                for (int o = 1; o < 64; o <<= 1) {
                    below0 += (uint32_t)__shfl_xor((int)below0, o);
                    below1 += (uint32_t)__shfl_xor((int)below1, o);
                }
                if (threadIdx.x % 64u == 0u) {
                    if (below0) atomicAdd(&next[chunk0], below0);
                    if (below1) atomicAdd(&next[chunk0 + 1u], below1);
                }
            }
        }
        return j;
    };
    if (count <= kLevelThreads) {
        if (blockIdx.x != 0) return;
        uint32_t depth = st->depth;
        for (; count > 0u && count <= kLevelThreads; ++depth) {
            const uint32_t end = base + count, j = number(0, count, end, 0u, 0u);
            if (j > max_nodes) {
                if (threadIdx.x == 0) st->bad = 1u;
                count = 0u;
                base = end;
                break;
            }
            __syncthreads();  // the next level's queue entries are written
            base = end;
            count = j - end;
        }
        const uint32_t chunk = collapse_chunk(count);
        for (uint32_t e0 = 0; e0 < count; e0 += kLevelThreads) {  // chunk is a multiple of kLevelThreads
            uint32_t sum;
            const uint32_t e = e0 + threadIdx.x;
            (void)block_exclusive_scan<kLevelThreads>(e < count ? (uint32_t)__popc((uint32_t)mask[queue[base + e]]) : 0u, &sum);
            if (threadIdx.x == 0) atomicAdd(&next[e0 / chunk], sum);
        }
        if (threadIdx.x == 0) {
            st->base[(launch + 1u) & 1u] = base;
            st->count[(launch + 1u) & 1u] = count;
            st->depth = depth;
        }
        return;
    }
    const uint32_t chunk = collapse_chunk(count), lo = min(blockIdx.x * chunk, count), hi = min(lo + chunk, count);
    const uint32_t v = threadIdx.x * (uint64_t)chunk < count ? now[threadIdx.x] : 0u;
    uint32_t total, before;
    (void)block_exclusive_scan<kLevelThreads>(v, &total);
    (void)block_exclusive_scan<kLevelThreads>(threadIdx.x < blockIdx.x ? v : 0u, &before);
    const uint32_t end = base + count;
    const bool bad = (uint64_t)end + total > max_nodes;  // cannot happen, as above
    if (!bad && lo < hi) (void)number(lo, hi, end + before, end, collapse_chunk(total));
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (bad) st->bad = 1u;
        st->base[(launch + 1u) & 1u] = end;
        st->count[(launch + 1u) & 1u] = bad ? 0u : total;
        st->depth += 1u;
    }
}

// min, max and bitwise or over the four lanes of a quad
__device__ inline float quad_min(float x) {
    x = fminf(x, __shfl_xor(x, 1, 4));
    return fminf(x, __shfl_xor(x, 2, 4));
}
__device__ inline float quad_max(float x) {
    x = fmaxf(x, __shfl_xor(x, 1, 4));
    return fmaxf(x, __shfl_xor(x, 2, 4));
}
__device__ inline uint32_t quad_or(uint32_t x) {
    x |= (uint32_t)__shfl_xor((int)x, 1, 4);
    return x | (uint32_t)__shfl_xor((int)x, 2, 4);
}

// A caller's node buffer may hold any boxes; compressed nodes need every box to hold what is below it.
// *bad = 1 when one does not (one store per wave).
__global__ void k_check_boxes(const rt_bvh_node *nodes, uint32_t n, const rt_triangle *tris, const rt_sphere *sph,
                              const uint32_t *slot_prim, uint32_t *bad) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2u * n - 1u) return;
    const rt_bvh_node nd = nodes[i];
    const float lo[3] = {nd.minX, nd.minY, nd.minZ}, hi[3] = {nd.maxX, nd.maxY, nd.maxZ};
    bool ok = true;
    if (i < n - 1u) {
        for (uint32_t c : {nd.left, nd.right}) {
            const rt_bvh_node b = nodes[c];
            ok = ok && lo[0] <= b.minX && b.maxX <= hi[0] && lo[1] <= b.minY && b.maxY <= hi[1] && lo[2] <= b.minZ &&
                 b.maxZ <= hi[2];
        }
    } else {
        const uint32_t p = slot_prim[i - (n - 1u)];
        for (int a = 0; a < 3; ++a) {
            if (p & RT_SPHERE_BIT) {
                const rt_sphere &s = sph[p & ~RT_SPHERE_BIT];
                const float r = fabsf(s.radius);
                ok = ok && lo[a] <= s.center[a] - r && s.center[a] + r <= hi[a];
            } else {
                const rt_triangle &t = tris[p];
                ok = ok && lo[a] <= t.v0[a] && lo[a] <= t.v1[a] && lo[a] <= t.v2[a] && t.v0[a] <= hi[a] &&
                     t.v1[a] <= hi[a] && t.v2[a] <= hi[a];
            }
        }
    }
    const unsigned long long fail = __ballot(!ok);
    if (fail != 0ull && __lane_id() == (uint32_t)__ffsll((long long)fail) - 1u) *bad = 1u;
}

// Writes the wide nodes, a lane per child, and of width-4 ones (qwide non-null) the compressed copies (rt_device.hpp) and the
// node and child that hold each leaf slot.  info[0] = 1 when some node cannot be compressed, because a plane
// is not finite or too large or a box is inverted: its exact tests do not order the two planes (one store per
// wave); info[1], info[2]: the scene's largest coordinate in magnitude and its largest extent (the root's planes);
// info[6]: among the leaves of every `sample`-th block, those that ray_pad makes a quarter larger or more on
// each axis for rays from within the scene.
// 330,000 nodes in 43 us (42 MB and 21 MB written); writing them by level, copying them and compressing the copies took
// 16 us for the copy and 69 us for the compression alone.
template <int W>
__global__ __launch_bounds__(kB) void k_collapse_emit(CollapseArgs a, uint32_t nwide, const uint32_t *queue,
                                                      const uint32_t *first, const uint32_t *chosen, const uint8_t *mask,
                                                      uint32_t *wide, uint32_t *qwide, uint32_t *slot_ref,
                                                      uint32_t *info, float inv_radius, uint32_t sample) {
    const uint64_t t = (uint64_t)blockIdx.x * kB + threadIdx.x;
    const uint32_t node = (uint32_t)(t / W), k = (uint32_t)(t % W);
    if (t / W >= nwide) return;
    const uint32_t b = queue[node], c = chosen[(size_t)b * W + k], m = mask[b];
    const float inf = __uint_as_float(0x7F800000u);
    float lo[3] = {inf, inf, inf}, hi[3] = {inf, inf, inf};
    uint32_t ce = kEmpty;
    if (c != kEmpty) {
        const rt_bvh_node nd = a.nodes[c];
        lo[0] = nd.minX; hi[0] = nd.maxX;
        lo[1] = nd.minY; hi[1] = nd.maxY;
        lo[2] = nd.minZ; hi[2] = nd.maxZ;
        if (m >> k & 1u) {
            ce = first[node] + (uint32_t)__popc(m & ((1u << k) - 1u));
        } else if (is_internal(a, c)) {
            const uint2 r = a.range[c];
            ce = leaf_entry(r.x, r.y - r.x + 1u);
        } else {
            ce = leaf_entry(c - (a.n - 1u), 1u);
        }
    }
    uint32_t *nd = wide + (size_t)node * 8u * W + k;
    for (int q = 0; q < 3; ++q) {
        nd[2 * q * W] = __float_as_uint(lo[q]);
        nd[(2 * q + 1) * W] = __float_as_uint(hi[q]);
    }
    nd[6 * W] = ce;
    nd[7 * W] = 0u;
    if (W != 4 || !qwide) return;
    bool ok = true;
    float org[3], scale[3], far = 0.0f, ext = 0.0f;
    uint32_t qlo[3], qhi[3];
    for (int q = 0; q < 3; ++q) {
        const bool have = c != kEmpty;
        ok = ok && (!have || (fabsf(lo[q]) < 0x1p24f && fabsf(hi[q]) < 0x1p24f && lo[q] <= hi[q]));
        const float mn = quad_min(have ? lo[q] : inf), mx = quad_max(have ? hi[q] : -inf);
        far = fmaxf(far, fmaxf(fabsf(mn), fabsf(mx)));
        ext = fmaxf(ext, mx - mn);
        // 248 steps over the extent; a step is no finer than the origin's rounding, at most a quarter of it
        scale[q] = fmaxf(fmaxf((mx - mn) * (1.0f / 248.0f), 0x1p-22f * fmaxf(fabsf(mn), fabsf(mx))), 0x1p-100f);
        org[q] = (float)((double)mn - 1026.0 * (double)scale[q]);
        double l = 255.0, h = 0.0;
        if (have) {
            const double s = 1.0 / (double)scale[q];
            l = floor(((double)lo[q] - (double)org[q]) * s - (1024.0 + kPlaneMargin));
            h = ceil(((double)hi[q] - (double)org[q]) * s - (1024.0 - kPlaneMargin));
            ok = ok && l >= 0.0 && h <= 255.0;
        }
        qlo[q] = quad_or(((uint32_t)l & 255u) << (8 * k));
        qhi[q] = quad_or(((uint32_t)h & 255u) << (8 * k));
    }
    const uint32_t first_of_pair = (uint32_t)__shfl((int)ce, k == 2u ? 2 : 0, 4);
    const uint32_t second_of_pair = (uint32_t)__shfl((int)ce, k == 2u ? 3 : 1, 4);
    uint4 w;
    if (k == 0u)
        w = make_uint4(__float_as_uint(org[0]), __float_as_uint(org[1]), __float_as_uint(org[2]), __float_as_uint(scale[0]));
    else if (k == 3u)
        w = make_uint4(qlo[2], qhi[2], __float_as_uint(scale[1]), __float_as_uint(scale[2]));
    else
        w = make_uint4(first_of_pair, qlo[k - 1u], second_of_pair, qhi[k - 1u]);
    reinterpret_cast<uint4 *>(qwide)[t] = w;
    if (ce != kEmpty && (ce & kLeafBit))
        for (uint32_t s = leaf_first(ce), e = s + leaf_count(ce); s < e; ++s) slot_ref[s] = (uint32_t)t;
    const unsigned long long fail = __ballot(!ok);
    if (fail != 0ull && __lane_id() == (uint32_t)__ffsll((long long)fail) - 1u) info[0] = 1u;
    if (blockIdx.x % sample == 0u) {
        const rt_bvh_node root = a.nodes[0];
        const float coord = fmaxf(fmaxf(fmaxf(fabsf(root.minX), fabsf(root.maxX)), fmaxf(fabsf(root.minY), fabsf(root.maxY))),
                                  fmaxf(fabsf(root.minZ), fabsf(root.maxZ)));
        const float pad = 0x1p-18f * coord * (1.0f + 2.0f * coord * inv_radius);
        const bool small = ce != kEmpty && (ce & kLeafBit) &&
                           fmaxf(fmaxf(hi[0] - lo[0], hi[1] - lo[1]), hi[2] - lo[2]) < 8.0f * pad;
        const unsigned long long m = __ballot(small);
        if (m != 0ull && __lane_id() == (uint32_t)__ffsll((long long)m) - 1u) atomicAdd(&info[6], (uint32_t)__popcll(m));
    }
    if (t == 0) {
        info[1] = __float_as_uint(far);
        info[2] = __float_as_uint(ext);
    }
}

// the first level is the root; info: see build_scene
__global__ void k_build_init(CollapseState *st, uint32_t *queue, uint32_t *sums, uint32_t *info, uint32_t all) {
    if (threadIdx.x == 0) *st = CollapseState{{0u, 0u}, {1u, 0u}, 0u, 0u};
    if (threadIdx.x == 0) queue[0] = 0u;
    for (uint32_t i = threadIdx.x; i < 3u * kLevelBlocks; i += blockDim.x) sums[i] = 0u;
    if (all && threadIdx.x < 7) info[threadIdx.x] = threadIdx.x == 4 || threadIdx.x == 5 ? 0xFFFFFFFFu : 0u;
}

template <class T> void upload(rt_context *ctx, DevBuf &b, const T *src, size_t count) {
    const size_t bytes = sizeof(T) * count;
    b.alloc(bytes, &ctx->pool);
    if (bytes >= HostStage::kMin) ctx->stage.copy(ctx->device, b.p, src, bytes);
    else if (count) RT_HIP(hipMemcpy(b.p, src, bytes, hipMemcpyHostToDevice));
}

// The first primitive with an index out of range, as 2 * index + kind (0 material, 1 model): the smallest into
// bad[0] for triangles and bad[1] for spheres.  One pass over the host's arrays took 1.2 ms for 1 M triangles.
__global__ void k_check_indices(const rt_triangle *tris, uint32_t ntri, const rt_sphere *sph, uint32_t nsph, uint32_t nmat,
                                uint32_t nmodels, uint32_t has_models, uint32_t *bad) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ntri + nsph) return;
    const bool tri = i < ntri;
    const uint32_t k = tri ? i : i - ntri;
    const uint32_t mat = tri ? tris[k].materialIndex : sph[k].materialIndex;
    const uint32_t model = tri ? tris[k].modelIndex : sph[k].modelIndex;
    if (mat >= nmat) atomicMin(&bad[tri ? 0 : 1], 2u * k);
    else if (has_models && model >= nmodels) atomicMin(&bad[tri ? 0 : 1], 2u * k + 1u);
}

void throw_bad_index(const uint32_t *bad) {
    for (int s = 0; s < 2; ++s)
        RT_REQUIRE(bad[s] == 0xFFFFFFFFu, (s ? "sphere " : "triangle ") + std::to_string(bad[s] >> 1) +
                                              ((bad[s] & 1u) ? ": modelIndex out of range" : ": materialIndex out of range"));
}

// Validate a caller-supplied binary node buffer and derive leaf slots and subtree ranges.
void validate_nodes(const rt_bvh_node *nodes, uint32_t n, uint32_t ntri, uint32_t nsph,
                    std::vector<uint32_t> &slot_prim, std::vector<uint2> &range, uint32_t &leaf_size) {
    slot_prim.assign(n, 0);
    range.assign(n > 1 ? n - 1 : 1, make_uint2(0, 0));
    std::vector<uint8_t> seen(2u * n - 1u, 0);
    for (uint32_t i = 0; i < n; ++i) {
        const rt_bvh_node &lf = nodes[n - 1 + i];
        RT_REQUIRE(lf.left == 0 && lf.right == 0, "node buffer: node N-1+i must be a leaf");
        if (lf.primitiveType == RT_TRIANGLE_PRIMITIVE) {
            RT_REQUIRE(lf.primitiveIndex < ntri, "node buffer: triangle index out of range");
            slot_prim[i] = lf.primitiveIndex;
        } else {
            RT_REQUIRE(lf.primitiveType == RT_SPHERE_PRIMITIVE && lf.primitiveIndex < nsph,
                       "node buffer: bad sphere leaf");
            slot_prim[i] = RT_SPHERE_BIT | lf.primitiveIndex;
        }
    }
    if (n == 1) return;
    // iterative post-order over internal nodes: reachability, no cycles, ranges
    std::vector<uint32_t> cnt(n - 1, 0);
    std::vector<uint32_t> stack;
    stack.push_back(0);
    seen[0] = 1;
    bool contiguous = true;
    std::vector<uint8_t> expanded(n - 1, 0);
    while (!stack.empty()) {
        uint32_t id = stack.back();
        const rt_bvh_node &nd = nodes[id];
        RT_REQUIRE(nd.left < 2u * n - 1u && nd.right < 2u * n - 1u && nd.left != 0 && nd.right != 0,
                   "node buffer: child index out of range");
        if (!expanded[id]) {
            expanded[id] = 1;
            for (uint32_t c : {nd.right, nd.left}) {
                RT_REQUIRE(!seen[c], "node buffer: node reachable twice (cycle or shared child)");
                seen[c] = 1;
                if (c < n - 1) stack.push_back(c);
            }
            continue;
        }
        stack.pop_back();
        uint32_t lo = 0xFFFFFFFFu, hi = 0, total = 0;
        for (uint32_t c : {nd.left, nd.right}) {
            if (c >= n - 1) { lo = std::min(lo, c - (n - 1)); hi = std::max(hi, c - (n - 1)); total += 1; }
            else { lo = std::min(lo, range[c].x); hi = std::max(hi, range[c].y); total += cnt[c]; }
        }
        range[id] = make_uint2(lo, hi);
        cnt[id] = total;
        if (hi - lo + 1 != total) contiguous = false;
    }
    for (uint32_t i = 0; i < 2u * n - 1u; ++i) RT_REQUIRE(seen[i], "node buffer: unreachable node");
    if (!contiguous) leaf_size = 1;  // multi-primitive leaves need contiguous slot ranges
}

}  // namespace

void build_scene(rt_context *ctx, Scene &sc, const rt_triangle *tris, uint32_t ntri, const rt_sphere *sph,
                 uint32_t nsph, const rt_material *mats, uint32_t nmat, const float *models, uint32_t nmodels,
                 const rt_bvh_node *nodes, uint32_t nnodes, const rt_build_options &opts) {
    const uint32_t W = opts.width ? opts.width : 4u;
    RT_REQUIRE(W == 2 || W == 4 || W == 8, "width must be 2, 4 or 8");
    uint32_t L = opts.leaf_size ? opts.leaf_size : 1u;
    RT_REQUIRE(L >= 1 && L <= 8, "leaf_size must be 1..8");
    const uint64_t n64 = (uint64_t)ntri + nsph;
    RT_REQUIRE(n64 < (1ull << 27) - 16, "too many primitives (max 2^27-17)");
    const uint32_t n = (uint32_t)n64;
    RT_REQUIRE(ntri == 0 || tris, "tris is NULL");
    RT_REQUIRE(nsph == 0 || sph, "spheres is NULL");
    RT_REQUIRE(nmat == 0 || mats, "materials is NULL");
    RT_REQUIRE(nmodels == 0 || models, "models is NULL");
    const bool wrong_nodes = nodes && !(n > 0 && nnodes == 2u * n - 1u);  // reported after a bad index

    sc.ntri = ntri; sc.nsph = nsph; sc.nmat = nmat; sc.nprim = n;
    sc.width = W; sc.flags = opts.flags;
    upload(ctx, sc.materials, mats, nmat);
    if (n == 0) {
        RT_REQUIRE(!wrong_nodes, "node buffer must hold 2N-1 nodes");
        sc.nwide = 0; sc.wide_depth = 0; sc.stack_bound = 0; sc.leaf_size = L;
        return;
    }
    hipStream_t st = nullptr;
    Event ev0, ev1;
    DevBuf dtris, dsph, dmodels;
    upload(ctx, dtris, tris, ntri);
    upload(ctx, dsph, sph, nsph);
    RT_HIP(hipEventRecord(ev0.e, st));
    if (models) {
        upload(ctx, dmodels, models, 16ull * nmodels);
        k_model_to_world<<<grid_for(n), kB, 0, st>>>(dtris.as<rt_triangle>(), ntri, dsph.as<rt_sphere>(), nsph,
                                                     dmodels.as<float>(), nmodels);
    }
    // centre-based u, v of every sphere (raytraceBVH.comp:172-173), from its world-space centre
    DevBuf duv;
    float min_radius = std::numeric_limits<float>::max();
    if (nsph) {
        std::vector<rt_sphere> world(sph, sph + nsph);
        if (models)  // as k_model_to_world, the same operations in the same order
            for (rt_sphere &s : world)
                if (s.modelIndex < nmodels) mat_vec1(models + 16u * s.modelIndex, s.center);
        std::vector<float2> uv(nsph);
        for (uint32_t i = 0; i < nsph; ++i) {
            sphere_uv(world[i].center, uv[i].x, uv[i].y);
            min_radius = std::fmin(min_radius, std::fabs(world[i].radius));
        }
        upload(ctx, duv, uv.data(), nsph);
    }
    sc.slot_prim.alloc(sizeof(uint32_t) * n, &ctx->pool);
    sc.slot_mat.alloc(sizeof(uint32_t) * n, &ctx->pool);
    sc.records.alloc(sizeof(LeafRecord) * n, &ctx->pool);
    // every temporary of the build from one block of the scratch cache
    const bool keep_binary = (opts.flags & RT_BUILD_KEEP_BINARY) != 0;
    const uint32_t max_nodes = std::max<uint32_t>(n - 1, 1);
    const uint64_t sort_bytes = round256(24ull * kBoundsBlocks) + 2 * round256(4ull * n) +
                                std::max(sort_temp_bytes(n), refit_temp_bytes(n));
    const uint64_t collapse_bytes = round256(4ull * W * max_nodes) + round256(4ull * max_nodes) + round256(max_nodes);
    const uint64_t temp_bytes = (keep_binary ? 0 : round256(sizeof(rt_bvh_node) * (2ull * n - 1))) +
                                round256(sizeof(uint2) * max_nodes) + round256(sizeof(CollapseState)) + round256(28) +
                                round256(4ull * max_nodes) + round256(12ull * kLevelBlocks) +
                                std::max(sort_bytes, collapse_bytes);
    Temps tmp(ctx, temp_bytes, st);
    DevBuf kept;  // the binary nodes, when they stay resident
    rt_bvh_node *binary = nullptr;
    if (keep_binary) {
        kept.alloc(sizeof(rt_bvh_node) * (2ull * n - 1), &ctx->pool);
        binary = kept.as<rt_bvh_node>();
    } else {
        binary = tmp.take<rt_bvh_node>(2ull * n - 1);
    }
    uint2 *range = tmp.take<uint2>(max_nodes);
    CollapseState *state = tmp.take<CollapseState>(1);
    uint32_t *info = tmp.take<uint32_t>(7);  // k_collapse_emit's words 0..2 and 6, k_leaves' NaN flag, k_check_indices' two words
    uint32_t *queue = tmp.take<uint32_t>(max_nodes), *sums = tmp.take<uint32_t>(3ull * kLevelBlocks);
    k_build_init<<<1, 1024, 0, st>>>(state, queue, sums, info, 1u);
    k_check_indices<<<grid_for(n), kB, 0, st>>>(dtris.as<rt_triangle>(), ntri, dsph.as<rt_sphere>(), nsph, nmat, nmodels,
                                                models ? 1u : 0u, info + 4);
    const uint64_t mk = tmp.mark();
    if (nodes) {
        uint32_t bad[2];
        RT_HIP(hipMemcpy(bad, info + 4, sizeof bad, hipMemcpyDeviceToHost));
        throw_bad_index(bad);
        RT_REQUIRE(!wrong_nodes, "node buffer must hold 2N-1 nodes");
        std::vector<uint32_t> hslots;
        std::vector<uint2> hrange;
        validate_nodes(nodes, n, ntri, nsph, hslots, hrange, L);
        RT_HIP(hipMemcpy(binary, nodes, sizeof(rt_bvh_node) * (2ull * n - 1), hipMemcpyHostToDevice));
        RT_HIP(hipMemcpy(sc.slot_prim.p, hslots.data(), sizeof(uint32_t) * n, hipMemcpyHostToDevice));
        RT_HIP(hipMemcpy(range, hrange.data(), sizeof(uint2) * hrange.size(), hipMemcpyHostToDevice));
        k_records<<<grid_for(n), kB, 0, st>>>(dtris.as<rt_triangle>(), dsph.as<rt_sphere>(), duv.as<float2>(),
                                              sc.slot_prim.as<uint32_t>(), n, sc.records.as<LeafRecord>(),
                                              sc.slot_mat.as<uint32_t>());
    } else {
        uint32_t *partial = tmp.take<uint32_t>(6ull * kBoundsBlocks);
        uint32_t *keys = tmp.take<uint32_t>(n), *vals = tmp.take<uint32_t>(n);
        const uint32_t g = std::min<uint32_t>(grid_for(n), kBoundsBlocks);
        k_centroid_bounds<<<g, kB, 0, st>>>(dtris.as<rt_triangle>(), ntri, dsph.as<rt_sphere>(), n, partial);
        k_morton<<<grid_for(n), kB, 0, st>>>(dtris.as<rt_triangle>(), ntri, dsph.as<rt_sphere>(), n, partial, g,
                                             (opts.flags & RT_BUILD_REFERENCE_MORTON) ? 1u : 0u, keys, vals);
        const uint64_t sort_mk = tmp.mark();
        sort_pairs(keys, vals, n, st, tmp);
        if (n > 1) k_karras<<<grid_for(n - 1), kB, 0, st>>>(keys, (int)n, binary, range);
        k_leaves<<<grid_for(n), kB, 0, st>>>(dtris.as<rt_triangle>(), ntri, dsph.as<rt_sphere>(), duv.as<float2>(), vals,
                                             (opts.flags & RT_BUILD_REFERENCE_LEAVES) ? 1u : 0u, n,
                                             sc.slot_prim.as<uint32_t>(), binary + (n - 1), sc.records.as<LeafRecord>(),
                                             sc.slot_mat.as<uint32_t>(), info + 3);
        tmp.release(sort_mk);
        if (n > 1) refit(binary, range, n, st, tmp);
        tmp.release(mk);
    }
    RT_HIP(hipGetLastError());

    CollapseArgs a{binary, range, n, W, L};
    uint32_t *chosen = tmp.take<uint32_t>((uint64_t)W * max_nodes), *first = tmp.take<uint32_t>(max_nodes);
    uint8_t *mask = tmp.take<uint8_t>(max_nodes);
    struct { CollapseState state; uint32_t pad[58]; uint32_t info[6]; } out{};  // as the two lie in the temporaries
    static_assert(sizeof(CollapseState) == 24 && offsetof(decltype(out), info) == 256, "state and info are read together");
    const auto with_width = [&](auto f) {
        if (W == 2) f(std::integral_constant<int, 2>{});
        else if (W == 4) f(std::integral_constant<int, 4>{});
        else f(std::integral_constant<int, 8>{});
    };
    const auto collapse = [&] {
        // The levels of up to kLevelThreads nodes at both ends take one launch each, and about log2(n) / 2 levels lie
        // between them; the host looks after these and then after every four more.
        uint32_t launch = 0, ahead = 1;
        for (uint64_t m = n; m > 1024; m >>= 1) ++ahead;
        uint64_t widest = 1;  // no level can hold more nodes
        with_width([&](auto w) { k_collapse_choose<w.value><<<grid_for(max_nodes), kB, 0, st>>>(a, chosen, mask); });
        do {
            for (uint32_t end = launch + ahead; launch < end; ++launch) {
                widest = launch == 0 ? std::min<uint64_t>(kLevelThreads * W, max_nodes) : std::min<uint64_t>(widest * W, max_nodes);
                const uint32_t grid = launch == 0 ? 1u : std::min<uint32_t>((widest + kLevelThreads - 1u) / kLevelThreads, kLevelBlocks);
                with_width([&](auto w) {
                    k_collapse_levels<w.value><<<grid, kLevelThreads, 0, st>>>(launch, state, queue, first, chosen, mask, sums,
                                                                              max_nodes);
                });
            }
            ahead = 4;
            RT_HIP(hipMemcpy(&out, state, sizeof out, hipMemcpyDeviceToHost));
        } while (out.state.count[launch & 1u] != 0u);
    };
    collapse();
    throw_bad_index(out.info + 4);
    if (out.info[3] && n > 1) {  // NaN planes: unions in the tree's own order, then the collapse again
        DevBuf other;
        other.alloc_own(sizeof(rt_bvh_node) * (2ull * n - 1), ctx->pool);
        for (int pass = 0; pass < 64; pass += 2) {
            k_refit_pass<<<grid_for(2ull * n - 1), kB, 0, st>>>(binary, other.as<rt_bvh_node>(), n);
            k_refit_pass<<<grid_for(2ull * n - 1), kB, 0, st>>>(other.as<rt_bvh_node>(), binary, n);
        }
        k_build_init<<<1, 1024, 0, st>>>(state, queue, sums, info, 0u);
        collapse();
        RT_HIP(hipStreamSynchronize(st));  // `other` is freed
    }
    RT_REQUIRE(!out.state.bad, "internal: wide node count exceeds bound");
    const uint32_t depth = out.state.depth;
    sc.nwide = std::max(out.state.base[0], out.state.base[1]);
    sc.wide.alloc((size_t)sc.nwide * 32u * W, &ctx->pool);
    if (W == 4) {
        sc.qwide.alloc((size_t)sc.nwide * 64u, &ctx->pool);
        sc.slot_ref.alloc(sizeof(uint32_t) * n, &ctx->pool);
        if (nodes)
            k_check_boxes<<<grid_for(2ull * n - 1), kB, 0, st>>>(binary, n, dtris.as<rt_triangle>(), dsph.as<rt_sphere>(),
                                                                 sc.slot_prim.as<uint32_t>(), info);
    }
    const float inv_radius = nsph ? 1.0f / min_radius : 0.0f;
    const uint32_t emit_blocks = grid_for((uint64_t)sc.nwide * W), sample = (emit_blocks + 255u) / 256u;
    with_width([&](auto w) {
        k_collapse_emit<w.value><<<emit_blocks, kB, 0, st>>>(a, sc.nwide, queue, first, chosen, mask, sc.wide.as<uint32_t>(),
                                                             sc.qwide.as<uint32_t>(), sc.slot_ref.as<uint32_t>(), info, inv_radius,
                                                             sample);
    });
    RT_HIP(hipGetLastError());
    RT_HIP(hipEventRecord(ev1.e, st));
    RT_HIP(hipEventSynchronize(ev1.e));
    float ms = 0.0f;
    RT_HIP(hipEventElapsedTime(&ms, ev0.e, ev1.e));

    if (W == 4) {
        struct { uint32_t bad; float far, extent; uint32_t pad[3]; uint32_t small; } whole{};
        RT_HIP(hipMemcpy(&whole, info, sizeof whole, hipMemcpyDeviceToHost));
        // see Scene::reach: origins may lie this far outside the scene's coordinates
        const float reach = std::min(400.0f * whole.extent, 512.0f * min_radius);
        sc.reach = Reach{whole.far + reach, whole.far, inv_radius};
        // Where a third of the leaves or more are hardly larger than a hit's rounding, the larger boxes hold too much
        // (32,000 triangles of 0.03, shifted by 1,000 from the origin: 4.6 M paths 1.5 ms and 1.5 over the exact nodes; by 3,000 2.2
        // and 1.6, by 10,000 7.4 and 1.9).
        const uint32_t sampled = std::min<uint32_t>(sc.nwide, (emit_blocks + sample - 1u) / sample * (kB / 4u));
        if (whole.bad || whole.small >= sampled || !(reach >= 1.8f * whole.extent)) {  // also where a sphere is too small to be seen across the scene
            sc.qwide.release();
            sc.slot_ref.release();
        }
    }
    sc.wide_depth = depth;
    sc.leaf_size = L;
    sc.stack_bound = (W - 1u) * depth + 1u;
    sc.build_ms = ms;
    if (keep_binary) sc.binary = std::move(kept);
    sc.tris = std::move(dtris);  // world space: the ray queries' refinement reads the vertices
    sc.spheres = std::move(dsph);
}

}  // namespace rtgpu
