// bvh.hip — GPU LBVH builder for the BLASes and the instance TLAS (gfx950).
//
// Replaces the driver's acceleration-structure builds that the reference
// requests in RayTracer::createBottomLevelAS / buildBlas (rt.cpp:142-370) and
// RayTracer::buildTlas / updateTlas (rt.cpp:372-495).
//
// One batched build handles every geometry at once (segments): primitives of
// segment s get 64-bit keys (s << 30 | morton30(centroid)), one radix sort
// orders all of them and the Karras (2012) hierarchy is emitted per segment,
// each child box as the union of its range of sorted leaves.
//   k_seg_bounds   centroid bounds per segment (ordered-int atomics, one set
//                  per wave where its primitives are of one segment)
//   k_morton       30-bit Morton codes, key = seg << 30 | code
//   radix sort     8-bit digits: per-tile histogram, one scan block per
//                  digit, stable scatter with wave64 ballot multi-split ranks
//   k_pyramid      boxes of the aligned runs of 2, 4, 8, ... sorted leaves
//   k_karras       internal nodes (ranges, splits, child refs) and, from the
//                  pyramid, their child boxes
#include "kf_internal.h"
#include <algorithm>
#include <array>
#include <climits>
#include <cmath>
#include <cstring>
#include <map>

namespace kf {

#define KF_DEV_INLINE __device__ __forceinline__

namespace {

constexpr int kSortThreads = 256;
constexpr int kSortItems = 8;
constexpr int kSortTile = kSortThreads * kSortItems;
constexpr int kDigitBits = 8;
constexpr int kDigits = 1 << kDigitBits;

__device__ __forceinline__ int f2ord(float f) {
    int i = __float_as_int(f);
    return i >= 0 ? i : i ^ 0x7fffffff;
}
__device__ __forceinline__ float ord2f(int o) { return __int_as_float(o >= 0 ? o : o ^ 0x7fffffff); }

// Centroid bounds start empty: lo = ord(+inf), hi = ord(-inf) per segment.
__global__ void k_seg_init(uint32_t n_seg, int* __restrict__ sb) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 6 * n_seg) return;
    sb[i] = (i % 6) < 3 ? 0x7f800000 : (int)(0xff800000u ^ 0x7fffffffu);
}

// Primitives of a segment are consecutive, so nearly every wave holds one
// segment: it reduces the six bounds across its lanes and lane k updates
// bound k.  With an atomic per primitive and bound the build of 1.3 M
// triangles in 256 segments spent 3.6 ms here, now 34 us.
__global__ void k_seg_bounds(uint32_t n, const float4* __restrict__ lo, const float4* __restrict__ hi,
                             const uint32_t* __restrict__ seg, int* __restrict__ sb /* 6 per seg */) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u;
    const float4 a = i < n ? lo[i] : make_float4(INFINITY, 0.f, 0.f, 0.f);
    const float4 b = i < n ? hi[i] : make_float4(-INFINITY, 0.f, 0.f, 0.f);
    const bool full = a.x <= b.x;  // not an empty box
    const uint32_t s = i < n ? seg[i] : 0u;
    const unsigned long long m = __ballot(full);
    if (!m) return;
    const float c[3] = {0.5f * (a.x + b.x), 0.5f * (a.y + b.y), 0.5f * (a.z + b.z)};
    const int first = __ffsll((long long)m) - 1;
    const uint32_t s0 = (uint32_t)__builtin_amdgcn_readlane((int)s, first);
    if (__ballot(full && s != s0) == 0ull) {
        int mine = 0;
        for (int k = 0; k < 3; ++k) {
            int l = full ? f2ord(c[k]) : INT_MAX, h = full ? f2ord(c[k]) : INT_MIN;
            for (int off = 32; off > 0; off >>= 1) {
                l = min(l, __shfl_xor(l, off));
                h = max(h, __shfl_xor(h, off));
            }
            mine = lane == (uint32_t)k ? l : lane == (uint32_t)k + 3u ? h : mine;
        }
        if (lane < 3u) atomicMin(&sb[6 * s0 + lane], mine);
        else if (lane < 6u) atomicMax(&sb[6 * s0 + lane], mine);
        return;
    }
    if (!full) return;
    for (int k = 0; k < 3; ++k) {
        atomicMin(&sb[6 * s + k], f2ord(c[k]));
        atomicMax(&sb[6 * s + 3 + k], f2ord(c[k]));
    }
}

__device__ __forceinline__ uint32_t spread10(uint32_t v) {
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// 30-bit Morton code of centroid c in the bounds [l, h]; 0 for an empty box.
__device__ __forceinline__ uint32_t morton30(bool full, const float c[3], const float l[3], const float h[3]) {
    if (!full) return 0u;
    uint32_t q[3];
    for (int k = 0; k < 3; ++k) {
        float e = h[k] - l[k];
        float u = e > 0.0f ? (c[k] - l[k]) / e : 0.5f;
        u = fminf(fmaxf(u, 0.0f), 1.0f);
        q[k] = min((uint32_t)(u * 1024.0f), 1023u);
    }
    return (spread10(q[0]) << 2) | (spread10(q[1]) << 1) | spread10(q[2]);
}

__global__ void k_morton(uint32_t n, const float4* __restrict__ lo, const float4* __restrict__ hi,
                         const uint32_t* __restrict__ seg, const int* __restrict__ sb,
                         unsigned long long* __restrict__ keys, uint32_t* __restrict__ vals) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t s = seg[i];
    float4 a = lo[i], b = hi[i];
    const float c[3] = {0.5f * (a.x + b.x), 0.5f * (a.y + b.y), 0.5f * (a.z + b.z)};
    float l[3], h[3];
    for (int k = 0; k < 3; ++k) {
        l[k] = ord2f(sb[6 * s + k]);
        h[k] = ord2f(sb[6 * s + 3 + k]);
    }
    keys[i] = ((unsigned long long)s << 30) | morton30(a.x <= b.x, c, l, h);
    vals[i] = i;
}

// ---------------------------------------------------------------- radix sort
__global__ __launch_bounds__(kSortThreads) void k_rs_hist(uint32_t n, const unsigned long long* __restrict__ keys,
                                                          int shift, uint32_t n_tiles, uint32_t* __restrict__ hist) {
    __shared__ uint32_t cnt[kDigits];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    uint32_t base = blockIdx.x * kSortTile;
    for (int r = 0; r < kSortItems; ++r) {
        uint32_t i = base + r * kSortThreads + threadIdx.x;
        if (i < n) atomicAdd(&cnt[(keys[i] >> shift) & (kDigits - 1)], 1u);
    }
    __syncthreads();
    hist[(size_t)threadIdx.x * n_tiles + blockIdx.x] = cnt[threadIdx.x];
}

// Exclusive scan of each digit's tile counts (block d: row d of the
// histogram) and the digit's total; k_rs_scatter adds the digits before its
// own.  One block over all n_tiles x 256 counts took 0.30 ms per pass at 640
// tiles (1.3 M keys), 256 blocks 5 us.
__global__ __launch_bounds__(kSortThreads) void k_rs_scan(uint32_t n_tiles, uint32_t* __restrict__ hist,
                                                          uint32_t* __restrict__ total) {
    __shared__ uint32_t wsum[kSortThreads / 64];
    uint32_t* h = hist + (size_t)blockIdx.x * n_tiles;
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    uint32_t run = 0;
    for (uint32_t base = 0; base < n_tiles; base += kSortThreads) {
        const uint32_t i = base + threadIdx.x;
        const uint32_t v = i < n_tiles ? h[i] : 0u;
        uint32_t x = v;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)x, off);
            if (lane >= (uint32_t)off) x += y;
        }
        if (lane == 63u) wsum[w] = x;
        __syncthreads();
        uint32_t before = run, sum = 0;
        for (uint32_t k = 0; k < kSortThreads / 64; ++k) {
            if (k < w) before += wsum[k];
            sum += wsum[k];
        }
        if (i < n_tiles) h[i] = before + x - v;
        run += sum;
        __syncthreads();
    }
    if (threadIdx.x == 0) total[blockIdx.x] = run;
}

__global__ __launch_bounds__(kSortThreads) void k_rs_scatter(uint32_t n, const unsigned long long* __restrict__ kin,
                                                             const uint32_t* __restrict__ vin, int shift,
                                                             uint32_t n_tiles, const uint32_t* __restrict__ hist,
                                                             const uint32_t* __restrict__ total,
                                                             unsigned long long* __restrict__ kout,
                                                             uint32_t* __restrict__ vout) {
    constexpr int kWaves = kSortThreads / 64;
    static_assert(kSortThreads == kDigits, "one thread per digit");
    __shared__ uint32_t gbase[kDigits];
    __shared__ uint32_t run[kDigits];
    __shared__ uint32_t wcnt[kWaves][kDigits];
    const uint32_t t = threadIdx.x, lane = t & 63, w = t >> 6;
    {  // keys of smaller digits, then those of this digit in earlier tiles
        const uint32_t v = total[t];
        uint32_t x = v;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)x, off);
            if (lane >= (uint32_t)off) x += y;
        }
        if (lane == 63u) run[w] = x;
        __syncthreads();
        uint32_t before = x - v;
        for (uint32_t k = 0; k < w; ++k) before += run[k];
        __syncthreads();
        gbase[t] = before + hist[(size_t)t * n_tiles + blockIdx.x];
    }
    run[t] = 0;
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    uint32_t base = blockIdx.x * kSortTile;
    for (int r = 0; r < kSortItems; ++r) {
        for (int k = 0; k < kWaves; ++k) wcnt[k][t] = 0;
        __syncthreads();
        uint32_t i = base + r * kSortThreads + t;
        bool valid = i < n;
        unsigned long long key = valid ? kin[i] : 0ull;
        uint32_t d = (uint32_t)(key >> shift) & (kDigits - 1);
        unsigned long long mask = __ballot(valid);
#pragma unroll
        for (int b = 0; b < kDigitBits; ++b) {
            bool bit = (d >> b) & 1u;
            unsigned long long m = __ballot(bit);
            mask &= bit ? m : ~m;
        }
        uint32_t rank = __popcll(mask & lt);
        if (valid && rank == 0) wcnt[w][d] = __popcll(mask);
        __syncthreads();
        {
            uint32_t s = run[t];
            for (int k = 0; k < kWaves; ++k) {
                uint32_t c = wcnt[k][t];
                wcnt[k][t] = s;
                s += c;
            }
            run[t] = s;
        }
        __syncthreads();
        if (valid) {
            uint32_t pos = gbase[d] + wcnt[w][d] + rank;
            if (pos < n) {
                kout[pos] = key;
                vout[pos] = vin[i];
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------- boxes
// Level 0 of a pyramid holds the boxes of the sorted leaves, entry i of level
// k + 1 the union of entries 2i and 2i + 1 of level k.  The box of a range of
// leaves is then the union of at most two entries per level, so a node's
// child boxes follow from its range alone: no bottom-up walk, in which the
// second of two children, on whatever XCD, has to see the first one's box
// (with an acquire-release atomic per node the walk took 5.3 ms for 1.3 M
// triangles; k_pyramid takes 44 us and the boxes 48 us of k_karras).
// Unions are minima and maxima, so the boxes are the same bits.
struct Box {
    float4 lo, hi;
};
constexpr int kMaxLevels = 32;
struct Pyramid {
    Box* at = nullptr;
    uint32_t off[kMaxLevels] = {};  // first entry of each level
    int levels = 0;
};
KF_DEV_INLINE Box box_union(const Box& a, const Box& b) {
    Box r;
    r.lo = make_float4(fminf(a.lo.x, b.lo.x), fminf(a.lo.y, b.lo.y), fminf(a.lo.z, b.lo.z), 0.f);
    r.hi = make_float4(fmaxf(a.hi.x, b.hi.x), fmaxf(a.hi.y, b.hi.y), fmaxf(a.hi.z, b.hi.z), 0.f);
    return r;
}
KF_DEV_INLINE Box box_empty() {
    return {make_float4(INFINITY, INFINITY, INFINITY, 0.f), make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f)};
}
// Union of leaves l .. r (l <= r).
KF_DEV_INLINE Box range_box(const Pyramid& P, uint32_t l, uint32_t r) {
    Box b = P.at[l];
    if (l == r) return b;
    b = box_empty();
    for (int k = 0; k < P.levels && l <= r; ++k) {
        const Box* L = P.at + P.off[k];
        if (l & 1u) b = box_union(b, L[l++]);
        if (!(r & 1u)) {
            b = box_union(b, L[r]);
            if (r == 0u) break;
            --r;
        }
        l >>= 1;
        r >>= 1;
    }
    return b;
}

// Nine levels above level k0, whose n entries are there already, or (first)
// are gathered here: entry i is primitive order[i] (order: may be null, the
// identity).  Each block reduces 512 entries in LDS.
constexpr int kPyrThreads = 256, kPyrItems = 2 * kPyrThreads, kPyrLevels = 9;
__global__ __launch_bounds__(kPyrThreads) void k_pyramid(Pyramid P, int k0, uint32_t n, bool first,
                                                        const uint32_t* __restrict__ order,
                                                        const float4* __restrict__ lo, const float4* __restrict__ hi) {
    __shared__ Box s[kPyrThreads];
    const uint32_t t = threadIdx.x;
    Box* L0 = P.at + P.off[k0];
    Box b = box_empty();
    for (int j = 0; j < 2; ++j) {
        const uint32_t i = blockIdx.x * kPyrItems + 2u * t + j;
        if (i >= n) break;
        Box c;
        if (first) {
            const uint32_t p = order ? order[i] : i;
            c.lo = lo[p];
            c.hi = hi[p];
            L0[i] = c;
        } else {
            c = L0[i];
        }
        b = box_union(b, c);
    }
    uint32_t m = n;
    for (int k = 1; k <= kPyrLevels && k0 + k < P.levels; ++k) {
        m = (m + 1u) >> 1;
        const uint32_t w = kPyrItems >> k, i = blockIdx.x * w + t;  // this block's entries of the level
        if (t < w && i < m) P.at[P.off[k0 + k] + i] = b;
        s[t] = b;
        __syncthreads();
        if (t < w / 2) b = box_union(s[2 * t], s[2 * t + 1]);
        __syncthreads();
    }
}

// ---------------------------------------------------------------- Karras
// Node i of the hierarchy over n >= 2 sorted keys: its leaves first .. last,
// the left child's being first .. split.
struct KarrasNode {
    int first, split, last;
};
template <class Key>
KF_DEV_INLINE KarrasNode karras_node(Key key, int n, int i) {
    auto delta = [&](int a, int b) {
        if (b < 0 || b >= n) return -1;
        const unsigned long long x = key(a) ^ key(b);
        return x ? __clzll(x) : 64 + __clz((uint32_t)(a ^ b));
    };
    const int d = (delta(i, i + 1) - delta(i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = delta(i, i - d);
    int lmax = 2;
    while (delta(i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = delta(i, j);
    int sp = 0;
    int div = 2;
    int t = (l + div - 1) / div;
    while (true) {
        if (delta(i, i + (sp + t) * d) > dnode) sp += t;
        if (t == 1) break;
        div <<= 1;
        t = (l + div - 1) / div;
    }
    return {min(i, j), i + sp * d + min(d, 0), max(i, j)};
}

// A node from its range of leaves: child boxes, child refs and (d.zw) the
// range itself, first and last leaf in sorted order, which a refit needs.
KF_DEV_INLINE Node make_node(const Pyramid& P, uint32_t first, uint32_t split, uint32_t last, int lref, int rref) {
    const Box L = range_box(P, first, split), R = range_box(P, split + 1u, last);
    Node n;
    n.a = make_float4(L.lo.x, L.hi.x, L.lo.y, L.hi.y);
    n.b = make_float4(R.lo.x, R.hi.x, R.lo.y, R.hi.y);
    n.c = make_float4(L.lo.z, L.hi.z, R.lo.z, R.hi.z);
    n.d = make_int4(lref, rref, (int)first, (int)last);
    return n;
}

__global__ void k_karras(uint32_t n, const unsigned long long* __restrict__ keys, const uint32_t* __restrict__ order,
                         const uint32_t* __restrict__ seg_off, const uint32_t* __restrict__ node_off, Pyramid P,
                         Node* __restrict__ nodes, int leaf_is_slot) {
    uint32_t gi = blockIdx.x * blockDim.x + threadIdx.x;
    if (gi >= n) return;
    uint32_t s = (uint32_t)(keys[gi] >> 30);
    uint32_t so = seg_off[s];
    int ns = (int)(seg_off[s + 1] - so);
    int i = (int)(gi - so);
    if (i >= ns - 1) return;
    const unsigned long long* k = keys + so;
    const KarrasNode kn = karras_node([&](int a) { return k[a]; }, ns, i);
    const int first = kn.first, gamma = kn.split, last = kn.last, nb = (int)node_off[s];
    auto leaf = [&](int q) { return ~(leaf_is_slot ? (int)so + q : (int)order[so + q]); };
    const int lref = first == gamma ? leaf(gamma) : nb + gamma;
    const int rref = last == gamma + 1 ? leaf(gamma + 1) : nb + gamma + 1;
    nodes[nb + i] = make_node(P, so + first, so + gamma, so + last, lref, rref);
}

__global__ void k_seg_root(uint32_t n_seg, const uint32_t* __restrict__ seg_off, const uint32_t* __restrict__ node_off,
                           const uint32_t* __restrict__ order, int* __restrict__ root, int leaf_is_slot) {
    uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n_seg) return;
    uint32_t ns = seg_off[s + 1] - seg_off[s];
    if (ns == 0) root[s] = kEmptyRef;
    else if (ns == 1) root[s] = ~(leaf_is_slot ? (int)seg_off[s] : (int)order[seg_off[s]]);
    else root[s] = (int)node_off[s];
}

template <class T> T* dalloc(size_t n) {
    T* p = nullptr;
    if (n) KF_CHECK(hipMallocAsync((void**)&p, n * sizeof(T), stream()));
    return p;
}
template <class T> void dfree(T* p) {
    if (p) KF_CHECK(hipFreeAsync(p, stream()));
}

inline uint32_t blocks(uint32_t n, uint32_t b) { return (n + b - 1) / b; }

// The pyramid over n > 0 leaves with the boxes lo / hi of order[0 .. n), in
// `at` (pyramid_size(n) boxes).
size_t pyramid_size(uint32_t n) { return 2 * (size_t)n + kMaxLevels; }
Pyramid build_pyramid(uint32_t n, const uint32_t* order, const float4* lo, const float4* hi, Box* at, hipStream_t st) {
    Pyramid P;
    uint32_t len[kMaxLevels], total = 0;
    for (uint32_t m = n;; m = (m + 1u) / 2u) {
        len[P.levels] = m;
        P.off[P.levels++] = total;
        total += m;
        if (m == 1u) break;
    }
    P.at = at;
    for (int k = 0; k == 0 || k + 1 < P.levels; k += kPyrLevels)
        k_pyramid<<<blocks(len[k], kPyrItems), kPyrThreads, 0, st>>>(P, k, len[k], k == 0, order, lo, hi);
    return P;
}

// ---------------------------------------------------------------- BLAS inputs
__global__ void k_tri_geom(uint32_t n_tri, uint32_t n_geom, const uint32_t* __restrict__ toff,
                           uint32_t* __restrict__ tri_geom) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_tri) return;
    uint32_t lo = 0, hi = n_geom;  // largest g with toff[g] <= i
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (toff[mid] <= i) lo = mid; else hi = mid;
    }
    tri_geom[i] = lo;
}

__global__ void k_tri_bounds(uint32_t n_tri, const float4* __restrict__ verts, const uint32_t* __restrict__ idx,
                             const uint32_t* __restrict__ voff, const uint32_t* __restrict__ tri_geom,
                             float4* __restrict__ lo, float4* __restrict__ hi) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_tri) return;
    uint32_t vb = voff[tri_geom[i]];
    float3 p[3];
    for (int k = 0; k < 3; ++k) {
        float4 v = verts[3 * (size_t)(vb + idx[3 * (size_t)i + k])];
        p[k] = make_float3(v.x, v.y, v.z);
    }
    lo[i] = make_float4(fminf(p[0].x, fminf(p[1].x, p[2].x)), fminf(p[0].y, fminf(p[1].y, p[2].y)),
                        fminf(p[0].z, fminf(p[1].z, p[2].z)), 0.f);
    hi[i] = make_float4(fmaxf(p[0].x, fmaxf(p[1].x, p[2].x)), fmaxf(p[0].y, fmaxf(p[1].y, p[2].y)),
                        fmaxf(p[0].z, fmaxf(p[1].z, p[2].z)), 0.f);
}

// Triangle slot s, by axis: tri[3s + a] = (v0[a], v1[a], v2[a], w), w the
// local prim id bits on line 0 and 0 on lines 1-2.  Line a minus the ray
// origin's axis a is what a node's low planes subtract too, so the traversal
// step shares those differences between its node and triangle tests.
KF_DEV_INLINE void put_tri_slot(float4* __restrict__ tri, size_t s, const float3 p[3], uint32_t prim) {
    tri[3 * s + 0] = make_float4(p[0].x, p[1].x, p[2].x, __uint_as_float(prim));
    tri[3 * s + 1] = make_float4(p[0].y, p[1].y, p[2].y, 0.f);
    tri[3 * s + 2] = make_float4(p[0].z, p[1].z, p[2].z, 0.f);
}
// Box of triangle slot s.
KF_DEV_INLINE void tri_slot_box(const float4* __restrict__ tri, size_t s, float lo[3], float hi[3]) {
    for (int a = 0; a < 3; ++a) {
        const float4 l = tri[3 * s + a];
        lo[a] = fminf(l.x, fminf(l.y, l.z));
        hi[a] = fmaxf(l.x, fmaxf(l.y, l.z));
    }
}

// Triangle slots in BVH leaf order.
__global__ void k_tri_reorder(uint32_t n_tri, const uint32_t* __restrict__ order, const float4* __restrict__ verts,
                              const uint32_t* __restrict__ idx, const uint32_t* __restrict__ voff,
                              const uint32_t* __restrict__ toff, const uint32_t* __restrict__ tri_geom,
                              float4* __restrict__ tri) {
    uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n_tri) return;
    uint32_t i = order[s];
    uint32_t g = tri_geom[i];
    uint32_t vb = voff[g];
    float3 p[3];
    for (int k = 0; k < 3; ++k) {
        const float4 v = verts[3 * (size_t)(vb + idx[3 * (size_t)i + k])];
        p[k] = make_float3(v.x, v.y, v.z);
    }
    put_tri_slot(tri, s, p, i - toff[g]);
}

// Object-space bounds of each BLAS (union of the root's children, or the
// single triangle).
__global__ void k_blas_box(uint32_t n_geom, const int* __restrict__ root, const Node* __restrict__ nodes,
                           const float4* __restrict__ tri, float4* __restrict__ glo, float4* __restrict__ ghi) {
    uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n_geom) return;
    int r = root[g];
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0);
    if (r == kEmptyRef) {
    } else if (r < 0) {
        float l[3], h[3];
        tri_slot_box(tri, (size_t)(~r), l, h);
        lo = make_float4(l[0], l[1], l[2], 0);
        hi = make_float4(h[0], h[1], h[2], 0);
    } else {
        Node n = nodes[r];
        lo = make_float4(fminf(n.a.x, n.b.x), fminf(n.a.z, n.b.z), fminf(n.c.x, n.c.z), 0);
        hi = make_float4(fmaxf(n.a.y, n.b.y), fmaxf(n.a.w, n.b.w), fmaxf(n.c.y, n.c.w), 0);
    }
    glo[g] = lo;
    ghi[g] = hi;
}

// What an instance record is made from.  root: BVH4 root ref of each geometry
// (node index, ~triangle slot for a BLAS of one triangle, kEmptyRef); blas4:
// the BVH4 nodes it indexes; glo / ghi: its BLAS box; mesh: (voff, toff) of
// the arrays each geometry's shading reads; toff: each geometry's own triangle
// offset.
struct InstArgs {
    const kf_instance* src;
    uint32_t n_geom;
    const uint32_t* gflags;
    const int* root;
    const Node4* blas4;
    uint32_t n_blas4;
    const float4 *glo, *ghi;
    const uint2* mesh;
    const uint32_t* toff;
    Inst* out;
    float4 *ilo, *ihi;
};

// Record and padded world AABB (corners transformed in double) of instance i.
KF_DEV_INLINE Box make_instance(const InstArgs& A, uint32_t i) {
    const kf_instance in = A.src[i];
    const uint32_t g = in.geometry_index, n_geom = A.n_geom;
    Inst rec;
    float w2o[12];
    world_to_object(in.transform, w2o);
    for (int r = 0; r < 3; ++r) rec.w2o[r] = make_float4(w2o[4 * r], w2o[4 * r + 1], w2o[4 * r + 2], w2o[4 * r + 3]);
    const int r4 = g < n_geom ? A.root[g] : kEmptyRef;
    bool valid = g < n_geom && !(A.gflags[g] & KF_GEOM_HIDDEN) && r4 != kEmptyRef && (r4 < 0 || (uint32_t)r4 < A.n_blas4);
    int flags = (valid ? kInstValid : 0) | ((g < n_geom && (A.gflags[g] & KF_GEOM_OPAQUE)) ? kInstOpaque : 0);
    rec.info = make_int4(valid ? r4 : kEmptyRef, (int)g, flags, 0);
    rec.shade = g < n_geom ? make_int4((int)A.mesh[g].x, (int)A.mesh[g].y, (int)A.toff[g], 0) : make_int4(0, 0, 0, 0);
    // the BLAS root node, as the traversal's instance step tests it
    const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    rec.lox = rec.hix = rec.loy = rec.hiy = rec.loz = rec.hiz = z;
    rec.ref = make_int4((int)kEmptyItem, (int)kEmptyItem, (int)kEmptyItem, (int)kEmptyItem);
    if (valid && r4 >= 0) {
        const Node4 nd = A.blas4[r4];
        rec.lox = nd.lox; rec.hix = nd.hix; rec.loy = nd.loy; rec.hiy = nd.hiy; rec.loz = nd.loz; rec.hiz = nd.hiz;
        rec.ref = nd.ref;
    } else if (valid) {  // one triangle: its box (the geometry's) as the only child
        const float4 a = A.glo[g], b = A.ghi[g];
        rec.lox.x = a.x; rec.hix.x = b.x; rec.loy.x = a.y; rec.hiy.x = b.y; rec.loz.x = a.z; rec.hiz.x = b.z;
        rec.ref.x = (int)((3u << 30) | (uint32_t)~r4);  // triangle item
    }
    A.out[i] = rec;
    Box box = box_empty();
    if (valid) {
        const float4 a = A.glo[g], b = A.ghi[g];
        double l[3] = {INFINITY, INFINITY, INFINITY}, h[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (int c = 0; c < 8; ++c) {
            double p[3] = {(c & 1) ? b.x : a.x, (c & 2) ? b.y : a.y, (c & 4) ? b.z : a.z};
            for (int r = 0; r < 3; ++r) {
                const float* t = in.transform;
                double v = (double)t[r] * p[0] + (double)t[4 + r] * p[1] + (double)t[8 + r] * p[2] + (double)t[12 + r];
                l[r] = fmin(l[r], v);
                h[r] = fmax(h[r], v);
            }
        }
        double ext = fmax(h[0] - l[0], fmax(h[1] - l[1], h[2] - l[2]));
        float fl[3], fh[3];
        for (int r = 0; r < 3; ++r) {
            double pad = 1e-5 * (ext + fabs(l[r]) + fabs(h[r])) + 1e-6;
            fl[r] = nextafterf((float)(l[r] - pad), -INFINITY);
            fh[r] = nextafterf((float)(h[r] + pad), INFINITY);
        }
        box.lo = make_float4(fl[0], fl[1], fl[2], 0);
        box.hi = make_float4(fh[0], fh[1], fh[2], 0);
    }
    A.ilo[i] = box.lo;
    A.ihi[i] = box.hi;
    return box;
}

__global__ void k_instances(uint32_t n, InstArgs A, const uint32_t* __restrict__ inst_env, uint32_t* __restrict__ iseg) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    make_instance(A, i);
    iseg[i] = inst_env ? inst_env[i] : 0u;  // the LBVH segment is the environment
}

// ---------------------------------------------------------------- BVH4
KF_DEV_INLINE float half_area(const float lo[3], const float hi[3]) {
    float dx = hi[0] - lo[0], dy = hi[1] - lo[1], dz = hi[2] - lo[2];
    return dx * dy + dy * dz + dz * dx;
}

// One item of the collapse: (BVH2 node b, BVH4 slot w) writes BVH4 node w
// and queues its inner children for the next level.  b2 holds the n_b2 nodes
// from node b2_base on.  err is set on any index
// outside the arrays (malformed input), and nothing is written out of bounds.
KF_DEV_INLINE void collapse_item(const Node* __restrict__ b2, uint32_t b2_base, uint32_t n_b2, int2 it, int2* __restrict__ out,
                                 uint32_t* out_count, uint32_t out_cap, Node4* __restrict__ wide,
                                 uint32_t* wide_count, uint32_t wide_cap, uint32_t inner_kind, int* err) {
    if ((uint32_t)it.x - b2_base >= n_b2 || (uint32_t)it.y >= wide_cap) {
        *err = 1;
        return;
    }
    float lo[4][3], hi[4][3];
    int ref[4];
    auto take = [&](int node, int s0, int s1) {
        const Node n = b2[(uint32_t)node - b2_base];
        lo[s0][0] = n.a.x; hi[s0][0] = n.a.y; lo[s0][1] = n.a.z; hi[s0][1] = n.a.w; lo[s0][2] = n.c.x; hi[s0][2] = n.c.y;
        lo[s1][0] = n.b.x; hi[s1][0] = n.b.y; lo[s1][1] = n.b.z; hi[s1][1] = n.b.w; lo[s1][2] = n.c.z; hi[s1][2] = n.c.w;
        ref[s0] = n.d.x;
        ref[s1] = n.d.y;
    };
    take(it.x, 0, 1);
    int cnt = 2;
    while (cnt < 4) {
        int best = -1;
        float ba = -1.0f;
        for (int j = 0; j < cnt; ++j)
            if (ref[j] >= 0) {
                const float a = half_area(lo[j], hi[j]);
                if (a > ba) {
                    ba = a;
                    best = j;
                }
            }
        if (best < 0) break;
        if ((uint32_t)ref[best] - b2_base >= n_b2) {
            *err = 1;
            return;
        }
        take(ref[best], best, cnt);
        ++cnt;
    }
    int k = 0;
    for (int j = 0; j < cnt; ++j) k += ref[j] >= 0 ? 1 : 0;
    const uint32_t base = k ? atomicAdd(wide_count, (uint32_t)k) : 0u;
    if (base + (uint32_t)k > wide_cap) {
        *err = 1;
        return;
    }
    float blo[3][4], bhi[3][4];
    int wref[4];
    int m = 0;
    for (int j = 0; j < 4; ++j) {
        const bool used = j < cnt;
        for (int a = 0; a < 3; ++a) {
            blo[a][j] = used ? lo[j][a] : 0.0f;
            bhi[a][j] = used ? hi[j][a] : 0.0f;
        }
        // child refs are stored as traversal items: kind (inner_kind for an
        // inner node, inner_kind + 2 for a leaf) in bits 31:30, index below
        if (!used) {
            wref[j] = (int)kEmptyItem;
        } else if (ref[j] >= 0) {
            wref[j] = (int)((inner_kind << 30) | (base + m));
            const uint32_t q = atomicAdd(out_count, 1u);
            if (q < out_cap) out[q] = make_int2(ref[j], (int)(base + m));
            else *err = 1;
            ++m;
        } else {
            wref[j] = (int)(((inner_kind + 2u) << 30) | (uint32_t)~ref[j]);
        }
    }
    Node4 W;
    W.lox = make_float4(blo[0][0], blo[0][1], blo[0][2], blo[0][3]);
    W.hix = make_float4(bhi[0][0], bhi[0][1], bhi[0][2], bhi[0][3]);
    W.loy = make_float4(blo[1][0], blo[1][1], blo[1][2], blo[1][3]);
    W.hiy = make_float4(bhi[1][0], bhi[1][1], bhi[1][2], bhi[1][3]);
    W.loz = make_float4(blo[2][0], blo[2][1], blo[2][2], blo[2][3]);
    W.hiz = make_float4(bhi[2][0], bhi[2][1], bhi[2][2], bhi[2][3]);
    W.ref = make_int4(wref[0], wref[1], wref[2], wref[3]);
    // the BVH2 ref each child was taken from (a refit recomputes the child
    // boxes from these); the traversal never reads this line
    W.pad = make_int4(0 < cnt ? ref[0] : kEmptyRef, 1 < cnt ? ref[1] : kEmptyRef, 2 < cnt ? ref[2] : kEmptyRef,
                      3 < cnt ? ref[3] : kEmptyRef);
    wide[it.y] = W;
}

// A block collapses one tree of n_e >= 2 leaves, level after level: BVH2
// nodes [base, base + n_e - 1) (at b2), root first, into BVH4 slots [base,
// base + n_e - 1) of `wide` (a BVH4 never has more nodes than its BVH2), root
// first; qa / qb hold its level queues.  cnt[0]: next free BVH4 slot, cnt[1]:
// next-level queue length.
KF_DEV_INLINE void collapse_tree(const Node* b2, uint32_t base, uint32_t n_e, int2* qa, int2* qb,
                                 Node4* __restrict__ wide, uint32_t inner_kind, uint32_t* cnt, uint32_t* n_in, int* err) {
    const uint32_t cap_e = n_e - 1u;
    if (threadIdx.x == 0) {
        *n_in = 1u;
        cnt[0] = base + 1u;
        cnt[1] = 0u;
        qa[0] = make_int2((int)base, (int)base);
    }
    __syncthreads();
    for (uint32_t level = 0; *n_in > 0u; ++level) {
        if (level > cap_e + 1u) {  // deeper than a well-formed tree can be
            if (threadIdx.x == 0) *err = 1;
            break;
        }
        for (uint32_t i = threadIdx.x; i < *n_in; i += blockDim.x)
            collapse_item(b2, base, cap_e, qa[i], qb, &cnt[1], cap_e, wide, &cnt[0], base + cap_e, inner_kind, err);
        __syncthreads();
        if (threadIdx.x == 0) {
            *n_in = min(cnt[1], cap_e);
            cnt[1] = 0u;
        }
        __syncthreads();
        int2* t = qa;
        qa = qb;
        qb = t;
    }
}

// The whole collapse of a forest with no host round trip: block e collapses
// tree e, the n_e = seg_off[e+1] - seg_off[e] leaves of its LBVH segment, whose
// nodes start at node_off[e].  cnt_all + 2e: collapse_tree's counters.
constexpr int kTreeThreads = 1024;
__global__ __launch_bounds__(kTreeThreads) void k_collapse_forest(const Node* __restrict__ b2, uint32_t n_b2,
                                                                  const uint32_t* __restrict__ seg_off,
                                                                  const uint32_t* __restrict__ node_off, int2* qa_all,
                                                                  int2* qb_all, Node4* __restrict__ wide,
                                                                  uint32_t inner_kind, uint32_t* cnt_all, int* err) {
    __shared__ uint32_t n_in;
    const uint32_t e = blockIdx.x;
    const uint32_t n_e = seg_off[e + 1] - seg_off[e];
    if (n_e < 2u) return;  // a single instance or none: the root is a leaf or empty
    const uint32_t base = node_off[e];
    if (base + n_e - 1u > n_b2) {
        if (threadIdx.x == 0) *err = 1;
        return;
    }
    collapse_tree(b2 + base, base, n_e, qa_all + base, qb_all + base, wide, inner_kind, cnt_all + 2 * e, &n_in, err);
}

// ---------------------------------------------------------------- small TLAS
// The TLAS of environment blockIdx.x in one block, for at most M instances:
// instance records and boxes, centroid bounds, Morton codes, a bitonic sort on
// (code, instance), the box pyramid, the Karras nodes and the BVH4 collapse,
// all in LDS but for the results; the same trees as the general path, whose
// 27 launches and 30 allocations took 281 us per update of 65 instances.  Now
// 41 us, 32 of them this kernel: a chain of short steps (the double-precision
// record, 28 compare-exchange rounds, four collapse levels) on one CU.
// env_off, node_off: null for one environment of n instances.
template <int M>
__global__ __launch_bounds__(M) void k_tlas_small(uint32_t n, InstArgs A, const uint32_t* __restrict__ env_off,
                                                  const uint32_t* __restrict__ node_off, Node* __restrict__ nodes,
                                                  Node4* __restrict__ wide, uint32_t* __restrict__ cnt_all, int* err) {
    struct Box6 {
        float v[6];  // lo, hi
    };
    __shared__ unsigned long long key[M];
    __shared__ Box6 pyr[2 * M];  // level k from entry 2M - (2M >> k)
    __shared__ Node tree[M];
    __shared__ int2 qa[M], qb[M];
    __shared__ float bounds[6][M / 64];
    __shared__ uint32_t cnt[2], n_in;
    const uint32_t e = blockIdx.x, t = threadIdx.x;
    const uint32_t so = env_off ? env_off[e] : 0u, n_e = (env_off ? env_off[e + 1] : n) - so;
    const uint32_t nb = node_off ? node_off[e] : 0u;
    if (n_e > (uint32_t)M) {  // the host sizes M for the largest environment
        if (t == 0) *err = 1;
        return;
    }
    const bool on = t < n_e;
    Box box = box_empty();
    if (on) box = make_instance(A, so + t);
    if (n_e < 2u) return;  // uniform: a single instance or none has no node
    // centroid bounds of the non-empty boxes
    const bool full = on && box.lo.x <= box.hi.x;
    const float c[3] = {0.5f * (box.lo.x + box.hi.x), 0.5f * (box.lo.y + box.hi.y), 0.5f * (box.lo.z + box.hi.z)};
    float bl[3], bh[3];
    for (int k = 0; k < 3; ++k) {
        float l = full ? c[k] : INFINITY, h = full ? c[k] : -INFINITY;
        for (int off = 32; off > 0; off >>= 1) {
            l = fminf(l, __shfl_xor(l, off));
            h = fmaxf(h, __shfl_xor(h, off));
        }
        if ((t & 63u) == 0u) {
            bounds[k][t >> 6] = l;
            bounds[3 + k][t >> 6] = h;
        }
    }
    __syncthreads();
    for (int k = 0; k < 3; ++k) {
        bl[k] = INFINITY;
        bh[k] = -INFINITY;
        for (int w = 0; w < M / 64; ++w) {
            bl[k] = fminf(bl[k], bounds[k][w]);
            bh[k] = fmaxf(bh[k], bounds[3 + k][w]);
        }
    }
    key[t] = on ? ((unsigned long long)morton30(full, c, bl, bh) << 32) | t : ~0ull;
    // boxes by instance, where the pyramid's upper levels go later
    for (int k = 0; k < 3; ++k) {
        pyr[M + t].v[k] = k == 0 ? box.lo.x : k == 1 ? box.lo.y : box.lo.z;
        pyr[M + t].v[3 + k] = k == 0 ? box.hi.x : k == 1 ? box.hi.y : box.hi.z;
    }
    for (uint32_t size = 2; size < 2u * n_e; size <<= 1)
        for (uint32_t j = size >> 1; j > 0; j >>= 1) {
            __syncthreads();
            const uint32_t q = t ^ j;
            if (q > t) {
                const unsigned long long a = key[t], b = key[q];
                if ((a > b) == ((t & size) == 0u)) {
                    key[t] = b;
                    key[q] = a;
                }
            }
        }
    __syncthreads();
    Box6 mine = pyr[M + (on ? (uint32_t)key[t] : 0u)];
    if (!on)
        for (int k = 0; k < 6; ++k) mine.v[k] = k < 3 ? INFINITY : -INFINITY;
    pyr[t] = mine;
    __syncthreads();
    for (uint32_t k = 1, w = M / 2; w > 0; ++k, w >>= 1) {
        const uint32_t from = 2u * M - (2u * M >> (k - 1)), to = 2u * M - (2u * M >> k);
        if (t < w)
            for (int j = 0; j < 6; ++j) {
                const float x = pyr[from + 2 * t].v[j], y = pyr[from + 2 * t + 1].v[j];
                pyr[to + t].v[j] = j < 3 ? fminf(x, y) : fmaxf(x, y);
            }
        __syncthreads();
    }
    auto range = [&](uint32_t l, uint32_t r, Box6& b) {
        b = pyr[l];
        if (l == r) return;
        for (int j = 0; j < 6; ++j) b.v[j] = j < 3 ? INFINITY : -INFINITY;
        auto add = [&](uint32_t i) {
            for (int j = 0; j < 6; ++j) b.v[j] = j < 3 ? fminf(b.v[j], pyr[i].v[j]) : fmaxf(b.v[j], pyr[i].v[j]);
        };
        for (uint32_t at = 0, w = M; l <= r; at += w, w >>= 1) {
            if (l & 1u) add(at + l++);
            if (!(r & 1u)) {
                add(at + r);
                if (r == 0u) break;
                --r;
            }
            l >>= 1;
            r >>= 1;
        }
    };
    if (t + 1u < n_e) {
        const KarrasNode kn = karras_node([&](int a) { return key[a] >> 32; }, (int)n_e, (int)t);
        auto leaf = [&](int q) { return ~(int)(so + (uint32_t)key[q]); };
        const int lref = kn.first == kn.split ? leaf(kn.split) : (int)nb + kn.split;
        const int rref = kn.last == kn.split + 1 ? leaf(kn.split + 1) : (int)nb + kn.split + 1;
        Box6 L, R;
        range((uint32_t)kn.first, (uint32_t)kn.split, L);
        range((uint32_t)kn.split + 1u, (uint32_t)kn.last, R);
        Node m;
        m.a = make_float4(L.v[0], L.v[3], L.v[1], L.v[4]);
        m.b = make_float4(R.v[0], R.v[3], R.v[1], R.v[4]);
        m.c = make_float4(L.v[2], L.v[5], R.v[2], R.v[5]);
        m.d = make_int4(lref, rref, (int)so + kn.first, (int)so + kn.last);
        tree[t] = m;
        nodes[nb + t] = m;
    }
    collapse_tree(tree, nb, n_e, qa, qb, wide, 0u, cnt, &n_in, err);
    if (t == 0) {
        cnt_all[2 * e] = cnt[0];
        cnt_all[2 * e + 1] = 0u;
    }
}

}  // namespace

void lbvh_build(uint32_t n, const float4* d_lo, const float4* d_hi, const uint32_t* d_seg, uint32_t n_seg,
                const uint32_t* d_seg_off, const uint32_t* d_node_off, Node* d_nodes, uint32_t* d_order, int* d_root,
                bool leaf_is_slot, hipStream_t st) {
    const uint32_t TB = 256;
    if (n == 0) {
        k_seg_root<<<blocks(n_seg, TB), TB, 0, st>>>(n_seg, d_seg_off, d_node_off, d_order, d_root, leaf_is_slot);
        return;
    }
    int* sb = dalloc<int>(6 * (size_t)n_seg);
    unsigned long long* k0 = dalloc<unsigned long long>(n);
    unsigned long long* k1 = dalloc<unsigned long long>(n);
    uint32_t* v0 = dalloc<uint32_t>(n);
    uint32_t* v1 = dalloc<uint32_t>(n);
    uint32_t n_tiles = blocks(n, kSortTile);
    uint32_t* hist = dalloc<uint32_t>((size_t)n_tiles * kDigits + kDigits);
    uint32_t* total = hist + (size_t)n_tiles * kDigits;

    k_seg_init<<<blocks(6 * n_seg, TB), TB, 0, st>>>(n_seg, sb);
    k_seg_bounds<<<blocks(n, TB), TB, 0, st>>>(n, d_lo, d_hi, d_seg, sb);
    k_morton<<<blocks(n, TB), TB, 0, st>>>(n, d_lo, d_hi, d_seg, sb, k0, v0);

    int seg_bits = 0;
    while ((1u << seg_bits) < n_seg) ++seg_bits;
    int total_bits = 30 + seg_bits;
    for (int shift = 0; shift < total_bits; shift += kDigitBits) {
        const bool last = shift + kDigitBits >= total_bits;  // the order goes where the caller wants it
        uint32_t* vo = last ? d_order : v1;
        k_rs_hist<<<n_tiles, kSortThreads, 0, st>>>(n, k0, shift, n_tiles, hist);
        k_rs_scan<<<kDigits, kSortThreads, 0, st>>>(n_tiles, hist, total);
        k_rs_scatter<<<n_tiles, kSortThreads, 0, st>>>(n, k0, v0, shift, n_tiles, hist, total, k1, vo);
        std::swap(k0, k1);
        if (!last) std::swap(v0, v1);
    }
    Box* pyr = dalloc<Box>(pyramid_size(n));
    const Pyramid P = build_pyramid(n, d_order, d_lo, d_hi, pyr, st);
    k_karras<<<blocks(n, TB), TB, 0, st>>>(n, k0, d_order, d_seg_off, d_node_off, P, d_nodes, leaf_is_slot);
    k_seg_root<<<blocks(n_seg, TB), TB, 0, st>>>(n_seg, d_seg_off, d_node_off, d_order, d_root, leaf_is_slot);
    KF_CHECK(hipGetLastError());
    dfree(sb); dfree(k0); dfree(k1); dfree(v0); dfree(v1);
    dfree(hist); dfree(pyr);
}

// The geometry of every triangle.
void map_triangles(Scene& s) {
    s.d_tri_geom = dalloc<uint32_t>(std::max<uint32_t>(s.n_tri, 1));
    if (s.n_tri)
        k_tri_geom<<<blocks(s.n_tri, 256), 256, 0, stream()>>>(s.n_tri, s.n_geom, s.d_toff, s.d_tri_geom);
    KF_CHECK(hipGetLastError());
}

// d_glo / d_ghi, after a build or refit.
void blas_boxes(Scene& s) {
    if (s.n_geom)
        k_blas_box<<<blocks(s.n_geom, 256), 256, 0, stream()>>>(s.n_geom, s.d_blas_root, s.d_blas, s.d_tri, s.d_glo,
                                                                s.d_ghi);
}

void build_blas(Scene& s) {
    hipStream_t st = stream();
    const uint32_t TB = 256;
    uint32_t n = s.n_tri;
    s.h_node_off.assign(s.n_geom, 0);
    uint32_t acc = 0;
    for (uint32_t g = 0; g < s.n_geom; ++g) {
        s.h_node_off[g] = acc;
        uint32_t ng = s.h_toff[g + 1] - s.h_toff[g];
        acc += ng > 1 ? ng - 1 : 0;
    }
    s.n_blas_nodes = acc;
    dfree(s.d_blas);
    dfree(s.d_tri);
    dfree(s.d_blas_root);
    s.d_blas = dalloc<Node>(std::max<uint32_t>(acc, 1));
    s.d_tri = dalloc<float4>(3 * (size_t)std::max<uint32_t>(n, 1));
    s.d_blas_root = dalloc<int>(std::max<uint32_t>(s.n_geom, 1));
    uint32_t* d_node_off = dalloc<uint32_t>(std::max<uint32_t>(s.n_geom, 1));
    if (s.n_geom)
        KF_CHECK(hipMemcpyAsync(d_node_off, s.h_node_off.data(), s.n_geom * sizeof(uint32_t), hipMemcpyHostToDevice, st));
    float4* lo = dalloc<float4>(std::max<uint32_t>(n, 1));
    float4* hi = dalloc<float4>(std::max<uint32_t>(n, 1));
    uint32_t* order = dalloc<uint32_t>(std::max<uint32_t>(n, 1));
    if (n) {
        k_tri_bounds<<<blocks(n, TB), TB, 0, st>>>(n, s.d_verts, s.d_idx, s.d_voff, s.d_tri_geom, lo, hi);
    }
    lbvh_build(n, lo, hi, s.d_tri_geom, s.n_geom, s.d_toff, d_node_off, s.d_blas, order, s.d_blas_root, true, st);
    if (n)
        k_tri_reorder<<<blocks(n, TB), TB, 0, st>>>(n, order, s.d_verts, s.d_idx, s.d_voff, s.d_toff, s.d_tri_geom,
                                                    s.d_tri);
    KF_CHECK(hipGetLastError());
    s.h_blas_root.resize(s.n_geom);
    if (s.n_geom)
        KF_CHECK(hipMemcpyAsync(s.h_blas_root.data(), s.d_blas_root, s.n_geom * sizeof(int), hipMemcpyDeviceToHost, st));
    dfree(d_node_off); dfree(lo); dfree(hi); dfree(order);
    KF_CHECK(hipStreamSynchronize(st));
    // BVH4 for the traversal: geometry g's nodes in [node_off[g], node_off[g]
    // + n_g - 1), root first, so roots are known by construction and a refit
    // of one geometry touches only its own range
    dfree(s.d_blas4);
    dfree(s.d_blas_root4);
    dfree(s.d_node_off);
    dfree(s.d_blas_cnt);
    const uint32_t cap4 = std::max<uint32_t>(acc, 1);
    s.d_blas4 = dalloc<Node4>(cap4);
    s.d_node_off = dalloc<uint32_t>(std::max<uint32_t>(s.n_geom, 1));
    s.d_blas_cnt = dalloc<uint32_t>(2 * (size_t)std::max<uint32_t>(s.n_geom, 1));
    if (s.n_geom)
        KF_CHECK(hipMemcpyAsync(s.d_node_off, s.h_node_off.data(), s.n_geom * sizeof(uint32_t), hipMemcpyHostToDevice,
                                st));
    int* err = dalloc<int>(1);
    KF_CHECK(hipMemsetAsync(err, 0, sizeof(int), st));
    if (acc) {
        int2* qa = dalloc<int2>(acc);
        int2* qb = dalloc<int2>(acc);
        k_collapse_forest<<<s.n_geom, kTreeThreads, 0, st>>>(s.d_blas, acc, s.d_toff, s.d_node_off, qa, qb, s.d_blas4,
                                                               1u, s.d_blas_cnt, err);
        KF_CHECK(hipGetLastError());
        dfree(qa);
        dfree(qb);
    }
    s.h_blas_root4.assign(s.n_geom, kEmptyRef);
    for (uint32_t g = 0; g < s.n_geom; ++g) {
        const uint32_t ng = s.h_toff[g + 1] - s.h_toff[g];
        s.h_blas_root4[g] = ng >= 2 ? (int)s.h_node_off[g] : (ng == 1 ? ~(int)s.h_toff[g] : kEmptyRef);
    }
    s.n_blas4 = cap4;  // index bound; used nodes per geometry are counted in d_blas_cnt
    s.d_blas_root4 = dalloc<int>(std::max<uint32_t>(s.n_geom, 1));
    if (s.n_geom)
        KF_CHECK(hipMemcpyAsync(s.d_blas_root4, s.h_blas_root4.data(), s.n_geom * sizeof(int), hipMemcpyHostToDevice, st));
    int h_err = 0;
    KF_CHECK(hipMemcpyAsync(&h_err, err, sizeof(int), hipMemcpyDeviceToHost, st));
    KF_CHECK(hipStreamSynchronize(st));
    dfree(err);
    if (h_err) throw Error("BLAS build: malformed BVH2");
    s.d_glo = dalloc<float4>(std::max<uint32_t>(s.n_geom, 1));
    s.d_ghi = dalloc<float4>(std::max<uint32_t>(s.n_geom, 1));
    blas_boxes(s);
    upload_trav_roots(s);
    upload_mesh_sources(s);
}

// d_trav_root4[g] = the BVH4 root of the geometry whose BVH g traverses.
void upload_trav_roots(Scene& s) {
    if (s.h_canon.size() != s.n_geom) {
        s.h_canon.resize(s.n_geom);
        for (uint32_t g = 0; g < s.n_geom; ++g) s.h_canon[g] = g;
    }
    std::vector<int> roots(std::max<uint32_t>(s.n_geom, 1), kEmptyRef);
    for (uint32_t g = 0; g < s.n_geom; ++g) roots[g] = s.h_blas_root4[s.h_canon[g]];
    if (!s.d_trav_root4) s.d_trav_root4 = dalloc<int>(std::max<uint32_t>(s.n_geom, 1));
    KF_CHECK(hipMemcpy(s.d_trav_root4, roots.data(), roots.size() * sizeof(int), hipMemcpyHostToDevice));
}

// d_mesh[g] = (voff, toff) of the geometry whose arrays g's shading reads.
void upload_mesh_sources(Scene& s) {
    if (s.h_mesh.size() != s.n_geom) {
        s.h_mesh.resize(s.n_geom);
        for (uint32_t g = 0; g < s.n_geom; ++g) s.h_mesh[g] = g;
    }
    std::vector<uint2> src(std::max<uint32_t>(s.n_geom, 1), make_uint2(0u, 0u));
    for (uint32_t g = 0; g < s.n_geom; ++g) src[g] = make_uint2(s.h_voff[s.h_mesh[g]], s.h_toff[s.h_mesh[g]]);
    if (!s.d_mesh) s.d_mesh = dalloc<uint2>(std::max<uint32_t>(s.n_geom, 1));
    KF_CHECK(hipMemcpy(s.d_mesh, src.data(), src.size() * sizeof(uint2), hipMemcpyHostToDevice));
}

namespace {
// ---------------------------------------------------------------- scene data
// Words of a geometry, each mixed with its place and added up: equal data
// have equal sums, and equal sums are compared word for word below.  (The
// same filter as a byte-wise FNV on one host thread took 70 of the 97 ms that
// loading 256 meshes of 5120 triangles took; the kernels read the uploaded
// arrays in 86 us.)
KF_DEV_INLINE unsigned long long mix_word(uint32_t w, uint32_t place) {
    unsigned long long z = (((unsigned long long)place << 32) | w) + 0x9e3779b97f4a7c15ull;  // splitmix64
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}
// Adds v to sum[g]: once per wave where all its lanes hold the same g.
// Lanes with g = ~0 take no part.
KF_DEV_INLINE void geom_add(unsigned long long* sum, uint32_t g, unsigned long long v) {
    const unsigned long long m = __ballot(g != ~0u);
    if (!m) return;
    const uint32_t g0 = (uint32_t)__builtin_amdgcn_readlane((int)g, __ffsll((long long)m) - 1);
    if (__ballot(g != ~0u && g != g0) == 0ull) {
        if (g == ~0u) v = 0ull;
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
        if ((threadIdx.x & 63u) == 0u) atomicAdd(&sum[g0], v);
    } else if (g != ~0u) {
        atomicAdd(&sum[g], v);
    }
}
KF_DEV_INLINE uint32_t geom_of(const uint32_t* __restrict__ off, uint32_t n_geom, uint32_t i) {
    uint32_t lo = 0, hi = n_geom;  // largest g with off[g] <= i
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (off[mid] <= i) lo = mid; else hi = mid;
    }
    return lo;
}
KF_DEV_INLINE uint3 corner_words(const float4* __restrict__ verts, uint32_t v) {
    const float4 p = verts[3 * (size_t)v];
    return make_uint3(__float_as_uint(p.x), __float_as_uint(p.y), __float_as_uint(p.z));
}

// sum[g]: the corner positions of g's triangles in order; sum[n_geom + g]:
// its indices (here) and vertex records (k_hash_vertices).
__global__ void k_hash_triangles(uint32_t n_tri, uint32_t n_geom, const float4* __restrict__ verts,
                                 const uint32_t* __restrict__ idx, const uint32_t* __restrict__ voff,
                                 const uint32_t* __restrict__ toff, const uint32_t* __restrict__ tri_geom,
                                 unsigned long long* __restrict__ sum) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t g = i < n_tri ? tri_geom[i] : ~0u;
    unsigned long long a = 0, b = 0;
    if (i < n_tri) {
        const uint32_t t = i - toff[g];
        for (uint32_t k = 0; k < 3; ++k) {
            const uint32_t v = idx[3 * (size_t)i + k];
            const uint3 p = corner_words(verts, voff[g] + v);
            a += mix_word(p.x, 9u * t + 3u * k) + mix_word(p.y, 9u * t + 3u * k + 1u) + mix_word(p.z, 9u * t + 3u * k + 2u);
            b += mix_word(v, 3u * t + k);
        }
    }
    geom_add(sum, g, a);
    geom_add(sum + n_geom, g, b);
}
__global__ void k_hash_vertices(uint32_t n_vert, uint32_t n_geom, const uint4* __restrict__ verts,
                                const uint32_t* __restrict__ voff, unsigned long long* __restrict__ sum) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t g = i < n_vert ? geom_of(voff, n_geom, i) : ~0u;
    unsigned long long b = 0;
    if (i < n_vert) {
        const uint32_t j = i - voff[g];
        for (uint32_t k = 0; k < 3; ++k) {
            const uint4 w = verts[3 * (size_t)i + k];
            const uint32_t at = 0x80000000u + 12u * j + 4u * k;  // apart from the indices' places
            b += mix_word(w.x, at) + mix_word(w.y, at + 1u) + mix_word(w.z, at + 2u) + mix_word(w.w, at + 3u);
        }
    }
    geom_add(sum + n_geom, g, b);
}

// differs[g] / differs[n_geom + g]: g's corners / its indices and vertex
// records are not those of cand[g] / cand[n_geom + g] (of the same counts).
__global__ void k_equal_triangles(uint32_t n_tri, uint32_t n_geom, const float4* __restrict__ verts,
                                  const uint32_t* __restrict__ idx, const uint32_t* __restrict__ voff,
                                  const uint32_t* __restrict__ toff, const uint32_t* __restrict__ tri_geom,
                                  const uint32_t* __restrict__ cand, uint32_t* __restrict__ differs) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_tri) return;
    const uint32_t g = tri_geom[i], t = i - toff[g], ca = cand[g], cb = cand[n_geom + g];
    for (uint32_t k = 0; k < 3; ++k) {
        const uint32_t v = idx[3 * (size_t)i + k];
        if (ca != g) {
            const uint3 p = corner_words(verts, voff[g] + v);
            const uint3 q = corner_words(verts, voff[ca] + idx[3 * (size_t)(toff[ca] + t) + k]);
            if (p.x != q.x || p.y != q.y || p.z != q.z) differs[g] = 1u;
        }
        if (cb != g && idx[3 * (size_t)(toff[cb] + t) + k] != v) differs[n_geom + g] = 1u;
    }
}
__global__ void k_equal_vertices(uint32_t n_vert, uint32_t n_geom, const uint4* __restrict__ verts,
                                 const uint32_t* __restrict__ voff, const uint32_t* __restrict__ cand,
                                 uint32_t* __restrict__ differs) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_vert) return;
    const uint32_t g = geom_of(voff, n_geom, i), c = cand[n_geom + g];
    if (c == g) return;
    const size_t p = 3 * (size_t)i, q = 3 * (size_t)(voff[c] + (i - voff[g]));
    for (uint32_t k = 0; k < 3; ++k) {
        const uint4 a = verts[p + k], b = verts[q + k];
        if (a.x != b.x || a.y != b.y || a.z != b.z || a.w != b.w) differs[n_geom + g] = 1u;
    }
}

// g leaves its group: the next member leads the rest.  False when it was
// alone already.
bool leave_group(std::vector<uint32_t>& lead, uint32_t g) {
    bool moved = lead[g] != g;
    if (lead[g] == g) {
        uint32_t m = UINT32_MAX;
        for (uint32_t d = 0; d < lead.size(); ++d)
            if (d != g && lead[d] == g) {
                if (m == UINT32_MAX) m = d;
                lead[d] = m;
            }
        moved = m != UINT32_MAX;
    }
    lead[g] = g;
    return moved;
}
}  // namespace

void share_geometry(Scene& s, const kf_vertex* verts, const uint32_t* idx, bool separate) {
    hipStream_t st = stream();
    const uint32_t n = s.n_geom, TB = 256;
    s.h_canon.resize(n);
    s.h_mesh.resize(n);
    for (uint32_t g = 0; g < n; ++g) s.h_canon[g] = s.h_mesh[g] = g;
    if (separate || n < 2) return;
    auto ntri = [&](uint32_t g) { return (size_t)(s.h_toff[g + 1] - s.h_toff[g]); };
    auto nvert = [&](uint32_t g) { return (size_t)(s.h_voff[g + 1] - s.h_voff[g]); };
    auto corner = [&](uint32_t g, size_t t, int k) -> const float* {
        return verts[s.h_voff[g] + idx[3 * (s.h_toff[g] + t) + k]].pos;
    };
    // the exact comparisons, for geometries whose sums collide
    auto same_corners = [&](uint32_t c, uint32_t g) {
        if (ntri(c) != ntri(g)) return false;
        for (size_t t = 0; t < ntri(g); ++t)
            for (int k = 0; k < 3; ++k)
                if (std::memcmp(corner(c, t, k), corner(g, t, k), 12)) return false;
        return true;
    };
    auto same_mesh = [&](uint32_t c, uint32_t g) {
        return nvert(c) == nvert(g) && ntri(c) == ntri(g) &&
               (!nvert(g) ||
                !std::memcmp(verts + s.h_voff[c], verts + s.h_voff[g], nvert(g) * sizeof(kf_vertex))) &&
               (!ntri(g) || !std::memcmp(idx + 3 * (size_t)s.h_toff[c], idx + 3 * (size_t)s.h_toff[g],
                                         3 * ntri(g) * sizeof(uint32_t)));
    };
    unsigned long long* d_sum = dalloc<unsigned long long>(2 * (size_t)n);
    KF_CHECK(hipMemsetAsync(d_sum, 0, 2 * (size_t)n * sizeof(*d_sum), st));
    if (s.n_tri)
        k_hash_triangles<<<blocks(s.n_tri, TB), TB, 0, st>>>(s.n_tri, n, s.d_verts, s.d_idx, s.d_voff, s.d_toff,
                                                             s.d_tri_geom, d_sum);
    if (s.n_vert)
        k_hash_vertices<<<blocks(s.n_vert, TB), TB, 0, st>>>(s.n_vert, n, (const uint4*)s.d_verts, s.d_voff, d_sum);
    KF_CHECK(hipGetLastError());
    std::vector<unsigned long long> sum(2 * (size_t)n);
    KF_CHECK(hipMemcpyAsync(sum.data(), d_sum, sum.size() * sizeof(sum[0]), hipMemcpyDeviceToHost, st));
    KF_CHECK(hipStreamSynchronize(st));
    dfree(d_sum);
    // the first geometry of the same counts and sum, as a candidate
    std::vector<uint32_t> cand(2 * (size_t)n);
    std::map<std::array<unsigned long long, 2>, std::vector<uint32_t>> by_corners;
    std::map<std::array<unsigned long long, 3>, std::vector<uint32_t>> by_mesh;
    bool any = false;
    for (uint32_t g = 0; g < n; ++g) {
        auto& a = by_corners[{ntri(g), sum[g]}];
        auto& b = by_mesh[{nvert(g), ntri(g), sum[n + g]}];
        a.push_back(g);
        b.push_back(g);
        cand[g] = a[0];
        cand[n + g] = b[0];
        any = any || a[0] != g || b[0] != g;
    }
    if (!any) return;
    uint32_t* d_cand = dalloc<uint32_t>(4 * (size_t)n);  // candidates, then flags
    uint32_t* d_differs = d_cand + 2 * (size_t)n;
    KF_CHECK(hipMemcpyAsync(d_cand, cand.data(), 2 * (size_t)n * sizeof(uint32_t), hipMemcpyHostToDevice, st));
    KF_CHECK(hipMemsetAsync(d_differs, 0, 2 * (size_t)n * sizeof(uint32_t), st));
    if (s.n_tri)
        k_equal_triangles<<<blocks(s.n_tri, TB), TB, 0, st>>>(s.n_tri, n, s.d_verts, s.d_idx, s.d_voff, s.d_toff,
                                                              s.d_tri_geom, d_cand, d_differs);
    if (s.n_vert)
        k_equal_vertices<<<blocks(s.n_vert, TB), TB, 0, st>>>(s.n_vert, n, (const uint4*)s.d_verts, s.d_voff, d_cand,
                                                              d_differs);
    KF_CHECK(hipGetLastError());
    std::vector<uint32_t> differs(2 * (size_t)n);
    KF_CHECK(hipMemcpyAsync(differs.data(), d_differs, differs.size() * sizeof(uint32_t), hipMemcpyDeviceToHost, st));
    KF_CHECK(hipStreamSynchronize(st));
    dfree(d_cand);
    // a group without collisions is led by its first member; with one, each
    // member joins the first earlier one that it equals
    auto lead = [&](const std::vector<uint32_t>& group, std::vector<uint32_t>& out, uint32_t base, auto same) {
        bool collision = false;
        for (uint32_t g : group) collision = collision || differs[base + g];
        for (size_t i = 1; i < group.size(); ++i) {
            const uint32_t g = group[i];
            if (!collision) out[g] = group[0];
            else
                for (size_t j = 0; j < i && out[g] == g; ++j)
                    if (out[group[j]] == group[j] && same(group[j], g)) out[g] = group[j];
        }
    };
    for (const auto& e : by_corners) lead(e.second, s.h_canon, 0, same_corners);
    for (const auto& e : by_mesh) lead(e.second, s.h_mesh, n, same_mesh);
}

void unshare_geometry(Scene& s, uint32_t g) {
    if (g >= s.n_geom) return;
    if (s.h_canon.size() == s.n_geom && leave_group(s.h_canon, g)) upload_trav_roots(s);
    if (s.h_mesh.size() == s.n_geom && leave_group(s.h_mesh, g)) upload_mesh_sources(s);
}

// ---------------------------------------------------------------- refit
// Refit of one geometry after its vertices moved (same triangles): the
// triangle slots take the new positions, the BVH2 boxes follow from each
// node's range of slots over a new pyramid (82 k triangles: 339 us for the
// bottom-up walk, 26 us now), then every BVH4 child box is the box of the
// BVH2 ref it was collapsed from.  The trees keep their shape.
__global__ void k_geom_slots(uint32_t g, const float4* __restrict__ verts, const uint32_t* __restrict__ idx,
                             const uint32_t* __restrict__ voff, const uint32_t* __restrict__ toff, float4* tri,
                             float4* __restrict__ lo, float4* __restrict__ hi) {
    const uint32_t t0 = toff[g], n = toff[g + 1] - t0;
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const size_t slot = t0 + j;
    const uint32_t prim = __float_as_uint(tri[3 * slot].w);
    if (prim >= n) return;  // not a slot of this geometry (malformed)
    const size_t i = t0 + prim;
    float3 p[3];
    for (int k = 0; k < 3; ++k) {
        const float4 v = verts[3 * (size_t)(voff[g] + idx[3 * i + k])];
        p[k] = make_float3(v.x, v.y, v.z);
    }
    put_tri_slot(tri, slot, p, prim);
    lo[j] = make_float4(fminf(p[0].x, fminf(p[1].x, p[2].x)), fminf(p[0].y, fminf(p[1].y, p[2].y)),
                        fminf(p[0].z, fminf(p[1].z, p[2].z)), 0.f);
    hi[j] = make_float4(fmaxf(p[0].x, fmaxf(p[1].x, p[2].x)), fmaxf(p[0].y, fmaxf(p[1].y, p[2].y)),
                        fmaxf(p[0].z, fmaxf(p[1].z, p[2].z)), 0.f);
}

// Child boxes of geometry g's BVH2 nodes over the pyramid P of its slots.
__global__ void k_geom_refit2(uint32_t g, const uint32_t* __restrict__ toff, const uint32_t* __restrict__ node_off,
                              uint32_t n_nodes, Pyramid P, Node* nodes) {
    const uint32_t t0 = toff[g], n = toff[g + 1] - t0, nb = node_off[g];
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (n < 2 || j >= n - 1 || nb + j >= n_nodes) return;
    const int4 d = nodes[nb + j].d;
    // the left child's last slot: its leaf, or (Karras) its node's index
    const uint32_t first = (uint32_t)d.z - t0, last = (uint32_t)d.w - t0;
    const uint32_t split = d.x < 0 ? (uint32_t)~d.x - t0 : (uint32_t)d.x - nb;
    if (!(first <= split && split < last && last < n)) return;  // malformed
    Node m = make_node(P, first, split, last, d.x, d.y);
    m.d = d;
    nodes[nb + j] = m;
}

__global__ void k_geom_refit4(uint32_t g, const uint32_t* __restrict__ toff, const uint32_t* __restrict__ node_off,
                              const uint32_t* __restrict__ cnt4, const Node* __restrict__ nodes, uint32_t n_nodes,
                              const float4* __restrict__ tri, Node4* wide) {
    const uint32_t t0 = toff[g], n = toff[g + 1] - t0, nb = node_off[g];
    if (n < 2) return;
    const uint32_t used = min(cnt4[2 * g] - nb, n - 1);
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= used) return;
    Node4& W = wide[nb + j];
    const int4 pr = W.pad;
    float blo[3][4], bhi[3][4];
    for (int c = 0; c < 4; ++c) {
        const int r = c == 0 ? pr.x : (c == 1 ? pr.y : (c == 2 ? pr.z : pr.w));
        float lo[3] = {0.f, 0.f, 0.f}, hi[3] = {0.f, 0.f, 0.f};
        if (r == kEmptyRef) {
        } else if (r >= 0) {
            if ((uint32_t)r < n_nodes) {
                const Node m = nodes[r];
                lo[0] = fminf(m.a.x, m.b.x); hi[0] = fmaxf(m.a.y, m.b.y);
                lo[1] = fminf(m.a.z, m.b.z); hi[1] = fmaxf(m.a.w, m.b.w);
                lo[2] = fminf(m.c.x, m.c.z); hi[2] = fmaxf(m.c.y, m.c.w);
            }
        } else if ((uint32_t)~r >= t0 && (uint32_t)~r < t0 + n) {
            tri_slot_box(tri, (size_t)~r, lo, hi);
        }
        for (int a = 0; a < 3; ++a) {
            blo[a][c] = lo[a];
            bhi[a][c] = hi[a];
        }
    }
    W.lox = make_float4(blo[0][0], blo[0][1], blo[0][2], blo[0][3]);
    W.hix = make_float4(bhi[0][0], bhi[0][1], bhi[0][2], bhi[0][3]);
    W.loy = make_float4(blo[1][0], blo[1][1], blo[1][2], blo[1][3]);
    W.hiy = make_float4(bhi[1][0], bhi[1][1], bhi[1][2], bhi[1][3]);
    W.loz = make_float4(blo[2][0], blo[2][1], blo[2][2], blo[2][3]);
    W.hiz = make_float4(bhi[2][0], bhi[2][1], bhi[2][2], bhi[2][3]);
}

__global__ void k_tlas_aux(uint32_t n, uint32_t* aux) {
    aux[0] = 0u;  // segment offsets {0, n}
    aux[1] = n;
    aux[2] = 0u;  // node offset
}

// Root refs of each environment's BVH4, known by construction: an LBVH of
// n_e >= 2 leaves has its root at its first node and the collapse puts the
// BVH4 root at the first slot of the environment's range; one instance is a
// leaf root, none an empty one.
void env_roots(const std::vector<uint32_t>& env_off, const std::vector<uint32_t>& node_off, std::vector<int>& roots) {
    const size_t ne = env_off.size() - 1;
    roots.assign(ne, kEmptyRef);
    for (size_t e = 0; e < ne; ++e) {
        const uint32_t n_e = env_off[e + 1] - env_off[e];
        roots[e] = n_e >= 2 ? (int)node_off[e] : (n_e == 1 ? ~(int)env_off[e] : kEmptyRef);
    }
}

// TLAS (re)build, once per instance update: instance records + world boxes,
// an LBVH over the instances of each environment (one segment each), the
// BVH4 collapse of every environment's tree, in one launch when no environment
// has more than kTlasSmall instances (what a block's LDS holds).  Up to
// kTlasDirect instances the kernel reads them from the pinned staging (80
// bytes each over the bus, less than a copy's launch), beyond after a copy.  Nothing here
// waits for the GPU: roots are known by construction (env_roots) and the
// host inputs go through pinned staging.  One environment: its segment and
// node offsets are written on the device (the instance count may change);
// several: they are fixed at scene creation (the count may not).
constexpr uint32_t kTlasSmall = 1024, kTlasDirect = 2048;
void build_tlas(Scene& s, const kf_instance* h_inst, uint32_t n) {
    hipStream_t st = stream();
    const uint32_t TB = 256;
    const bool multi = s.n_env > 1;
    if (multi && n != s.h_env_off.back())
        throw Error("kf_scene_update_instances: a scene with environments keeps its instance count");
    if (h_inst != s.h_inst.data()) s.h_inst.assign(h_inst, h_inst + n);
    if (n != s.n_inst || !s.d_inst) {
        dfree(s.d_inst); dfree(s.d_tlas); dfree(s.d_inst_src); dfree(s.d_ilo); dfree(s.d_ihi);
        s.d_inst = dalloc<Inst>(std::max<uint32_t>(n, 1));
        s.d_ilo = dalloc<float4>(std::max<uint32_t>(n, 1));
        s.d_ihi = dalloc<float4>(std::max<uint32_t>(n, 1));
        s.d_tlas = dalloc<Node>(std::max<uint32_t>(n, 1));
        s.d_inst_src = dalloc<kf_instance>(std::max<uint32_t>(n, 1));
        s.n_inst = n;
    }
    if (!s.d_gflags) {  // static per scene
        s.d_gflags = dalloc<uint32_t>(std::max<uint32_t>(s.n_geom, 1));
        if (s.n_geom)
            KF_CHECK(hipMemcpy(s.d_gflags, s.h_gflags.data(), s.n_geom * sizeof(uint32_t), hipMemcpyHostToDevice));
        s.d_tlas_aux = dalloc<uint32_t>(8);
        s.d_tlas_err = dalloc<int>(1);
        KF_CHECK(hipMemsetAsync(s.d_tlas_err, 0, sizeof(int), st));
        KF_CHECK(hipEventCreateWithFlags(&s.stage_ev, hipEventDisableTiming));
    }
    // host instances -> pinned staging, read by the kernel there (few) or
    // copied to the device (many)
    const size_t inst_bytes = sizeof(kf_instance) * (size_t)n;
    if (s.stage_pending) KF_CHECK(hipEventSynchronize(s.stage_ev));  // the previous update has read it
    s.stage_pending = false;
    if (inst_bytes > s.stage_cap) {
        if (s.h_stage) KF_CHECK(hipHostFree(s.h_stage));
        s.h_stage = nullptr;
        s.stage_cap = 0;
        const size_t cap = std::max<size_t>(inst_bytes, 4096);
        KF_CHECK(hipHostMalloc((void**)&s.h_stage, cap, hipHostMallocDefault));
        s.stage_cap = cap;
    }
    if (n) std::memcpy(s.h_stage, h_inst, inst_bytes);
    uint32_t most = n;  // instances of the largest environment
    if (multi) {
        most = 0;
        for (uint32_t e = 0; e < s.n_env; ++e) most = std::max(most, s.h_env_off[e + 1] - s.h_env_off[e]);
    }
    const bool small = most <= kTlasSmall;
    const bool direct = small && n <= kTlasDirect;
    if (n && !direct) KF_CHECK(hipMemcpyAsync(s.d_inst_src, s.h_stage, inst_bytes, hipMemcpyHostToDevice, st));
    InstArgs A{};
    A.src = direct ? (const kf_instance*)s.h_stage : s.d_inst_src;
    A.n_geom = s.n_geom;
    A.gflags = s.d_gflags;
    A.root = s.d_trav_root4;
    A.blas4 = s.d_blas4;
    A.n_blas4 = s.n_blas4;
    A.glo = s.d_glo;
    A.ghi = s.d_ghi;
    A.mesh = s.d_mesh;
    A.toff = s.d_toff;
    A.out = s.d_inst;
    A.ilo = s.d_ilo;  // kept: the renderer culls instances per pixel tile with them
    A.ihi = s.d_ihi;
    const uint32_t n_seg = multi ? s.n_env : 1u;
    // BVH2 nodes: n_e - 1 per environment of n_e >= 2 instances
    uint32_t n_tlas2 = 0;
    if (multi)
        n_tlas2 = s.h_env_node_off.back();
    else
        n_tlas2 = n > 1 ? n - 1 : 0;
    std::vector<int> roots;
    if (multi)
        env_roots(s.h_env_off, s.h_env_node_off, roots);
    else
        env_roots({0u, n}, {0u}, roots);
    s.tlas_root = roots[0];
    if (!s.d_tlas4 || s.tlas4_cap < std::max<uint32_t>(n_tlas2, 1)) {
        dfree(s.d_tlas4);
        s.tlas4_cap = std::max<uint32_t>(n_tlas2, 1);
        s.d_tlas4 = dalloc<Node4>(s.tlas4_cap);
    }
    uint32_t* cnt = multi ? s.d_env_cnt : s.d_tlas_aux + 3;
    if (small) {
        const uint32_t* eo = multi ? s.d_env_off : nullptr;
        const uint32_t* no = multi ? s.d_env_node_off : nullptr;
        if (!n) {
        } else if (most <= 64u) {
            k_tlas_small<64><<<n_seg, 64, 0, st>>>(n, A, eo, no, s.d_tlas, s.d_tlas4, cnt, s.d_tlas_err);
        } else if (most <= 256u) {
            k_tlas_small<256><<<n_seg, 256, 0, st>>>(n, A, eo, no, s.d_tlas, s.d_tlas4, cnt, s.d_tlas_err);
        } else {
            k_tlas_small<kTlasSmall><<<n_seg, kTlasSmall, 0, st>>>(n, A, eo, no, s.d_tlas, s.d_tlas4, cnt, s.d_tlas_err);
        }
    } else {
        const uint32_t* seg_off = multi ? s.d_env_off : s.d_tlas_aux;
        const uint32_t* node_off = multi ? s.d_env_node_off : s.d_tlas_aux + 2;
        uint32_t* iseg = dalloc<uint32_t>(n);
        uint32_t* order = dalloc<uint32_t>(n);
        int* d_root = dalloc<int>(n_seg);
        int2* qa = dalloc<int2>(n_tlas2);
        int2* qb = dalloc<int2>(n_tlas2);
        k_instances<<<blocks(n, TB), TB, 0, st>>>(n, A, multi ? s.d_inst_env : nullptr, iseg);
        if (!multi) k_tlas_aux<<<1, 1, 0, st>>>(n, s.d_tlas_aux);
        lbvh_build(n, A.ilo, A.ihi, iseg, n_seg, seg_off, node_off, s.d_tlas, order, d_root, false, st);
        k_collapse_forest<<<n_seg, kTreeThreads, 0, st>>>(s.d_tlas, n_tlas2, seg_off, node_off, qa, qb, s.d_tlas4, 0u,
                                                          cnt, s.d_tlas_err);
        dfree(iseg); dfree(order); dfree(d_root); dfree(qa); dfree(qb);
    }
    KF_CHECK(hipGetLastError());
    if (n) {
        KF_CHECK(hipEventRecord(s.stage_ev, st));
        s.stage_pending = true;
    }
    s.tlas_root4 = roots[0];  // BVH4 and BVH2 roots coincide by construction
    s.n_tlas4 = n_tlas2 ? s.tlas4_cap : 0;  // index bound; the node count stays on the device
}

// Geometry g's vertices were replaced on the device (same count, same
// triangles): refit its BLAS on the GPU, no host round trip.
void refit_blas(Scene& s, uint32_t g) {
    hipStream_t st = stream();
    const uint32_t TB = 256;
    const uint32_t n = s.h_toff[g + 1] - s.h_toff[g];
    if (n == 0) return;
    // the slots' boxes and their pyramid, in a workspace that the scene keeps
    // (96 bytes per triangle, half of what the geometry's own arrays take;
    // allocated per call an update of 1.3 M triangles takes 1.91 ms instead of
    // 1.58)
    const size_t need = 2 * (size_t)n * sizeof(float4) + pyramid_size(n) * sizeof(Box);
    if (need > s.refit_cap) {
        dfree(s.d_refit);
        s.d_refit = nullptr;
        s.refit_cap = 0;
        s.d_refit = dalloc<uint8_t>(need);
        s.refit_cap = need;
    }
    float4* lo = (float4*)s.d_refit;
    float4* hi = lo + n;
    k_geom_slots<<<blocks(n, TB), TB, 0, st>>>(g, s.d_verts, s.d_idx, s.d_voff, s.d_toff, s.d_tri, lo, hi);
    if (n >= 2) {
        const Pyramid P = build_pyramid(n, nullptr, lo, hi, (Box*)(hi + n), st);
        k_geom_refit2<<<blocks(n - 1, TB), TB, 0, st>>>(g, s.d_toff, s.d_node_off, s.n_blas_nodes, P, s.d_blas);
        k_geom_refit4<<<blocks(n - 1, TB), TB, 0, st>>>(g, s.d_toff, s.d_node_off, s.d_blas_cnt, s.d_blas,
                                                       s.n_blas_nodes, s.d_tri, s.d_blas4);
    }
    blas_boxes(s);
    KF_CHECK(hipGetLastError());
}

}  // namespace kf
