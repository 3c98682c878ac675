// traverse.h — stack-based two-level BVH traversal with the watertight
// ray/triangle test (gfx950 device code).
//
// Replaces the fixed-function traversal behind traceRayEXT in
// PathTrace.rgen:97-107 (closest hit, tMin 0.001, tMax 1e4) and
// PathTrace.rchit:186-197 (shadow rays: opaque, terminate on first hit).
// Semantics fixed by this build (the reference leaves them to the driver):
//   * watertight test of Woo, Benthin & Wald (JCGT 2013), double-precision
//     fallback when an edge function is exactly zero;
//   * accept t in [tmin, tmax]; closest hit = smallest t, ties broken by the
//     smaller (instance, primitive) pair.  Hits a few roundings of t apart may
//     cull each other (ChildOrder), so the visiting order is part of the result:
//     it is fixed by the tree and the ray;
//   * hit kind front-facing iff dot(d_obj, cross(v1 - v0, v2 - v0)) < 0;
//   * the object-space ray is (W2O * (o,1), W2O * (d,0)), t is shared.
#pragma once
#include "kf_internal.h"
#include "kf_math.h"

namespace kf {

constexpr int kStack = 65;
constexpr uint32_t kMaxSteps = 1u << 22;  // bound on loop iterations (malformed-tree guard)
// Slab margin: each computed slab distance (b - o) * rcp(d) carries three
// roundings, one of them the 1-ulp hardware reciprocal (2 units of 2^-24),
// so |relative error| <= gamma_4; near <= far * (1 + 2 gamma_5) then never
// rejects a box the exact ray meets (Ize, "Robust BVH ray traversal", 2013).
constexpr float kUnit = 5.96046448e-8f;  // 2^-24
constexpr float kGamma5 = 5.0f * kUnit / (1.0f - 5.0f * kUnit);
constexpr float kSlabScale = 1.0f + 2.0f * kGamma5;

// The shear of the watertight test for a wave's object-space rays: axes kx,
// ky, kz as wave-wide lane masks (bit l: lane l; k0: axis 0, k1: axis 1,
// neither: axis 2), which the compiler holds in scalar registers, and the
// scales Sz = 1 / d[kz] correctly rounded, Sx = d[kx] * Sz, Sy = d[ky] * Sz.
struct Axes {
    uint64_t x0, x1, y0, y1, z0, z1;
};
struct Pre {
    bool x0, x1, y0, y1, z0, z1;  // one lane's axes
    float Sx, Sy, Sz;
};

KF_DEV float comp2(v3 a, bool k0, bool k1) { return k0 ? a.x : (k1 ? a.y : a.z); }
// Component-wise choice.  (c ? a : b on structure lvalues compiles to a copy
// from a chosen address, which forces the traversal state into memory.)
KF_DEV v3 sel3(bool c, v3 a, v3 b) { return mk(c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z); }
KF_DEV v3 rcp3(v3 d) { return mk(__builtin_amdgcn_rcpf(d.x), __builtin_amdgcn_rcpf(d.y), __builtin_amdgcn_rcpf(d.z)); }
KF_DEV uint64_t lanes_of(bool c) { return __builtin_amdgcn_ballot_w64(c); }
KF_DEV bool lane_in(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// Shear axes of rays with direction d for the lanes in E; the others keep
// theirs.  kz = the dominant axis, (kx, ky) swapped when d[kz] < 0 to keep
// the winding: kz = (ax >= ay) ? ((ax >= az) ? 0 : 2) : ((ay >= az) ? 1 : 2),
// kx = kz + 1 and ky = kz + 2 (mod 3).  Scalar logic on the ballots of the
// four comparisons: as per-lane flags the compiler made 0/1 registers of them
// and compared those again (25 vector instructions per step).  Returns d[kz].
KF_DEV float shear_axes(v3 d, uint64_t E, Axes& A) {
    const float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    const uint64_t xy = lanes_of(ax >= ay), xz = lanes_of(ax >= az), yz = lanes_of(ay >= az);
    const uint64_t z0 = xy & xz, z1 = ~xy & yz, z2 = ~(z0 | z1);
    const float dz = comp2(d, lane_in(z0), lane_in(z1));
    const uint64_t sw = lanes_of(dz < 0.0f);
    A.z0 = (z0 & E) | (A.z0 & ~E);
    A.z1 = (z1 & E) | (A.z1 & ~E);
    A.x0 = (((sw & z1) | (~sw & z2)) & E) | (A.x0 & ~E);  // the (swapped) x axis is 0
    A.x1 = (((sw & z2) | (~sw & z0)) & E) | (A.x1 & ~E);  // ... is 1
    A.y0 = (((sw & z2) | (~sw & z1)) & E) | (A.y0 & ~E);  // the (swapped) y axis is 0
    A.y1 = (((sw & z0) | (~sw & z2)) & E) | (A.y1 & ~E);  // ... is 1
    return dz;
}

struct TriHit {
    float t, b1, b2;
    uint32_t back;
};

// Watertight ray/triangle test without early exits (the caller runs it for
// every lane of a wave) on the vertices relative to the ray origin, in two
// parts around its one division 1 / det, so that a caller can share that
// division: intersect_begin returns the edge
// functions, det and the scaled distance; intersect_end takes the correctly
// rounded 1 / det.  en gates the double-precision fallback so that lanes
// holding other records never take it.
struct TriEdge {
    float U, V, W, det, Tn;
    bool outside;
};
KF_DEV TriEdge intersect_begin(const Pre& p, v3 A, v3 B, v3 C, bool en) {  // A, B, C: vertices - ray origin
    float Akz = comp2(A, p.z0, p.z1), Bkz = comp2(B, p.z0, p.z1), Ckz = comp2(C, p.z0, p.z1);
    float Ax = comp2(A, p.x0, p.x1) - p.Sx * Akz;
    float Ay = comp2(A, p.y0, p.y1) - p.Sy * Akz;
    float Bx = comp2(B, p.x0, p.x1) - p.Sx * Bkz;
    float By = comp2(B, p.y0, p.y1) - p.Sy * Bkz;
    float Cx = comp2(C, p.x0, p.x1) - p.Sx * Ckz;
    float Cy = comp2(C, p.y0, p.y1) - p.Sy * Ckz;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (en && (U == 0.0f || V == 0.0f || W == 0.0f)) {
        U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
        V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
        W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
    }
    TriEdge e;
    e.outside = (U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f);
    e.det = U + V + W;
    const float Az = p.Sz * Akz;
    const float Bz = p.Sz * Bkz;
    const float Cz = p.Sz * Ckz;
    e.Tn = U * Az + V * Bz + W * Cz;
    e.U = U;
    e.V = V;
    e.W = W;
    return e;
}
KF_DEV bool intersect_end(const TriEdge& e, float rcp_det, float tmin, float tmax, TriHit& h) {
    const float t = e.Tn * rcp_det;
    h.t = t;
    h.b1 = e.V * rcp_det;
    h.b2 = e.W * rcp_det;
    h.back = __float_as_uint(e.det) & 0x80000000u;  // det < 0 (a hit's det is neither 0 nor NaN)
    return !e.outside && e.det != 0.0f && t >= tmin && t <= tmax;
}

KF_DEV float alpha_coin(uint32_t seed, uint32_t inst, uint32_t prim) {
    uint32_t h = tea(seed ^ (inst * 0x9e3779b9u), prim);
    return float(h & 0x00FFFFFFu) / float(0x01000000);
}

struct THit {
    float t, b1, b2;
    uint32_t inst, prim, back;
};

struct TCount {
    uint32_t nodes, tris, insts;  // BVH4 node records, triangle tests, instance records
    uint32_t tlas;                // of the node records, TLAS ones
};

KF_DEV v3 xform_point(const Inst& I, v3 v) {
    return mk(I.w2o[0].x * v.x + I.w2o[0].y * v.y + I.w2o[0].z * v.z + I.w2o[0].w,
              I.w2o[1].x * v.x + I.w2o[1].y * v.y + I.w2o[1].z * v.z + I.w2o[1].w,
              I.w2o[2].x * v.x + I.w2o[2].y * v.y + I.w2o[2].z * v.z + I.w2o[2].w);
}
KF_DEV v3 xform_dir(const Inst& I, v3 v) {
    return mk(I.w2o[0].x * v.x + I.w2o[0].y * v.y + I.w2o[0].z * v.z,
              I.w2o[1].x * v.x + I.w2o[1].y * v.y + I.w2o[1].z * v.z,
              I.w2o[2].x * v.x + I.w2o[2].y * v.y + I.w2o[2].z * v.z);
}

// ---------------------------------------------------------------- traversal
// The traversal is a state machine over 32-bit items: bits 31:30 the kind,
// bits 29:0 an index into that kind's array.  Every step fetches exactly one
// record (BVH4 node, instance record, triangle) and processes it, so all
// lanes of a wave wait on one memory round trip per step whatever kind of
// record each lane is on.  An instance record carries its BLAS root node:
// its step transforms the ray and tests the root's children at once, so
// entering an instance costs no step of its own.  The newest stack entry is
// read with every record fetch, so a pop costs no extra round trip.
enum : uint32_t { kTlasNode = 0u, kBlasNode = 1u, kInstance = 2u, kTriangle = 3u };
constexpr uint32_t kIdxMask = 0x3fffffffu;  // scenes are limited to 2^30 records of each kind
constexpr uint32_t kNoPrim = 0x7fffffffu;   // best.prim before the first hit

KF_DEV uint32_t make_item(uint32_t kind, uint32_t idx) { return (kind << 30) | (idx & kIdxMask); }

// Record arrays of the traversal.  Where a lane chooses between them by the
// kind of its record, each field passes through an empty asm first: that
// keeps the choice a register select, which the optimiser otherwise turns
// into a dynamically indexed private-memory copy of the whole structure.
typedef float vf4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) vf4 gf4;  // vf4 in the global address space

template <class T>
KF_DEV T opaque_sgpr(T v) {
    asm volatile("" : "+s"(v));
    return v;
}

struct TravScene {
    const float4 *tlas, *blas, *inst, *tri;
    uint32_t n_tlas, n_blas, n_inst, n_tri;
    const kf_material* mats;
    const uint32_t *matidx, *toff;
    KF_DEV explicit TravScene(const SceneView& S)
        : tlas((const float4*)S.tlas), blas((const float4*)S.blas), inst((const float4*)S.inst), tri(S.tri),
          n_tlas(S.n_tlas_nodes), n_blas(S.n_blas_nodes), n_inst(S.n_inst), n_tri(S.n_tri),
          mats(S.mats), matidx(S.matidx), toff(S.toff) {}
};

// ------------------------------------------------------------- stacks
// A lane's traversal stack.  Entry i is the i-th oldest; sp counts the
// entries.
//   peek(sp): entry sp - 1 (read speculatively every step; any in-range
//             address when sp == 0);
//   push(sp, k, e0, e1, e2): store the first k of e0, e1, e2 as entries sp,
//             sp + 1, sp + 2; returns the lanes that had room for them (a
//             malformed tree: not all);
//   popped(sp): entry sp has just been taken (sp is the new count).
struct PrivStack {  // everything in private memory
    static constexpr uint32_t kCap = kStack;
    uint32_t a[kStack];
    KF_DEV uint32_t peek(uint32_t sp) const { return a[sp > 0u ? sp - 1u : 0u]; }
    KF_DEV uint64_t push(uint32_t sp, uint32_t k, uint32_t e0, uint32_t e1, uint32_t e2) {
        const uint64_t room = lanes_of(sp + k <= kCap);
        k = sp + k <= kCap ? k : 0u;
        if (k > 0u) a[sp] = e0;
        if (k > 1u) a[sp + 1u] = e1;
        if (k > 2u) a[sp + 2u] = e2;
        return room;
    }
    KF_DEV void popped(uint32_t) {}
};

// The newest kRing entries in an LDS ring, one column per thread of the
// block (slot-major, so a wave's accesses hit 64 distinct banks whatever
// slots its lanes use); older entries spill to private memory.  Private
// stores dirty whole cache lines that end up written back to HBM, so the
// ring keeps the common shallow stack off the memory system entirely.
// The ring pointer is typed as an LDS (address space 3) pointer and the spill
// array lives outside the struct: with both in one struct the whole struct
// stayed in scratch, so every step reloaded the ring pointer from scratch and
// reached the ring through flat loads and stores (which wait on every
// outstanding global load as well).
constexpr uint32_t kRing = 16;            // power of two
constexpr uint32_t kRingThreads = 256;    // block size of kernels using RingStack
typedef __attribute__((address_space(3))) uint32_t lds_u32;
struct RingStack {
    static constexpr uint32_t kCap = kRing + kStack;
    lds_u32* ring;    // this thread's column: slot k at ring[k * kRingThreads]
    uint32_t* spill;  // kStack entries in private memory
    KF_DEV lds_u32& slot(uint32_t i) const { return ring[(i & (kRing - 1u)) * kRingThreads]; }
    KF_DEV uint32_t peek(uint32_t sp) const { return slot(sp - 1u); }
    KF_DEV uint64_t push(uint32_t sp, uint32_t k, uint32_t e0, uint32_t e1, uint32_t e2) {
        // While no lane of the wave is near the ring's end all three are
        // stored unasked: what lies above the new count is free.
        if (lanes_of(sp + 3u > kRing) == 0u) {
            lds_u32* w = ring + sp * kRingThreads;
            w[0] = e0;
            w[kRingThreads] = e1;
            w[2u * kRingThreads] = e2;
            return ~0ull;
        }
        const uint64_t room = lanes_of(sp + k <= kCap);
        k = sp + k <= kCap ? k : 0u;
        for (uint32_t i = 0; i < k; ++i) {
            const uint32_t s = sp + i;
            if (s >= kRing) spill[s - kRing] = slot(s);  // evict the entry that shares the slot
            slot(s) = i == 0u ? e0 : (i == 1u ? e1 : e2);
        }
        return room;
    }
    KF_DEV void popped(uint32_t sp) {
        if (sp >= kRing) slot(sp) = spill[sp - kRing];  // bring the next older entry back into the ring
    }
};

static_assert(RingStack::kCap < 256 && PrivStack::kCap < 256, "stack depth in the low byte of Trav::spx");

// One query: ray, t range, the TLAS root item it starts from (its
// environment's; kEmptyItem: nothing to hit), alpha coin seed and an opaque
// payload for the caller (where to write the result).
struct TRay {
    v3 o, d;
    float tmin, tmax;
    uint32_t root, alpha_seed, payload;
};

KF_DEV uint32_t root_item(int root) {
    return root >= 0 ? make_item(kTlasNode, (uint32_t)root) : make_item(kInstance, (uint32_t)~root);
}

// Root item of environment e's TLAS (the whole TLAS for a scene without
// environments); kEmptyItem when the environment has no instance.
KF_DEV uint32_t env_root_item(const SceneView& S, uint32_t e) {
    if (S.n_env > 1) return S.env_root[e < S.n_env ? e : 0u];
    return S.tlas_root == kEmptyRef ? kEmptyItem : root_item(S.tlas_root);
}

// The four children of a node in the order of their keys, by the sorting
// network (0,1)(2,3)(0,2)(1,3)(1,2).
// Closest hits exchange two children on their distances alone, so that the
// order follows from the ray and the children's places in the node.  Equal
// distances are the usual case (every box around a ray's origin is entered at
// tmin), and the order among them can decide a hit: the culling bound does not
// cover the rounding of a triangle's own distance, so of two surfaces hit
// within a few roundings of each other the first one found may drop the other.
// With the item as a second key, as below, that order followed the numbering
// of nodes and instances: 643 of 1 M rays from within 5 mm of bodies' feet got
// another hit (distances up to 3.4e-7 m apart over a ground of 4 m).  The
// selects cost 2 % on a 256x256 frame (866 -> 883 us), elsewhere below 1 %.
// An any-hit query is the same in every order.  It sorts (distance, item) as
// one 64-bit float, an exchange a min and a max instead of a comparison and
// selects (no key is a NaN: the high word is a float).
template <bool ANY> struct ChildOrder {
    uint32_t item[4];
    KF_DEV ChildOrder(const float (&k)[4], const uint32_t (&it)[4]) {
        float key[4] = {k[0], k[1], k[2], k[3]};
        for (int c = 0; c < 4; ++c) item[c] = it[c];
        auto cx = [&](int i, int j) __attribute__((always_inline)) {
            const bool sw = key[j] < key[i];
            const float ki = key[i], kj = key[j];
            const uint32_t ii = item[i], ij = item[j];
            key[i] = sw ? kj : ki;
            key[j] = sw ? ki : kj;
            item[i] = sw ? ij : ii;
            item[j] = sw ? ii : ij;
        };
        cx(0, 1);
        cx(2, 3);
        cx(0, 2);
        cx(1, 3);
        cx(1, 2);
    }
};
template <> struct ChildOrder<true> {
    uint32_t item[4];
    KF_DEV ChildOrder(const float (&k)[4], const uint32_t (&it)[4]) {
        double key[4];
        for (int c = 0; c < 4; ++c) key[c] = __hiloint2double((int)__float_as_uint(k[c]), (int)it[c]);
        auto cx = [&](int i, int j) __attribute__((always_inline)) {
            const double a = key[i], b = key[j];
            asm("v_min_f64 %0, %1, %2" : "=v"(key[i]) : "v"(a), "v"(b));
            asm("v_max_f64 %0, %1, %2" : "=v"(key[j]) : "v"(a), "v"(b));
        };
        cx(0, 1);
        cx(2, 3);
        cx(0, 2);
        cx(1, 3);
        cx(1, 2);
        for (int c = 0; c < 4; ++c) item[c] = (uint32_t)__double2loint(key[c]);
    }
};

// ANY: shadow-ray query (opaque, stop at the first hit in [tmin, tmax]).
// Closest-hit queries with use_alpha run the any-hit alpha test
// (PathTrace.rahit:30-48) for non-opaque instances, with an order-independent
// coin (alpha_coin).  MIXED (with ANY false): each lane's query is a shadow
// query or a closest-hit one (any_q), so that lanes of one wave trace both
// kinds with the same steps.
// What bounds it: the vector ALUs (about 345 instructions per step) and the
// vector L1 about equally.  Each lane loading its own record's lines only, the
// shear axes as scalar logic and a stack without a cached top took 17 % of the
// vector instructions and 26 % of the L1 accesses:
// 2 M rays 1.05 -> 0.97 ms, 1080p frame at 16 spp 18.7 -> 17.2 ms, 128
// environments of 512x512 at 8 spp 137.7 -> 129 ms.
template <bool ANY, bool COUNT, bool MIXED = false>
struct Trav {
    v3 o, d;         // world-space ray
    // The ray of the level the lane is at: the world-space one in a TLAS, the
    // current instance's object-space one in its BLAS (a BLAS's items lie on
    // the stack above all TLAS items, so the world-space one is back before
    // the next instance); ri: 1 / direction, culling only (hardware reciprocal).
    v3 ro, ri;
    Axes ax;         // shear of the current instance's object-space ray
    float Sx, Sy, Sz;
    float tmin;
    THit best;
    uint32_t cur_inst;  // instance whose BLAS the object-space ray belongs to
    uint32_t cur;    // item processed by the next step
    uint32_t spx;    // bits 7:0 the stack's entries, bits 31:8 the steps taken
                     // (malformed-tree guard); 0 without a query
    bool found, use_alpha;
    bool any_q;      // MIXED: this lane's query is a shadow query
    uint32_t alpha_seed;
    TCount cnt;

    // Benign state for a lane without a query.
    KF_DEV void reset() {
        o = d = ro = ri = mk(0.0f, 0.0f, 0.0f);
        ax.x0 = ax.y1 = ~0ull;  // kx = 0, ky = 1, kz = 2
        ax.x1 = ax.y0 = ax.z0 = ax.z1 = 0ull;
        Sx = Sy = Sz = 0.0f;
        tmin = 0.001f;  // the path tracer's constant, so that its kernels can fold it
        best.t = best.b1 = best.b2 = 0.0f;
        best.inst = ~0u;
        best.prim = kNoPrim;  // closest hit: bit 31 holds the hit kind while tracing
        best.back = 0u;
        cur_inst = 0u;
        cur = 0u;
        spx = 0u;
        found = false;
        use_alpha = false;
        any_q = false;
        alpha_seed = 0u;
        cnt.nodes = cnt.tris = cnt.insts = cnt.tlas = 0u;
    }

    // Lanes with f take a new query r starting at item root (the scene is
    // not empty); the others keep their state.  Written as selects so that
    // refilling some lanes does not copy the state of all of them.
    KF_DEV void start(bool f, const TRay& r, uint32_t root, bool use_alpha_) {
        o = sel3(f, r.o, o);
        d = sel3(f, r.d, d);
        tmin = f ? r.tmin : tmin;
        best.t = f ? r.tmax : best.t;
        best.inst = f ? ~0u : best.inst;
        best.prim = f ? kNoPrim : best.prim;
        best.b1 = f ? 0.0f : best.b1;
        best.b2 = f ? 0.0f : best.b2;
        best.back = f ? 0u : best.back;
        cur = f ? root : cur;
        spx = f ? 0u : spx;
        found = f ? false : found;
        use_alpha = f ? use_alpha_ : use_alpha;
        alpha_seed = f ? r.alpha_seed : alpha_seed;
        cnt.nodes = f ? 0u : cnt.nodes;
        cnt.tlas = f ? 0u : cnt.tlas;
        cnt.tris = f ? 0u : cnt.tris;
        cnt.insts = f ? 0u : cnt.insts;
    }

    // The query's result: closest hits keep the hit kind in bit 31 of
    // best.prim while tracing.
    KF_DEV THit result() const {
        THit r = best;
        const bool hit = !ANY && found;
        r.prim = hit ? (best.prim & 0x7fffffffu) : ~0u;
        r.back = hit ? (best.prim >> 31) : 0u;
        return r;
    }

    // One record for each lane in `live`, the lanes that hold a query; returns
    // those whose query has not finished.  stk: the
    // query's stack (a separate object so that the scalar state above stays in
    // registers).
    //
    // The newest stack entry is loaded speculatively together with the
    // record, so a pop needs no memory access of its own: every step costs
    // the wave one memory round trip.
    // Lanes without a query fetch nothing and have no side effects beyond
    // their own (discarded) state.  Sets of lanes are masks in scalar
    // registers; as per-lane flags they cost a select and a comparison each.
    template <class Stack>
    KF_DEV uint64_t step(const TravScene& S, Stack& stk, uint32_t& overflow, uint64_t live) {
        const uint32_t kind = cur >> 30, idx = cur & kIdxMask;
        // All operands of the per-lane choices are evaluated unconditionally,
        // so the choices stay selects (an asm cannot be speculated).
        const uint32_t n_tlas = opaque_sgpr(S.n_tlas), n_blas = opaque_sgpr(S.n_blas);
        const uint32_t n_inst = opaque_sgpr(S.n_inst), n_tri = opaque_sgpr(S.n_tri);
        const float4 *p_tlas = opaque_sgpr(S.tlas), *p_blas = opaque_sgpr(S.blas);
        const float4 *p_inst = opaque_sgpr(S.inst), *p_tri = opaque_sgpr(S.tri);
        const uint32_t lim = kind == kTlasNode ? n_tlas : kind == kBlasNode ? n_blas : kind == kInstance ? n_inst : n_tri;
        // Out-of-range record or step budget spent (malformed tree): fetch
        // nothing and finish the query with the overflow flag.  Kept free of
        // early exits: one here makes the compiler copy the whole traversal
        // state on every step.
        const uint32_t sp = spx & 0xffu;
        spx += 0x100u;  // this step counted
        const uint64_t ON = live & lanes_of(idx < lim) & lanes_of(spx <= ((kMaxSteps << 8) | 0xffu));
        const bool on = lane_in(ON);
        const float4* base = kind == kTlasNode ? p_tlas : kind == kBlasNode ? p_blas : kind == kInstance ? p_inst : p_tri;
        const uint32_t lines = kind <= kBlasNode ? 8u : (kind == kTriangle ? 3u : 12u);
        const gf4* G = (const gf4*)(base + (size_t)lines * idx);
        const uint64_t tri_kind = lanes_of(kind == kTriangle);
        const uint64_t E = ON & lanes_of(kind == kInstance);
        const bool is_node = lane_in(ON & ~tri_kind), is_tri = lane_in(ON & tri_kind), is_inst = lane_in(E);
        // 16-byte global loads issued together: lines 0-2 of any record, a
        // node's low planes or a triangle's x, y and z; lines 3-6 of a node or
        // of an instance record's root node; lines 7-9 of an instance record,
        // its transform.  Each lane loads only its record's lines: the vector
        // L1 serves one lane's line per cycle, so that ten loads by all 64
        // lanes kept it busy 87 % of the time beside vector ALUs at 82 % (2 M
        // rays, 256 icospheres).  The empty asm needs all results, which keeps the
        // compiler from sinking parts of the fetch into the kind-specific
        // code below (each sunk load would cost the wave another memory round
        // trip); what a lane did not load is any value.
        vf4 r0, r1, r2, r3, r4, r5, r6, r7, r8, r9;
        if (on) {
            r0 = G[0];
            r1 = G[1];
            r2 = G[2];
            if (is_node) {
                r3 = G[3];
                r4 = G[4];
                r5 = G[5];
                r6 = G[6];  // line 7 of a node is for its refits
                if (is_inst) {
                    r7 = G[7];
                    r8 = G[8];
                    r9 = G[9];
                }
            }
        }
        uint32_t below = stk.peek(sp);
        asm volatile("" : "+v"(r0), "+v"(r1), "+v"(r2), "+v"(r3), "+v"(r4), "+v"(r5), "+v"(r6), "+v"(r7), "+v"(r8),
                     "+v"(r9), "+v"(below));

        // Every lane evaluates the record as a node, an instance and a
        // triangle and keeps the result of its kind: per-lane branches would
        // copy the traversal state at each join, and a full wave64 has lanes
        // of all three kinds in nearly every step.  Waves with few queries
        // left do not: the instance and triangle evaluations are skipped when
        // no lane of the wave needs them (wave-uniform branches).  With the
        // branches 2 M rays against the 256-icosphere scene take 1.09 ms
        // instead of 1.13, 4096 rays 0.15 instead of 0.16 (whole calls), and
        // the long launches of full waves are no slower.  An instance record
        // is a node as well (its BLAS root's children).
        const bool any_inst = E != 0u;
        const bool any_tri = (ON & tri_kind) != 0u;

        // instance: its BLAS is entered with the object-space ray, which this
        // step's node test already uses for the BLAS root's children (an
        // invalid instance's record has no children, so entering it changes
        // nothing the traversal reads later).  Other lanes keep their ray.
        // A lane enters an instance or tests a triangle, never both: the two
        // correctly rounded reciprocals (1 / d[kz] of the new shear, 1 / det
        // of the triangle) share one division.
        const bool world = kind == kTlasNode;
        ro = sel3(world, o, ro);
        v3 nd = d;
        float dz = 1.0f;
        if (any_inst) {
            Inst I;
            I.w2o[0] = make_float4(r7.x, r7.y, r7.z, r7.w);
            I.w2o[1] = make_float4(r8.x, r8.y, r8.z, r8.w);
            I.w2o[2] = make_float4(r9.x, r9.y, r9.z, r9.w);
            ro = sel3(is_inst, xform_point(I, o), ro);
            nd = sel3(is_inst, xform_dir(I, d), d);
            dz = shear_axes(nd, E, ax);
            cur_inst = is_inst ? idx : cur_inst;
        }
        // one set of hardware reciprocals (culling only) where the ray
        // changes: the world ray of a TLAS node, the new object-space ray of
        // an instance
        ri = sel3(world || is_inst, rcp3(nd), ri);

        // The low planes against that ray's origin; on a triangle's lines the
        // triangle's vertices relative to the object-space origin.
        const float dlx[4] = {r0.x - ro.x, r0.y - ro.x, r0.z - ro.x, r0.w - ro.x};
        const float dly[4] = {r1.x - ro.y, r1.y - ro.y, r1.z - ro.y, r1.w - ro.y};
        const float dlz[4] = {r2.x - ro.z, r2.y - ro.z, r2.z - ro.z, r2.w - ro.z};

        // triangle, against the current instance's object-space ray (lanes
        // entering an instance discard it)
        Pre pre;
        pre.x0 = lane_in(ax.x0);
        pre.x1 = lane_in(ax.x1);
        pre.y0 = lane_in(ax.y0);
        pre.y1 = lane_in(ax.y1);
        pre.z0 = lane_in(ax.z0);
        pre.z1 = lane_in(ax.z1);
        pre.Sx = Sx;
        pre.Sy = Sy;
        pre.Sz = Sz;
        TriEdge te;
        te.det = 1.0f;
        if (any_tri)
            te = intersect_begin(pre, mk(dlx[0], dly[0], dlz[0]), mk(dlx[1], dly[1], dlz[1]),
                                 mk(dlx[2], dly[2], dlz[2]), is_tri);
        TriHit h;
        bool tri_hit = false;
        if (any_tri || any_inst) {
            const float q = 1.0f / (is_inst ? dz : te.det);
            if (any_tri) tri_hit = intersect_end(te, q, tmin, best.t, h) && is_tri;
            if (any_inst) {
                Sx = is_inst ? comp2(nd, pre.x0, pre.x1) * q : Sx;
                Sy = is_inst ? comp2(nd, pre.y0, pre.y1) * q : Sy;
                Sz = is_inst ? q : Sz;
            }
        }
        const uint32_t prim = __float_as_uint(r0.w);
        bool take = tri_hit;
        if (!ANY) {
            const bool closer = h.t < best.t || cur_inst < best.inst ||
                                (cur_inst == best.inst && prim < (best.prim & 0x7fffffffu));
            take = take && ((MIXED && any_q) || closer);
            // scenes with non-opaque geometry only: the instance's flags and
            // geometry are read here, for candidate hits
            if (take && use_alpha) {
                const float4 info = S.inst[12u * (size_t)cur_inst + 10u];  // Inst::info
                if (!(__float_as_int(info.z) & kInstOpaque)) {
                    const float a = S.mats[S.matidx[S.toff[__float_as_uint(info.y)] + prim]].alpha;
                    take = !(a == 0.0f || alpha_coin(alpha_seed, cur_inst, prim) > a);
                }
            }
        }
        best.t = take ? h.t : best.t;
        if (!ANY) {
            best.b1 = take ? h.b1 : best.b1;
            best.b2 = take ? h.b2 : best.b2;
            best.inst = take ? cur_inst : best.inst;
            best.prim = take ? (prim | h.back) : best.prim;
        }
        found = found || take;

        // node: four child boxes (lines lox, loy, loz, hix, hiy, hiz, ref)
        // against the level's ray, nearest first.
        const float hix[4] = {r3.x, r3.y, r3.z, r3.w};
        const float hiy[4] = {r4.x, r4.y, r4.z, r4.w};
        const float hiz[4] = {r5.x, r5.y, r5.z, r5.w};
        const uint32_t item[4] = {__float_as_uint(r6.x), __float_as_uint(r6.y), __float_as_uint(r6.z), __float_as_uint(r6.w)};
        float key[4];
        uint32_t n = 0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float l0x = dlx[c] * ri.x, l1x = (hix[c] - ro.x) * ri.x;
            const float l0y = dly[c] * ri.y, l1y = (hiy[c] - ro.y) * ri.y;
            const float l0z = dlz[c] * ri.z, l1z = (hiz[c] - ro.z) * ri.z;
            const float tn = fmaxf(fmaxf(fminf(l0x, l1x), fminf(l0y, l1y)), fmaxf(fminf(l0z, l1z), tmin));
            const float tf = fminf(fminf(fmaxf(l0x, l1x), fmaxf(l0y, l1y)), fminf(fmaxf(l0z, l1z), best.t));
            const bool h = tn <= tf * kSlabScale && item[c] != kEmptyItem;
            // Nearer child first; any-hit queries take leaf children
            // (triangles, instances: kinds 2 and 3) before inner ones, which
            // finds occluders sooner.
            key[c] = h ? (((ANY || (MIXED && any_q)) && (item[c] >> 31)) ? -INFINITY : tn) : INFINITY;
            n += h ? 1u : 0u;
        }
        const ChildOrder<ANY> order(key, item);
        const uint32_t c0 = order.item[0], c1 = order.item[1], c2 = order.item[2], c3 = order.item[3];

        if (COUNT) {
            cnt.nodes += (kind <= kBlasNode && on) ? 1u : 0u;
            cnt.tlas += (on && kind == kTlasNode) ? 1u : 0u;
            cnt.tris += is_tri ? 1u : 0u;
            cnt.insts += is_inst ? 1u : 0u;
        }
        // The nearest of n hit children is next and the n - 1 others are
        // pushed, farthest first; without one the newest entry is popped.
        n = is_node ? n : 0u;
        const bool pop = n == 0u;
        uint64_t alive = ON & lanes_of(n + sp != 0u);
        if (ANY || MIXED) alive &= ~lanes_of((ANY || any_q) && take);
        const uint64_t room = stk.push(sp, pop ? 0u : n - 1u, n == 2u ? c1 : (n == 3u ? c2 : c3), n == 3u ? c1 : c2, c1);
        overflow |= lane_in(live & ~(ON & room)) ? 1u : 0u;
        alive &= room;
        cur = pop ? below : c0;
        if (pop && sp > 0u) stk.popped(sp - 1u);
        spx = lane_in(alive) ? spx + n - 1u : 0u;
        return alive;
    }
};

// This thread's column of the block's stack ring (blocks of kRingThreads).
KF_DEV lds_u32* ring_column() {
    __shared__ uint32_t ring[kRing * kRingThreads];
    return (lds_u32*)(ring + threadIdx.x);
}

// Whole query for one lane (used where rays are generated inside a kernel).
template <bool ANY, bool COUNT>
KF_DEV bool traverse(const SceneView& S, uint32_t root, v3 o, v3 d, float tmin, float tmax, bool use_alpha,
                     uint32_t alpha_seed, THit& best, TCount& cnt, uint32_t& overflow) {
    const TravScene TS(S);
    Trav<ANY, COUNT> T;
    uint32_t spill[kStack];
    RingStack stk;
    stk.ring = ring_column();
    stk.spill = spill;
    T.reset();
    TRay r;
    r.o = o;
    r.d = d;
    r.tmin = tmin;
    r.tmax = tmax;
    r.root = root;
    r.alpha_seed = alpha_seed;
    r.payload = 0u;
    T.start(true, r, root, use_alpha);
    if (root != kEmptyItem)
        while (lane_in(T.step(TS, stk, overflow, lanes_of(true)))) {
        }
    best = T.result();
    cnt.nodes += T.cnt.nodes;
    cnt.tlas += T.cnt.tlas;
    cnt.tris += T.cnt.tris;
    cnt.insts += T.cnt.insts;
    return T.found;
}

// ------------------------------------------------------- persistent driver
// Queries [0, n) are split into 8 contiguous chunks, one per XCD (workgroups
// are dispatched to the 8 XCDs round-robin, so block b runs on XCD b % 8 and
// neighbouring queries share that XCD's L2).  A wave reserves queries from
// its chunk's counter and refills its idle lanes from that reserve once at
// least `refill` lanes are idle (or all are), so no lane waits for the
// slowest ray of a fixed group.  When its chunk is used up the wave looks at
// all eight counters at once and moves to the next chunk with queries left.
//
// Reservation size: half an equal share of what its chunk has left, from
// kGrabMin queries up to `grab`, so that a launch ends evenly; at most one
// query per lane in launches with fewer queries than lanes.  The counters sit
// on lines of their own (kChunkStride): with all eight on one line and 128
// queries per reservation the atomics of all XCDs queued up behind each other
// and bounded the long queues (whole frames with the default schedule: 128
// environments of 512x512 at 8 spp 397 -> 159 ms, with the batches and tail
// bounce of render_frame; 720p projector at 32 spp 57.4 -> 24.9 ms; 2 M rays
// 1.45 -> 1.03 ms).  Measured around it: at most 512 or 1024 queries 2 and 6 %
// slower on the 1080p frame (17.2 ms), 128 1 % slower on the projector and
// the environments; a quarter of the share 1-4 % slower on 2 M rays and the
// projector, all of it 18 % on 2 M rays; at least 32 queries 1 % slower on the
// 1080p frame, 4 % denoised at 1 spp; at least 256 3 % slower on 2 M rays; the
// queries of short launches spread at 4, 16 or 32 per wave instead of one per
// lane 11, 5 and 4 % slower on a 256x256 frame.
//   ctr[8 * kChunkStride]: per-chunk counters, zero before the launch.
//   load(q, TRay&) fills the ray of query q and its payload;
//   store(payload, best, found) writes a finished query.
constexpr uint32_t kGrab = 256, kGrabMin = 64;  // kGrab: default grab
constexpr uint32_t kChunkStride = 16;  // 8-byte counters per 128-byte line

KF_DEV uint64_t chunk_begin(uint32_t n, uint32_t c) { return (uint64_t)n * c / 8u; }

template <bool ANY, bool COUNT, class Load, class Store>
KF_DEV void trace_persistent(const SceneView& S, uint32_t n, unsigned long long* __restrict__ ctr, uint32_t refill,
                             uint32_t grab, bool use_alpha, Load load, Store store, uint32_t& overflow,
                             TCount& total) {
    const TravScene TS(S);
    Trav<ANY, COUNT> T;
    T.reset();
    uint32_t spill[kStack];
    RingStack stk;
    stk.ring = ring_column();
    stk.spill = spill;
    uint64_t live = 0;  // lanes that hold a query
    uint32_t payload = 0;
    const uint32_t waves = gridDim.x * (kRingThreads / 64u);
    const uint32_t most = n < 64u * waves ? 64u : ~0u;  // queries of one reservation
    uint32_t chunk = blockIdx.x & 7u;  // wave-uniform from here on
    bool more = n > 0u;                // some chunk may have queries left
    uint32_t seen = ~0u;               // queries of this chunk known to be taken (~0: not looked at yet)
    uint32_t res_q = 0, res_n = 0;     // reserved queries [res_q, res_q + res_n)
    auto finish = [&](uint64_t alive) __attribute__((always_inline)) {
        const bool done = lane_in(live & ~alive);
        live &= alive;
        if (done) {
            store(payload, T.result(), T.found);
            if (COUNT) {
                total.nodes += T.cnt.nodes;
                total.tlas += T.cnt.tlas;
                total.tris += T.cnt.tris;
                total.insts += T.cnt.insts;
            }
        }
    };
    while (true) {
        // lane numbers by mbcnt: no per-lane mask to keep
        const uint32_t lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        const uint64_t idle = ~live;
        const uint32_t nidle = (uint32_t)__popcll(idle);
        if ((res_n > 0u || more) && (nidle >= refill || nidle == 64u)) {
            bool fresh = false;
            TRay r;  // the ray this lane fetches, if any
            r.o = r.d = mk(0.0f, 0.0f, 0.0f);
            r.tmin = 0.001f;
            r.tmax = 0.0f;
            r.root = kEmptyItem;
            r.alpha_seed = r.payload = 0u;
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
            const bool wants = lane_in(idle);
            uint32_t got = 0;
            while (got < nidle && (res_n > 0u || more)) {
                if (res_n == 0u) {
                    if (seen == ~0u) {  // lane c < 8 looks at chunk c
                        const uint32_t c = lane & 7u;
                        const uint32_t len = (uint32_t)(chunk_begin(n, c + 1u) - chunk_begin(n, c));
                        const unsigned long long taken =
                            __hip_atomic_load(&ctr[c * kChunkStride], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        const uint32_t open = (uint32_t)__ballot(taken < len) & 0xffu;
                        if (open == 0u) {
                            more = false;
                            break;
                        }
                        // the first open chunk from this one on
                        const uint32_t turned = ((open | (open << 8)) >> chunk) & 0xffu;
                        chunk = (chunk + (uint32_t)__ffs((int)turned) - 1u) & 7u;
                        seen = (uint32_t)__builtin_amdgcn_readlane((int)min(taken, (unsigned long long)len), (int)chunk);
                    }
                    const uint64_t c0 = chunk_begin(n, chunk);
                    const uint32_t len = (uint32_t)(chunk_begin(n, chunk + 1u) - c0);
                    const uint32_t left = len - min(seen, len);
                    const uint32_t take = min(min(most, grab), max(kGrabMin, left / max(waves / 4u, 1u)));
                    unsigned long long base = 0;
                    if (lane == 0u) base = atomicAdd(&ctr[chunk * kChunkStride], (unsigned long long)take);
                    base = (unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)base) |
                           ((unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(base >> 32)) << 32);
                    if (base < len) {
                        res_q = (uint32_t)(c0 + base);
                        res_n = min(take, len - (uint32_t)base);
                        seen = (uint32_t)base + res_n;
                    }
                    if (base + take >= len) seen = ~0u;  // used up: look at the others
                    continue;
                }
                const uint32_t take = min(nidle - got, res_n);
                if (wants && rank >= got && rank < got + take) {
                    load(res_q + (rank - got), r);
                    fresh = true;
                }
                got += take;
                res_q += take;
                res_n -= take;
            }
            if (__ballot(fresh) != 0ull) {  // wave-uniform
                T.start(fresh, r, r.root, use_alpha);
                payload = fresh ? r.payload : payload;
                // An empty t range (tmax < tmin, or NaN) or an environment
                // without instances has nothing to trace: finish it at once
                // as a miss.
                const bool empty = fresh && (!(r.tmin <= r.tmax) || r.root == kEmptyItem);
                if (empty) store(r.payload, T.result(), false);
                live |= lanes_of(fresh) & ~lanes_of(empty);
            }
        }
        if (!more && res_n == 0u && live == 0u) break;
        // The step runs even when no lane holds a query (idle lanes fetch
        // nothing): a path that skipped it would make every step pay for
        // merging the two paths' registers, and the refill state lives only
        // in its branch.
        finish(T.step(TS, stk, overflow, live));
    }
}

}  // namespace kf
