// Device-side traversal routines shared by the ray-cast kernels and the wavefront stages.
// See traverse.hip for the reference behaviour they restate.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "rgpu_traverse.h"
#include "rgpu_types.h"

namespace rgpu {

struct F3 {
    float x, y, z;
};
__device__ __forceinline__ F3 f3(float x, float y, float z) { return F3{x, y, z}; }
__device__ __forceinline__ F3 sub3(F3 a, F3 b) { return F3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ float dot3(F3 a, F3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ F3 cross3(F3 a, F3 b) {
    return F3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// One axis of the slab test: entry/exit parameters with the NaN substitution of
// kernels/slab.cl:15-16 (t0 first, then t1 from the updated t0). kPlain leaves the
// substitution out; callers choose it only where neither product can be NaN, so both forms
// give the same bits there.
template <bool kPlain = false>
__device__ __forceinline__ void slab_axis(float lo, float hi, float o, float inv, float* tn, float* tf) {
    float t0 = (lo - o) * inv;
    float t1 = (hi - o) * inv;
    if (!kPlain) {
        t0 = __builtin_isnan(t0) ? -t1 : t0;
        t1 = __builtin_isnan(t1) ? -t0 : t1;
    }
    *tn = fminf(t0, t1);
    *tf = fmaxf(t0, t1);
}

// An inverse direction whose components are all non-zero, not all infinite, with a finite origin:
// the products of an infinite one (the ray does not move along that axis) are NaN where a plane
// holds the origin, and the axis then excludes nothing.
__device__ __forceinline__ bool flat_slabs(F3 o, F3 inv) {
    const bool fo = __builtin_isfinite(o.x) && __builtin_isfinite(o.y) && __builtin_isfinite(o.z);
    const bool numbers = inv.x == inv.x && inv.y == inv.y && inv.z == inv.z;
    const bool nonzero = inv.x != 0.0f && inv.y != 0.0f && inv.z != 0.0f;
    const bool moves = __builtin_isfinite(inv.x) || __builtin_isfinite(inv.y) || __builtin_isfinite(inv.z);
    return fo && numbers && nonzero && moves;
}

// (plane - o) * inv is never NaN when the planes and the origin are finite and every inverse
// direction component is finite and non-zero: a finite or overflowed difference times a finite
// non-zero factor. Then the NaN substitution of the slab test never fires. boxes_finite is a
// property of the scene (all node boxes finite).
__device__ __forceinline__ bool plain_slabs(bool boxes_finite, F3 o, F3 inv) {
    const bool fo = __builtin_isfinite(o.x) && __builtin_isfinite(o.y) && __builtin_isfinite(o.z);
    const bool fi = __builtin_isfinite(inv.x) && __builtin_isfinite(inv.y) && __builtin_isfinite(inv.z) &&
                    inv.x != 0.0f && inv.y != 0.0f && inv.z != 0.0f;
    return boxes_finite && fo && fi;
}

template <bool kPlain = false>
__device__ __forceinline__ bool slab_hit(const float* lo, const float* hi, F3 o, F3 inv, float farclip,
                                         float* h0, float* h1) {
    float nx, fx, ny, fy, nz, fz;
    slab_axis<kPlain>(lo[0], hi[0], o.x, inv.x, &nx, &fx);
    slab_axis<kPlain>(lo[1], hi[1], o.y, inv.y, &ny, &fy);
    slab_axis<kPlain>(lo[2], hi[2], o.z, inv.z, &nz, &fz);
    float rmin = fmaxf(fmaxf(nx, ny), nz);
    float rmax = fminf(fminf(fx, fy), fz);
    *h0 = fmaxf(0.0f, rmin);
    *h1 = fminf(rmax, farclip);
    return rmin <= rmax && 0.0f <= rmax && rmin <= farclip;
}

// One box; the wave takes the plain slab form when every active lane may (a wave-uniform branch,
// so no lane runs both forms).
__device__ __forceinline__ bool slab_one(const float* lo, const float* hi, F3 o, F3 inv, float farclip, bool plain,
                                         float* h0, float* h1) {
    if (__all(plain)) return slab_hit<true>(lo, hi, o, inv, farclip, h0, h1);
    return slab_hit<false>(lo, hi, o, inv, farclip, h0, h1);
}

// Test one primitive record; updates (tmin, u, v, prim) when it is the closest so far.
__device__ __forceinline__ void test_prim(const PrimRec* __restrict__ prims, uint32_t slot, int32_t sphere_begin,
                                          F3 ro, F3 rd, float* tmin, float* uo, float* vo, int32_t* prim) {
    const float4* rec = reinterpret_cast<const float4*>(prims + slot);
    const float4 q0 = rec[0], q1 = rec[1], q2 = rec[2];  // one round trip, whatever the primitive is
    int32_t pid = (int32_t)__float_as_uint(q2.y);
    if (pid < sphere_begin) {
        F3 v0 = f3(q0.x, q0.y, q0.z);
        F3 e1 = f3(q0.w, q1.x, q1.y);
        F3 e2 = f3(q1.z, q1.w, q2.x);
        F3 pvec = cross3(rd, e2);
        float det = dot3(e1, pvec);
        if (fabsf(det) < 1.0e-8f) return;
        float invDet = 1.0f / det;
        F3 tvec = sub3(ro, v0);
        float u = dot3(tvec, pvec) * invDet;
        if (u < 0.0f || u > 1.0f) return;
        F3 qvec = cross3(tvec, e1);
        float v = dot3(rd, qvec) * invDet;
        if (v < 0.0f || u + v > 1.0f) return;
        float t = dot3(e2, qvec) * invDet;
        if (t < 0.0f) return;
        if (*tmin < t) return;
        *tmin = t;
        *uo = u;
        *vo = v;
        *prim = pid;
    } else {
        // kernels/extension_ray_cast_stackless.cl:52-76
        F3 c = f3(q0.x, q0.y, q0.z);
        float r = q0.w;
        float r_sq = r * r;
        F3 S = sub3(ro, c);
        F3 crs = cross3(S, rd);
        float d_sq = dot3(crs, crs);
        float B = dot3(S, rd);
        float D = r_sq - d_sq;
        if (D < 0.0f) return;
        float Ds = __builtin_sqrtf(D);
        float t0 = -B - Ds;
        float t1 = -B + Ds;
        if (0.0f < t0 && t0 < *tmin) {
            *tmin = t0;
            *prim = pid;
            return;
        }
        if (0.0f < t1 && t1 < *tmin) {
            *tmin = t1;
            *prim = pid;
        }
    }
}

// Per-ray traversal event counts (the instrumented kernels only).
struct Cnt {
    uint32_t branch = 0, leaf = 0, parent = 0, prim = 0, node = 0;
    // The parents the reference's backtrack climbs (kernels/extension_ray_cast_stackless.cl:181-196),
    // one per zero bit below its bitstack's lowest set bit, from a bitstack kept alongside the
    // walk: a descent shifts it up and sets the bit where a far child is deferred.
    uint64_t bits = 0;
    __device__ __forceinline__ void step(bool descend, bool defer) {
        if (descend) {
            bits = bits << 1 | (defer ? 1u : 0u);
        } else if (bits != 0) {
            const uint32_t z = (uint32_t)__builtin_ctzll(bits);
            parent += z;
            bits = (bits >> z) ^ 1u;
        }
    }
};

// Ray-direction class of kernels/extension_ray_cast.cl:45-58.
__device__ __forceinline__ uint32_t direction_class(F3 rd) {
    float ax = fabsf(rd.x), ay = fabsf(rd.y), az = fabsf(rd.z);
    float maxYZ = fmaxf(ay, az);
    float maxXZ = fmaxf(ax, az);
    if (maxYZ < ax) return 0.0f < rd.x ? 0u : 1u;
    if (maxXZ < ay) return 0.0f < rd.y ? 2u : 3u;
    return 0.0f < rd.z ? 4u : 5u;
}

// The table a ray walks: its direction class for the multi-threaded BVH, the single table
// otherwise (common/threaded_bvh.hpp:527-547, 366-395).
template <int kVariant>
__device__ __forceinline__ const MTNode* threaded_table(const MTNode* tables, uint32_t nnodes, F3 rd) {
    const uint32_t order = kVariant == kVariantSingleThreaded ? (uint32_t)kMTSingleOrder : direction_class(rd);
    return tables + (size_t)order * nnodes;
}

// Threaded traversal of one ray (common/threaded_bvh.hpp:527-569, 366-395).
template <bool kCount, int kVariant>
__device__ __forceinline__ int32_t trace_threaded(const MTNode* __restrict__ tables, uint32_t nnodes,
                                                  const PrimRec* __restrict__ prims, int32_t sphere_begin,
                                                  bool boxes_finite, F3 ro, F3 rd, float* tmin_io, float* uo,
                                                  float* vo, Cnt* cnt) {
    const MTNode* tab = threaded_table<kVariant>(tables, nnodes, rd);
    const F3 inv = f3(1.0f / rd.x, 1.0f / rd.y, 1.0f / rd.z);
    const bool plain = plain_slabs(boxes_finite, ro, inv);
    float tmin = *tmin_io;
    float u = 0.0f, v = 0.0f;
    int32_t prim = -1;
    uint32_t node = 0;
    while (node != kInvalid) {
        const float4* rec = reinterpret_cast<const float4*>(tab + node);
        float4 q0 = rec[0], q1 = rec[1];
        float lo[3] = {q0.x, q0.y, q0.z}, hi[3] = {q0.w, q1.x, q1.y};
        uint32_t miss = __float_as_uint(q1.z), leaf = __float_as_uint(q1.w);
        float h0, h1;
        if (kCount) cnt->node++;
        bool hit = slab_one(lo, hi, ro, inv, tmin, plain, &h0, &h1);
        if (hit && leaf != 0) {
            const uint32_t beg = leaf & 0x0FFFFFFFu;
            const uint32_t end = beg + ((leaf >> 28) & 7u) + 1u;
            if (kCount) cnt->prim += end - beg;
            for (uint32_t s = beg; s < end; ++s) test_prim(prims, s, sphere_begin, ro, rd, &tmin, &u, &v, &prim);
        }
        node = (hit && leaf == 0) ? node + 1 : miss;
    }
    *tmin_io = tmin;
    *uo = u;
    *vo = v;
    return prim;
}

// ---------------------------------------------------------------- resumable traversal
// The same two traversals cut into single steps over explicit per-lane state, so that a lane
// whose ray has finished can take the next ray while the rest of its wave keeps going. Each
// ray still visits nodes and tests primitives in exactly the order above.

struct ThreadedRay {
    const MTNode* tab;
    F3 ro, rd, inv;
    float tmin, u, v;
    int32_t prim;
    bool plain;     // origin and inverse direction allow the plain slab form (set once per ray)
    uint32_t node;  // kInvalid when finished
    uint32_t leaf;  // primitive word of an entered leaf not yet tested (0: none)
};

template <int kVariant>
__device__ __forceinline__ void threaded_begin(ThreadedRay& r, const MTNode* tables, uint32_t nnodes, F3 ro, F3 rd,
                                               float tmax) {
    r.tab = threaded_table<kVariant>(tables, nnodes, rd);
    r.ro = ro;
    r.rd = rd;
    r.inv = f3(1.0f / rd.x, 1.0f / rd.y, 1.0f / rd.z);
    r.plain = plain_slabs(true, ro, r.inv);
    r.tmin = tmax;
    r.u = r.v = 0.0f;
    r.prim = -1;
    r.node = 0;
    r.leaf = 0;
}

// Box test of the current node of trace_threaded: a branch moves on (hit: next record, miss:
// miss link); an entered leaf is marked pending with its primitive word kept in r.leaf.
__device__ __forceinline__ void threaded_visit(ThreadedRay& r, bool boxes_finite) {
    const float4* rec = reinterpret_cast<const float4*>(r.tab + r.node);
    float4 q0 = rec[0], q1 = rec[1];
    float lo[3] = {q0.x, q0.y, q0.z}, hi[3] = {q0.w, q1.x, q1.y};
    uint32_t miss = __float_as_uint(q1.z), leaf = __float_as_uint(q1.w);
    float h0, h1;
    bool hit = slab_one(lo, hi, r.ro, r.inv, r.tmin, boxes_finite && r.plain, &h0, &h1);
    if (hit && leaf != 0) r.leaf = leaf;  // the miss link is where the walk goes on afterwards
    r.node = (hit && leaf == 0) ? r.node + 1 : miss;
}

// The pending leaf of a lane: its primitives; the walk goes on at the miss link already in node.
__device__ __forceinline__ void threaded_leaf(ThreadedRay& r, const PrimRec* __restrict__ prims, int32_t sphere_begin) {
    const uint32_t beg = r.leaf & 0x0FFFFFFFu;
    const uint32_t end = beg + ((r.leaf >> 28) & 7u) + 1u;
    for (uint32_t s = beg; s < end; ++s) test_prim(prims, s, sphere_begin, r.ro, r.rd, &r.tmin, &r.u, &r.v, &r.prim);
    r.leaf = 0;
}


// ---------------------------------------------------------------- stackless walk
// One ray's walk over the walk records (rgpu_types.h: WalkNode). `node` is the link in hand: a
// record's (>= 0 as a signed word), an entered leaf's primitive word (negative) or kInvalid once
// the walk has ended. What is still to visit sits on a stack: the newest link in `tos`, the next
// kWalkStackLds - 1 in the lane's column of the workgroup's LDS, deeper ones in private memory.
//
// The walk enters the leaves that the reference's binary walk enters, in its order
// (kernels/extension_ray_cast_stackless.cl:81-200), with the same far clip at each:
//  - a record holds the four boxes two levels down, and a node's box is the union of its
//    children's. With finite, ordered boxes and a finite origin the slab products are monotone
//    in the planes, rounding included, so the two children's entry and exit per axis are the
//    minimum and maximum of the grandchildren's: one visit makes the decisions of a node and of
//    the child that is entered next, and no leaf lies between them;
//  - a child none of whose children is hit contributes nothing and is skipped;
//  - the farther child is deferred as a half record and its two boxes are tested again when it
//    is popped, with the far clip of that moment. Where one of them was hit and that one is a
//    branch, its record is deferred directly: if the shrunk clip excludes its box, it excludes
//    the boxes inside it.
// A wave with a ray or a scene that breaks the premise takes the binary visits one by one.
//
// Measured on 4.19 M incoherent rays over 1.3M triangles (persistent kernel): one 64-byte record
// per binary node, leaves included, walked with a bitstack, a six-register short stack and parent
// climbs took 1.12-1.16 ms: 25.1 dependent visits a ray, 8,478 VALU operations per 64 rays (84 %
// busy at 38 % of the lanes) and 5.6 GB from beyond the L2. Links that need no decoding (a branch
// link is the record's 16-byte index, a leaf link the primitive range itself) and a stack whose
// push and pop are one LDS access: 1.00 ms. One 128-byte line for two levels, none for leaves:
// 0.77 ms, 13.5 visits a ray, 5,800 VALU operations (76 % busy at 48 %), 3.4 GB (4.4 TB/s). Both
// bounds are near; 8 waves per SIMD fetch more from beyond the L2 and are slower.
struct StacklessRay {
    F3 ro, rd, inv;
    float tmin, u, v;
    int32_t prim;
    bool plain, flat;  // the visits the ray allows (visit_kind, set once per ray)
    uint32_t node;
    uint32_t tos;   // newest deferred link; kInvalid when nothing is deferred
    int32_t sp;     // LDS byte of the stack's next free entry (past the end: in private memory)
};

// Where a lane's stack lives: entry k of a lane is the word at byte `base` + 256 * k + 4 * lane of
// the kernel's dynamic LDS, the lanes of a wave next to each other (no bank conflicts whatever
// their depths).
struct WalkStack {
    char* lds;
    uint32_t* spill;  // kWalkStackSpill private words
    int32_t base;     // wave-uniform
    __device__ __forceinline__ int32_t end() const { return base + 256 * (int32_t)kWalkStackLds; }
    __device__ __forceinline__ int32_t first() const { return base + 4 * (int32_t)(threadIdx.x & 63); }
    __device__ __forceinline__ uint32_t& entry(int32_t sp) const { return *reinterpret_cast<uint32_t*>(lds + sp); }
    __device__ __forceinline__ void push(StacklessRay& r, uint32_t link) const {
        if (__builtin_expect(r.sp < end(), 1)) entry(r.sp) = r.tos;
        else spill[(uint32_t)(r.sp - end()) >> 8] = r.tos;
        r.sp += 256;
        r.tos = link;
    }
    // Into r.node; kInvalid from an empty stack (the entry below the first push holds it). The
    // LDS read is unconditional, so that it stays an LDS read.
    __device__ __forceinline__ void pop(StacklessRay& r) const {
        r.node = r.tos;
        r.sp = max(r.sp - 256, base);
        r.tos = entry(min(r.sp, end() - 4));
        if (__builtin_expect(r.sp >= end(), 0)) r.tos = spill[(uint32_t)(r.sp - end()) >> 8];
    }
};

// A value that is the same in every lane, as a scalar (branches on it need no lane masks).
__device__ __forceinline__ int32_t wave_scalar(int32_t x) { return __builtin_amdgcn_readfirstlane(x); }

// The kernel's dynamic LDS: `top` walk records (the top levels of the tree, numbered breadth-first
// by the scene packer) without their padding, then kWalkStackLds words per lane, wave by wave.
// Seven 16-byte words a record: an odd stride spreads the lanes' records over the banks.
extern __shared__ float4 walk_lds[];

__device__ __forceinline__ WalkStack walk_stack(uint32_t top, uint32_t* spill) {
    const uint32_t wave = (uint32_t)wave_scalar((int32_t)(threadIdx.x >> 6));
    return WalkStack{reinterpret_cast<char*>(walk_lds), spill,
                     (int32_t)(kStagedBytes * top + wave * (256u * kWalkStackLds))};
}

__device__ __forceinline__ void stackless_begin(StacklessRay& r, const WalkStack& stk, uint32_t root, F3 ro, F3 rd,
                                                float tmax) {
    r.ro = ro;
    r.rd = rd;
    r.inv = f3(1.0f / rd.x, 1.0f / rd.y, 1.0f / rd.z);
    r.plain = plain_slabs(true, ro, r.inv) && tmax >= 0.0f;
    r.flat = flat_slabs(ro, r.inv) && tmax >= 0.0f;
    r.tmin = tmax;
    r.u = r.v = 0.0f;
    r.prim = -1;
    r.node = root;
    r.tos = kInvalid;
    r.sp = stk.first();
}

// How the rays of a wave may visit records (a scalar): kVisitPlain when no slab product can be
// NaN, kVisitFlat when only those of an axis the ray does not move along can (a zero direction
// component), both with a far clip that is a number >= 0 and a scene of finite, ordered boxes;
// otherwise kVisitBinary. A primitive test may accept a t that is NaN (of overflowed products):
// no box passes that clip, which only the binary visit's comparisons tell.
enum { kVisitBinary = 0, kVisitFlat = 1, kVisitPlain = 2 };
__device__ __forceinline__ int32_t visit_kind(const StacklessRay& r, bool boxes_finite) {
    const bool dead = r.node == kInvalid, ok = boxes_finite && r.tmin == r.tmin;
    const int32_t kind = __all(dead || (ok && r.plain))                ? kVisitPlain
                         : __all(dead || (ok && (r.plain || r.flat))) ? kVisitFlat
                                                                       : kVisitBinary;
    return wave_scalar(kind);
}
// The same after primitive tests, which only change clips.
__device__ __forceinline__ int32_t visit_kind_after(int32_t kind, const StacklessRay& r) {
    return __all(r.tmin == r.tmin) ? kind : (int32_t)kVisitBinary;
}

// Stages the first `top` records at the start of walk_lds (the whole workgroup; barrier after).
__device__ __forceinline__ void stage_records(const float4* __restrict__ recs, uint32_t top) {
    for (uint32_t j = threadIdx.x; j < 7u * top; j += blockDim.x) walk_lds[j] = recs[8u * (j / 7u) + j % 7u];
    __syncthreads();
}

// The two places of a record, kept apart by address space: as generic pointers the compiler
// joins the two reads into flat loads, which go to both memories.
#define LdsSpace __attribute__((address_space(3)))
#define GlobalSpace __attribute__((address_space(1)))
typedef float WalkWords __attribute__((ext_vector_type(4)));
typedef uint32_t WalkLinks __attribute__((ext_vector_type(4)));

// Entry and exit parameters of a box before the clip: the slab test is
// in <= out && 0 <= out && in <= far clip, its entry distance max(0, in), its exit min(out, clip).
struct Slab {
    float in, out;
    __device__ __forceinline__ bool hit(float farclip) const {
        return in <= out && 0.0f <= out && in <= farclip;
    }
};
// The clipped interval [max(0, in), min(out, clip)]. Where the clip is not below 0 (nor NaN) and
// in and out are numbers, it is non-empty exactly when the slab test passes.
struct Span {
    float enter, leave;
    __device__ __forceinline__ bool hit() const { return enter <= leave; }
};
__device__ __forceinline__ Span clipped(const Slab& s, float farclip) {
    return Span{fmaxf(0.0f, s.in), fminf(s.out, farclip)};
}
// Whether box a is the nearer of two entered ones: by entry, then by exit; of boxes that tie in
// both, b.
__device__ __forceinline__ bool nearer(const Span& a, const Span& b) {
    const bool before = a.enter < b.enter, level = a.enter == b.enter, shorter = a.leave < b.leave;
    return before | (level & shorter);
}
struct BoxPlanes {
    float lo[3], hi[3];
};
struct BoxSlabs {
    float n[3], f[3];
    __device__ __forceinline__ Slab clip() const {
        return Slab{fmaxf(fmaxf(n[0], n[1]), n[2]), fminf(fminf(f[0], f[1]), f[2])};
    }
};
// kVisitFlat: a box that a plane of an axis without motion touches spans that axis, as the
// reference's substitution makes it; a box of no extent there, whose products are both NaN, is
// given the same span (the reference's minima and maxima ignore the axis), so that unions of
// intervals stay intervals of unions.
template <int kKind>
__device__ __forceinline__ BoxSlabs box_slabs(const BoxPlanes& b, F3 o, F3 inv) {
    BoxSlabs s;
    const float oo[3] = {o.x, o.y, o.z}, ii[3] = {inv.x, inv.y, inv.z};
    for (int k = 0; k < 3; ++k) {
        if (kKind == kVisitFlat) {
            const float t0 = (b.lo[k] - oo[k]) * ii[k], t1 = (b.hi[k] - oo[k]) * ii[k];
            const bool touch = __builtin_isunordered(t0, t1);
            s.n[k] = touch ? -__builtin_inff() : fminf(t0, t1);
            s.f[k] = touch ? __builtin_inff() : fmaxf(t0, t1);
        } else {
            slab_axis<kKind == kVisitPlain>(b.lo[k], b.hi[k], oo[k], ii[k], &s.n[k], &s.f[k]);
        }
    }
    return s;
}
__device__ __forceinline__ BoxSlabs join(const BoxSlabs& a, const BoxSlabs& b) {
    BoxSlabs s;
    for (int k = 0; k < 3; ++k) {
        s.n[k] = fminf(a.n[k], b.n[k]);
        s.f[k] = fmaxf(a.f[k], b.f[k]);
    }
    return s;
}
__device__ __forceinline__ BoxPlanes join(const BoxPlanes& a, const BoxPlanes& b) {
    BoxPlanes s;
    for (int k = 0; k < 3; ++k) {
        s.lo[k] = fminf(a.lo[k], b.lo[k]);
        s.hi[k] = fmaxf(a.hi[k], b.hi[k]);
    }
    return s;
}

struct WalkRecord {
    BoxPlanes box[4];
    WalkLinks link;
};
// kTop: records below link `top8` (8 * records) come from LDS.
template <bool kTop>
__device__ __forceinline__ void load_record(uint32_t at, const float4* __restrict__ recs, uint32_t top8, WalkRecord* r) {
    WalkWords q[6];
    if (kTop && at < top8) {
        const auto* p = (const LdsSpace WalkWords*)((const LdsSpace char*)walk_lds + __umul24(at, kStagedBytes / 8u));
        for (int k = 0; k < 6; ++k) q[k] = p[k];
        r->link = *(const LdsSpace WalkLinks*)(p + 6);
    } else {
        const auto* p = (const GlobalSpace WalkWords*)recs + at;
        for (int k = 0; k < 6; ++k) q[k] = p[k];
        r->link = *(const GlobalSpace WalkLinks*)(p + 6);
    }
    for (int h = 0; h < 2; ++h) {
        const WalkWords a = q[3 * h], b = q[3 * h + 1], c = q[3 * h + 2];
        r->box[2 * h] = BoxPlanes{{a.x, a.y, a.z}, {a.w, b.x, b.y}};
        r->box[2 * h + 1] = BoxPlanes{{b.z, b.w, c.x}, {c.y, c.z, c.w}};
    }
}

// Visit of the record `node` names: descent two levels down, what else is hit deferred, or a pop
// when nothing is hit. kKind: kVisitPlain or kVisitFlat.
template <bool kTop, int kKind>
__device__ __forceinline__ void stackless_visit(StacklessRay& r, const WalkStack& stk, const float4* __restrict__ recs,
                                                uint32_t top8) {
    uint32_t at = r.node & ~7u;
    const uint32_t only = r.node & 7u;  // kFirstHalf, kSecondHalf or 0
    // (an opaque, different start keeps the compiler from joining the two kinds' common part,
    // which would hold all 24 products of a record in registers)
    if (kKind == kVisitPlain) asm("; plain visit" : "+v"(at));
    else asm("; flat visit" : "+v"(at));
    WalkRecord w;
    load_record<kTop>(at, recs, top8, &w);
    const BoxSlabs s0 = box_slabs<kKind>(w.box[0], r.ro, r.inv), s1 = box_slabs<kKind>(w.box[1], r.ro, r.inv);
    const Span c0 = clipped(s0.clip(), r.tmin), c1 = clipped(s1.clip(), r.tmin);
    const Span L = clipped(join(s0, s1).clip(), r.tmin);
    const BoxSlabs s2 = box_slabs<kKind>(w.box[2], r.ro, r.inv), s3 = box_slabs<kKind>(w.box[3], r.ro, r.inv);
    const Span c2 = clipped(s2.clip(), r.tmin), c3 = clipped(s3.clip(), r.tmin);
    const Span R = clipped(join(s2, s3).clip(), r.tmin);
    // (a leaf child's second box is its first again, so it changes neither union nor these)
    const bool aliveL = (c0.hit() || c1.hit()) && only != kSecondHalf;
    const bool aliveR = (c2.hit() || c3.hit()) && only != kFirstHalf;
    const bool takeL = aliveL && (nearer(L, R) || !aliveR);
    if (aliveL && aliveR) {
        // the other half: as a half of this record; directly where that is exact (a leaf child of
        // the node itself, whose second link is empty, or a single branch child hit)
        const uint32_t oa = takeL ? w.link.z : w.link.x, ob = takeL ? w.link.w : w.link.y;
        const Span ga{takeL ? c2.enter : c0.enter, takeL ? c2.leave : c0.leave};
        const Span gb{takeL ? c3.enter : c1.enter, takeL ? c3.leave : c1.leave};
        const uint32_t one = ga.hit() ? oa : ob;
        const bool both = ga.hit() && gb.hit();
        const bool direct = ob == kInvalid || (!both && (int32_t)one >= 0);
        stk.push(r, direct ? one : (at | (takeL ? kSecondHalf : kFirstHalf)));
    }
    if (aliveL || aliveR) {
        // the entered half: its children a and b
        const Span a{takeL ? c0.enter : c2.enter, takeL ? c0.leave : c2.leave};
        const Span b{takeL ? c1.enter : c3.enter, takeL ? c1.leave : c3.leave};
        const uint32_t la = takeL ? w.link.x : w.link.z, lb = takeL ? w.link.y : w.link.w;
        const bool ha = a.hit(), hb = b.hit() && lb != kInvalid;
        const bool takeA = ha && (nearer(a, b) || !hb);
        r.node = takeA ? la : lb;
        if (ha && hb) stk.push(r, takeA ? lb : la);
    } else {
        stk.pop(r);
    }
}

// The same walk one binary node at a time, as the reference visits them: a record's node itself
// first (its two children, boxed by the unions of the records' boxes), then each entered half.
// For waves that no other kind fits, and for the event counts.
template <bool kTop, bool kCount>
__device__ __forceinline__ void stackless_visit_binary(StacklessRay& r, const WalkStack& stk,
                                                       const float4* __restrict__ recs, uint32_t top8, Cnt* cnt) {
    const uint32_t at = r.node & ~7u, only = r.node & 7u;
    WalkRecord w;
    load_record<kTop>(at, recs, top8, &w);
    BoxPlanes A, B;
    uint32_t la, lb;
    if (only == 0) {
        A = join(w.box[0], w.box[1]);
        B = join(w.box[2], w.box[3]);
        // a leaf child of the node is entered by its word
        la = w.link.y == kInvalid ? w.link.x : at | kFirstHalf;
        lb = w.link.w == kInvalid ? w.link.z : at | kSecondHalf;
    } else {
        const bool first = only == kFirstHalf;
        A = first ? w.box[0] : w.box[2];
        B = first ? w.box[1] : w.box[3];
        la = first ? w.link.x : w.link.z;
        lb = first ? w.link.y : w.link.w;
    }
    const Slab a = box_slabs<kVisitBinary>(A, r.ro, r.inv).clip(), b = box_slabs<kVisitBinary>(B, r.ro, r.inv).clip();
    const bool ha = a.hit(r.tmin), hb = b.hit(r.tmin);
    const bool takeA = ha && (!hb || nearer(clipped(a, r.tmin), clipped(b, r.tmin)));
    if (kCount) {
        cnt->branch++;
        cnt->step(ha || hb, ha && hb);
    }
    r.node = takeA ? la : lb;
    if (ha && hb) stk.push(r, takeA ? lb : la);
    if (!(ha || hb)) stk.pop(r);
}

template <bool kTop, bool kCount>
__device__ __forceinline__ void stackless_visit_as(int32_t kind, StacklessRay& r, const WalkStack& stk,
                                                   const float4* __restrict__ recs, uint32_t top, Cnt* cnt) {
    if (!kCount && kind == kVisitPlain) stackless_visit<kTop, kVisitPlain>(r, stk, recs, 8 * top);
    else if (!kCount && kind == kVisitFlat) stackless_visit<kTop, kVisitFlat>(r, stk, recs, 8 * top);
    else stackless_visit_binary<kTop, kCount>(r, stk, recs, 8 * top, cnt);
}

// The primitives of an entered leaf, then the pop.
template <bool kCount>
__device__ __forceinline__ void stackless_leaf(StacklessRay& r, const WalkStack& stk,
                                               const PrimRec* __restrict__ prims, int32_t sphere_begin, Cnt* cnt) {
    const uint32_t beg = r.node & 0x0FFFFFFFu;
    const uint32_t end = beg + ((r.node >> 28) & 7u) + 1u;
    if (kCount) {
        cnt->leaf++;
        cnt->prim += end - beg;
    }
    for (uint32_t s = beg; s < end; ++s) test_prim(prims, s, sphere_begin, r.ro, r.rd, &r.tmin, &r.u, &r.v, &r.prim);
    stk.pop(r);
    if (kCount) cnt->step(false, false);
}

// Lane states of the resumable walks: live (a ray in progress), pending (stopped at an entered
// leaf whose primitives are not yet tested), walking (at a record to visit).
__device__ __forceinline__ bool walk_live(const StacklessRay& r) { return r.node != kInvalid; }
__device__ __forceinline__ bool walk_pending(const StacklessRay& r) { return (int32_t)r.node < -1; }
__device__ __forceinline__ bool walk_walking(const StacklessRay& r) { return (int32_t)r.node >= 0; }
__device__ __forceinline__ bool walk_live(const ThreadedRay& r) { return r.node != kInvalid || r.leaf != 0; }
__device__ __forceinline__ bool walk_pending(const ThreadedRay& r) { return r.leaf != 0; }
__device__ __forceinline__ bool walk_walking(const ThreadedRay& r) { return r.node != kInvalid && r.leaf == 0; }

__device__ __forceinline__ uint32_t count_lanes(bool b) { return (uint32_t)__popcll(__ballot(b)); }

// One ray per lane with leaves batched across the wave: a lane that enters a leaf waits until
// leaf_batch lanes wait, or at least as many lanes wait as still walk, then the wave tests their
// primitives together. The lane's own visits and tests are those of the one-ray walk.
// Lanes whose ray has ended stay in the loop, masked, until the wave is done.
// kTop: the kernel has staged the first `top` walk records in LDS (before the stacks).
template <int kVariant, bool kTop = false, bool kCount = false>
__device__ __forceinline__ int32_t trace_batched(const TraceScene& sc, F3 ro, F3 rd, float* tmin_io, float* uo,
                                                 float* vo, uint32_t leaf_batch, uint32_t top = 0,
                                                 Cnt* cnt = nullptr) {
    if constexpr (kVariant == kVariantStackless) {
        uint32_t spill[kWalkStackSpill];
        const WalkStack stk = walk_stack(top, spill);
        const float4* recs = reinterpret_cast<const float4*>(sc.walk_nodes);
        StacklessRay st;
        stackless_begin(st, stk, sc.root, ro, rd, *tmin_io);
        int32_t kind = visit_kind(st, sc.boxes_finite != 0);
        for (;;) {
            const uint32_t nwalk = count_lanes(walk_walking(st)), npending = count_lanes(walk_pending(st));
            if (nwalk + npending == 0) break;
            if (npending >= leaf_batch || npending >= nwalk) {
                if (walk_pending(st)) stackless_leaf<kCount>(st, stk, sc.prims, sc.sphere_begin, cnt);
                kind = visit_kind_after(kind, st);
            } else if (walk_walking(st)) {
                stackless_visit_as<kTop, kCount>(kind, st, stk, recs, top, cnt);
            }
        }
        *tmin_io = st.tmin;
        *uo = st.u;
        *vo = st.v;
        return st.prim;
    } else {
        ThreadedRay st;
        threaded_begin<kVariant>(st, sc.mt_nodes, sc.nnodes, ro, rd, *tmin_io);
        const bool finite = sc.boxes_finite != 0;
        for (;;) {
            if (__ballot(walk_live(st)) == 0) break;
            const bool pending = walk_pending(st);
            const bool walking = walk_walking(st);
            const uint32_t npending = count_lanes(pending);
            if (npending >= leaf_batch || npending >= count_lanes(walking)) {
                if (pending) threaded_leaf(st, sc.prims, sc.sphere_begin);
            } else if (walking) {
                threaded_visit(st, finite);
            }
        }
        *tmin_io = st.tmin;
        *uo = st.u;
        *vo = st.v;
        return st.prim;
    }
}

}  // namespace rgpu
