// bvht_trace.hpp -- the per-lane traversal loops (BLAS and two-level TLAS).
#pragma once

#include "bvht_device.hpp"

namespace bvht {

// LDS (address space 3) pointer, so stack accesses compile to ds_read/ds_write
// instead of flat accesses.
typedef __attribute__((address_space(3))) uint32_t lds_u32;
// 64-bit words of the same memory (may_alias: the two views of a wave's LDS
// follow one another, and their accesses must not be reordered)
typedef __attribute__((address_space(3), may_alias)) uint64_t lds_u64;

// 64 bytes at a wave-uniform, 4-byte aligned address, loaded once for the
// wave through the scalar data cache into 16 SGPRs.  The wait is inside the
// same asm block, so the registers hold the data when the block ends.
typedef int int16v __attribute__((ext_vector_type(16)));
__device__ __forceinline__ int16v scalar_load64(const void* p)
{
    int16v r;
    asm volatile("s_load_dwordx16 %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(r) : "s"(p));
    return r;
}

// Per-lane traversal stack: the first LDS_DEPTH entries live in LDS at
// lds[slot * WG] (lds already offset by the lane: the lanes of a wave hit
// distinct banks), deeper entries in a per-ray column of a global buffer
// (spill[(slot - LDS_DEPTH) * stride]).  `cap` bounds the total; a push beyond
// it is dropped rather than written out of bounds, and sets kStatusStack in
// *status, which the host reports as BVHT_ESTACK at the next fence.  cap comes
// from the tree depth, so only a caller's smaller stack limit (or a wrong
// depth bound) can drop a push.
template <int LDS_DEPTH, int WG>
struct Stack {
    lds_u32* lds;
    uint32_t* spill;
    size_t stride;
    uint32_t cap;
    uint32_t* status;

    __device__ __forceinline__ void push(uint32_t& sp, uint32_t v)
    {
        if (sp < (uint32_t)LDS_DEPTH) {
            lds[sp * WG] = v;
        } else {
            if (sp >= cap) {
                *status = 1u;  // kStatusStack
                return;
            }
            spill[(size_t)(sp - LDS_DEPTH) * stride] = v;
        }
        ++sp;
    }
    __device__ __forceinline__ uint32_t pop(uint32_t& sp)
    {
        --sp;
        return sp < (uint32_t)LDS_DEPTH ? lds[sp * WG] : spill[(size_t)(sp - LDS_DEPTH) * stride];
    }
};

// Trace kernel configurations: workgroup size x LDS stack entries per lane.
// The X-macro instantiates every kernel variant; the host picks one per
// launch from the context's configuration (set by the autotuner or the
// depth-based default).
#define BVHT_TRACE_CONFIGS(X) \
    X(64, 8) X(64, 16) X(64, 24) X(64, 32) \
    X(128, 8) X(128, 16) X(128, 24) X(128, 32) \
    X(256, 8) X(256, 16) X(256, 24) X(256, 32)

// A BLAS stack entry carries the pushed node's (left_first, count) itself
// when they fit -- bit 31 set, count in bits 25..30, left_first in bits
// 0..24 -- so a pop needs no node fetch; otherwise it is the node index
// (bit 31 clear: node indices stay below 2^31) and the pop reads the node.
// The visiting order is unchanged.
constexpr uint32_t kPackFlag = 0x80000000u;
constexpr uint32_t kPackShift = 25;
constexpr uint32_t kPackMask = (1u << kPackShift) - 1u;

__device__ __forceinline__ uint32_t pack_entry(uint32_t idx, uint32_t lf, uint32_t cnt)
{
    return (cnt < 64u && lf <= kPackMask) ? (kPackFlag | (cnt << kPackShift) | lf) : idx;
}

// Lanes of a wave that must still be descending for the node-pair loop to
// take another step (see traverse_blas).
#ifndef BVHT_DESCEND_MIN
#define BVHT_DESCEND_MIN 24
#endif
constexpr uint32_t kDescendMin = BVHT_DESCEND_MIN;

struct BlasResult {
    float t, u, v;
    uint32_t prim;
    bool found;
};

// cnt value of a lane that has finished its node (both children missed) or
// leaf and pops next.  A leaf's count is below the triangle count, so it
// never takes this value.
constexpr uint32_t kPopNext = 0xFFFFFFFFu;

// Bvh::intersect_subtree (bvh.rs:242-305) for one ray, starting at node 0.
// The stack is shared with an enclosing TLAS traversal: this call only uses
// slots at or above sp_base and leaves the stack as it found it.  PACKED:
// every node of the tree fits a packed stack entry (no leaf of 64 or more
// triangles, left_first below 2^25), so entries are packed without a check.
// FINITE: the ray's t is not above FLT_MAX, so every distance below the
// current nearest hit is below FLT_MAX and the child choice reduces to
// comparisons of slab_key values (same decisions as the general form).
template <bool STATS, bool PACKED, bool FINITE = false, class StackT>
__device__ __forceinline__ BlasResult traverse_blas(const float4* __restrict__ nodes,
                                                    const float* __restrict__ tris, const DRay& ray,
                                                    StackT& st, uint32_t sp_base, uint32_t& pairs,
                                                    uint32_t& tests)
{
    BlasResult res{0.0f, 0.0f, 0.0f, 0u, false};
    float closest = ray.t;
    uint32_t sp = sp_base;
    uint32_t lf = __float_as_uint(nodes[0].w);
    uint32_t cnt = __float_as_uint(nodes[1].w);
    while (true) {
        // Node-pair steps while the lane is at an interior node (cnt == 0).
        // After each step the wave leaves this loop once fewer than
        // kDescendMin of its lanes are still descending, instead of holding
        // the lanes that wait at a leaf or a pop until the longest descent
        // ends; the lanes still descending resume here on the next pass.
        // Every lane's own sequence of node steps, leaf tests and pops is
        // that of the one-loop traversal.
        while (cnt == 0) {
            if (STATS)
                ++pairs;
            float4 a0, a1, b0, b1;
            const uint32_t lf0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)lf);
            if (__builtin_amdgcn_ballot_w64(lf != lf0) == 0) {
                // every descending lane is at the same pair: one scalar load
                // of its 64 bytes, which leaves the vector memory path (the
                // texture address and data units) to the other waves
                const int16v p = scalar_load64(nodes + 2 * (size_t)lf0);
                a0 = make_float4(__int_as_float(p[0]), __int_as_float(p[1]), __int_as_float(p[2]),
                                 __int_as_float(p[3]));
                a1 = make_float4(__int_as_float(p[4]), __int_as_float(p[5]), __int_as_float(p[6]),
                                 __int_as_float(p[7]));
                b0 = make_float4(__int_as_float(p[8]), __int_as_float(p[9]), __int_as_float(p[10]),
                                 __int_as_float(p[11]));
                b1 = make_float4(__int_as_float(p[12]), __int_as_float(p[13]), __int_as_float(p[14]),
                                 __int_as_float(p[15]));
            } else {
                const float4* c = nodes + 2 * (size_t)lf;
                a0 = c[0];
                a1 = c[1];
                b0 = c[2];
                b1 = c[3];
            }
            bool left_near, near_hit, far_hit;
            if (FINITE) {
                float kl = slab_key(a0, a1, ray);
                float kr = slab_key(b0, b1, ray);
                // keys are never NaN, so the nearer and farther key are
                // selects on left_near (fmaxf would add two canonicalizes)
                left_near = kl < kr;
                near_hit = (left_near ? kl : kr) < closest;
                far_hit = (left_near ? kr : kl) < closest;
            } else {
                float dl, dr;
                bool hl = slab(a0, a1, ray, closest, dl);
                bool hr = slab(b0, b1, ray, closest, dr);
                float kl = hl ? dl : kFltMax;
                float kr = hr ? dr : kFltMax;
                left_near = kl < kr;
                near_hit = left_near ? hl : hr;
                far_hit = left_near ? hr : hl;
            }
            if (near_hit) {
                if (far_hit) {
                    uint32_t flf = __float_as_uint(left_near ? b0.w : a0.w);
                    uint32_t fcnt = __float_as_uint(left_near ? b1.w : a1.w);
                    st.push(sp, PACKED ? (kPackFlag | (fcnt << kPackShift) | flf)
                                       : pack_entry(left_near ? lf + 1 : lf, flf, fcnt));
                }
                uint32_t nlf = __float_as_uint(left_near ? a0.w : b0.w);
                cnt = __float_as_uint(left_near ? a1.w : b1.w);
                lf = nlf;
            } else {
                cnt = kPopNext;
            }
            if ((uint32_t)__popcll(__builtin_amdgcn_ballot_w64(cnt == 0)) < kDescendMin)
                break;
        }
        if (cnt != 0 && cnt != kPopNext) {
            for (uint32_t k = 0; k < cnt; ++k) {
                float t, u, v;
                if (STATS)
                    ++tests;
                if (tri_test(tris + 9 * (size_t)(lf + k), ray, t, u, v) && t < closest) {
                    closest = t;
                    res.t = t;
                    res.u = u;
                    res.v = v;
                    res.prim = lf + k;
                    res.found = true;
                }
            }
            cnt = kPopNext;
        }
        if (cnt == kPopNext) {
            if (sp == sp_base)
                break;
            uint32_t e = st.pop(sp);
            if (PACKED || (e & kPackFlag)) {
                lf = e & kPackMask;
                cnt = (e >> kPackShift) & 63u;
            } else {
                lf = __float_as_uint(nodes[2 * (size_t)e].w);
                cnt = __float_as_uint(nodes[2 * (size_t)e + 1].w);
            }
        }
        // One loop latch for every lane: without this convergent point the
        // compiler gives the no-pop path a back edge of its own and nests the
        // loops so that pops wait for every lane of the wave to finish its
        // node or leaf.
        __builtin_amdgcn_wave_barrier();
    }
    if (!(closest < kFltMax))
        res.found = false;
    return res;
}

// Bvh::intersect_subtree with G lanes a ray (4, 8 or 16, aligned), for trees
// with large leaves: every lane of a group holds the same ray and state and
// takes the same node steps, and a leaf's triangles are tested G at a time.
// The nearest accepted triangle, the first of equal ones, is the one the
// sequential loop keeps.  Its t, u and v come from testing it once more at the
// end (the same arithmetic).  `st` is the group's one stack.
template <int G, class StackT>
__device__ __forceinline__ BlasResult traverse_group(const float4* __restrict__ nodes, const float* __restrict__ tris,
                                                     const DRay& ray, StackT& st)
{
    static_assert(G == 4 || G == 8 || G == 16, "groups within a 16-lane row");
    const uint32_t lane = threadIdx.x & 63u, sub = lane & (G - 1);
    float closest = ray.t;
    uint32_t sp = 0, prim = BVHT_MISS;
    uint32_t lf = __float_as_uint(nodes[0].w);
    uint32_t cnt = __float_as_uint(nodes[1].w);
    while (true) {
        while (cnt == 0) {
            const float4* c = nodes + 2 * (size_t)lf;
            const float4 a0 = c[0], a1 = c[1], b0 = c[2], b1 = c[3];
            float dl, dr;
            const bool hl = slab(a0, a1, ray, closest, dl);
            const bool hr = slab(b0, b1, ray, closest, dr);
            const float kl = hl ? dl : kFltMax, kr = hr ? dr : kFltMax;
            const bool left_near = kl < kr;
            if (left_near ? hl : hr) {
                if (left_near ? hr : hl)
                    st.push(sp, left_near ? lf + 1 : lf);
                const uint32_t nlf = __float_as_uint(left_near ? a0.w : b0.w);
                cnt = __float_as_uint(left_near ? a1.w : b1.w);
                lf = nlf;
            } else {
                cnt = kPopNext;
            }
        }
        if (cnt != kPopNext) {
            float bt = closest;
            uint32_t bi = BVHT_MISS;
            for (uint32_t k = sub; k < cnt; k += G) {
                float t, u, v;
                if (tri_test(tris + 9 * (size_t)(lf + k), ray, t, u, v) && t < bt) {
                    bt = t;
                    bi = lf + k;
                }
            }
            auto take = [&](uint32_t ot, uint32_t oi) {
                const float o = __uint_as_float(ot);
                if (o < bt || (o == bt && oi < bi)) {
                    bt = o;
                    bi = oi;
                }
            };
            take(xor_lane<1>(__float_as_uint(bt), lane), xor_lane<1>(bi, lane));
            take(xor_lane<2>(__float_as_uint(bt), lane), xor_lane<2>(bi, lane));
            if constexpr (G >= 8)
                take(xor_lane<4>(__float_as_uint(bt), lane), xor_lane<4>(bi, lane));
            if constexpr (G >= 16)
                take(xor_lane<8>(__float_as_uint(bt), lane), xor_lane<8>(bi, lane));
            if (bi != BVHT_MISS) {
                closest = bt;
                prim = bi;
            }
        }
        if (sp == 0)
            break;
        const uint32_t e = st.pop(sp);
        lf = __float_as_uint(nodes[2 * (size_t)e].w);
        cnt = __float_as_uint(nodes[2 * (size_t)e + 1].w);
    }
    BlasResult res{0.0f, 0.0f, 0.0f, prim, false};
    if (prim != BVHT_MISS && closest < kFltMax)
        res.found = tri_test(tris + 9 * (size_t)prim, ray, res.t, res.u, res.v);
    return res;
}

// ------------------------------------------------------ wide records --
// Two binary levels in one fetch.  For every interior node x at even depth
// the record at wide + 4 * left_first(x) (128 bytes, one L2 line) holds x's up
// to four grandchildren, slots 0 and 1 below the left child and 2 and 3 below
// the right, each {lo.xyz, ref}{hi.xyz, 0} (packed trees only).  A leaf's ref
// is a packed stack entry (kPackFlag | count << kPackShift | left_first), an
// interior node's its left_first.  A child that is a leaf fills its first
// slot; the second has ref kNoRef and a box of NaNs, which nothing hits and
// minima and maxima pass over.  Record 0 belongs to no node (left_first >= 2);
// its first word is 1 when some node breaks what traverse_quad relies on or the
// records are older than the boxes (a refit that did not write them).
constexpr uint32_t kNoRef = 0xFFFFFFFFu;
constexpr uint32_t kPairRef = 1u << 26;  // side (bit 25) of the record in bits 0..24

__device__ __forceinline__ bool same_box(float4 lo, float4 hi, float4 alo, float4 ahi, float4 blo, float4 bhi)
{
    return lo.x == fminf(alo.x, blo.x) && lo.y == fminf(alo.y, blo.y) && lo.z == fminf(alo.z, blo.z) &&
           hi.x == fmaxf(ahi.x, bhi.x) && hi.y == fmaxf(ahi.y, bhi.y) && hi.z == fmaxf(ahi.z, bhi.z);
}
__device__ __forceinline__ bool ordered_box(float4 lo, float4 hi)
{
    return lo.x <= hi.x && lo.y <= hi.y && lo.z <= hi.z;
}

// Writes node k's wide record (nothing for a leaf).  Marks the tree when the
// node's box is not the union of its children's, a child's not the union of
// the grandchildren's, or a box has lo > hi or a NaN (uploaded trees, NaN
// vertices): called for every node at even depth it looks at every box.
__device__ __forceinline__ void write_wide(const float4* __restrict__ nodes, float4* __restrict__ wide, uint32_t k)
{
    const float4 xlo = nodes[2 * (size_t)k], xhi = nodes[2 * (size_t)k + 1];
    if (__float_as_uint(xhi.w) != 0)
        return;
    const uint32_t lf = __float_as_uint(xlo.w);
    const float4* c = nodes + 2 * (size_t)lf;
    float4 lo[4], hi[4];
    uint32_t ref[4];
    const float4 clo[2] = {c[0], c[2]}, chi[2] = {c[1], c[3]};
    bool ok = same_box(xlo, xhi, clo[0], chi[0], clo[1], chi[1]);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const uint32_t cnt = __float_as_uint(chi[s].w), clf = __float_as_uint(clo[s].w);
        if (cnt) {
            const float nan = __uint_as_float(0x7FC00000u);
            lo[2 * s] = clo[s];
            hi[2 * s] = chi[s];
            lo[2 * s + 1] = hi[2 * s + 1] = make_float4(nan, nan, nan, nan);
            ref[2 * s] = kPackFlag | cnt << kPackShift | clf;
            ref[2 * s + 1] = kNoRef;
        } else {
            const float4* g = nodes + 2 * (size_t)clf;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                lo[2 * s + j] = g[2 * j];
                hi[2 * s + j] = g[2 * j + 1];
                const uint32_t n = __float_as_uint(hi[2 * s + j].w), f = __float_as_uint(lo[2 * s + j].w);
                ref[2 * s + j] = n ? kPackFlag | n << kPackShift | f : f;
            }
            ok = ok && same_box(clo[s], chi[s], lo[2 * s], hi[2 * s], lo[2 * s + 1], hi[2 * s + 1]);
        }
        ok = ok && ordered_box(lo[2 * s], hi[2 * s]) && (cnt || ordered_box(lo[2 * s + 1], hi[2 * s + 1]));
    }
    float4* w = wide + 4 * (size_t)lf;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        w[2 * k] = make_float4(lo[k].x, lo[k].y, lo[k].z, __uint_as_float(ref[k]));
        w[2 * k + 1] = make_float4(hi[k].x, hi[k].y, hi[k].z, 0.0f);
    }
    if (!ok)
        *reinterpret_cast<uint32_t*>(wide) = 1u;
}

// Whether the wide records may trace this ray: t not above FLT_MAX, a finite
// origin, and no reciprocal direction that is 0 or NaN (an infinite one, from
// a zero direction component, is allowed).
__device__ __forceinline__ bool wide_ray(const DRay& r)
{
    return !(r.t > kFltMax) && fabsf(r.o.x) <= kFltMax && fabsf(r.o.y) <= kFltMax && fabsf(r.o.z) <= kFltMax &&
           fabsf(r.r.x) > 0.0f && fabsf(r.r.y) > 0.0f && fabsf(r.r.z) > 0.0f;
}
__device__ __forceinline__ bool finite_dir(const DRay& r)
{
    return fabsf(r.r.x) <= kFltMax && fabsf(r.r.y) <= kFltMax && fabsf(r.r.z) <= kFltMax;
}

// traverse_blas with four lanes a ray on the wide records: lane q of a quad
// holds slot q, so a step is one slab test instead of four, and a leaf's
// triangles are tested four at a time.  The same leaves are tested in the same
// order with the same nearest hit, in about half the steps.  Why the hits are
// the same bit for bit:
// - binary32 subtraction and multiplication are monotone and each child's
//   box is the union of its children's, so a child's distance on an axis is
//   the smaller of the grandchildren's, its key is the maximum of those over
//   the axes, and a grandchild is hit only if the child is.  So the child
//   order follows from the grandchildren's boxes, and a child whose
//   grandchildren all miss is entered in vain.
// - An infinite reciprocal and a bound equal to the origin give 0 * inf =
//   NaN, which breaks this: with such a ray in the wave (`degen`) the
//   children's boxes are tested too.
// - The near side's grandchildren are tested now, as in the binary loop.  The
//   far side's are tested in the binary loop when the far child is popped,
//   against the distance found by then: the far side is pushed as a pair
//   (the record and the side) and its half of the record tested at the pop.
// - Each entry has its key and is dropped at the pop when that is not below
//   the nearest hit: every test below it would fail.  A leaf already decided
//   on has key -inf.
// - A leaf's triangles are taken by distance, then by index: the sequential
//   loop's first nearest one.
// All four lanes of a quad hold the same ray and state.  st: this quad's
// column of kQuadSlots {ref, key} entries, 16 apart; a ray that
// needs more stops with `overflow`.
// The child order is worked out on lane masks (a bit a lane, in scalar
// registers): a step's logic then costs the vector units nothing.
constexpr uint32_t kQuadLds = 16;                 // LDS words a lane
constexpr uint32_t kQuadSlots = 2 * kQuadLds;     // entries a ray
constexpr int kQuadStack = 4 * (int)kQuadLds;     // LDS stack entries a ray of the binary loop

constexpr uint64_t kEven = 0x5555555555555555ull, kLow2 = 0x3333333333333333ull;  // lanes q & 1 == 0, q < 2
__device__ __forceinline__ uint64_t lanes_of(bool b) { return __builtin_amdgcn_ballot_w64(b); }
__device__ __forceinline__ bool lane_in(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }
__device__ __forceinline__ uint64_t mask_xor1(uint64_t m) { return (m & kEven) << 1 | (m >> 1 & kEven); }
// Orders a wave's LDS accesses for the compiler where one lane reads what
// another wrote (LDS serves a wave in order: no instruction).
__device__ __forceinline__ void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local"); }
__device__ __forceinline__ uint64_t mask_xor2(uint64_t m) { return (m & kLow2) << 2 | (m >> 2 & kLow2); }

__device__ __forceinline__ BlasResult traverse_quad(const float4* __restrict__ nodes, const float4* __restrict__ wide,
                                                    const float* __restrict__ tris, const DRay& ray, bool degen,
                                                    lds_u64* st, bool& overflow)
{
    constexpr uint32_t kPop = 0xFFFFFFFEu, kDone = 0xFFFFFFFDu, kFull = 0xFFFFFFFCu;  // no leaf's ref (packed_stack)
    const uint32_t q = threadIdx.x & 3u;
    const uint32_t pair_bits = kPairRef | (q >> 1) << kPackShift;
    const float neg_inf = __uint_as_float(0xFF800000u);
    float closest = ray.t;
    uint32_t prim = BVHT_MISS, sp = 0;
    const uint32_t root = __float_as_uint(nodes[0].w), root_cnt = __float_as_uint(nodes[1].w);
    // current node: an interior node or a pair below kPackFlag, a leaf below
    // kFull, kFull (out of entries), kDone, kPop
    uint32_t cur = root_cnt ? kPackFlag | root_cnt << kPackShift | root : root;
    while (true) {
        while ((int32_t)cur >= 0) {
            const uint32_t rec = cur & kPackMask;
            const float4* at = reinterpret_cast<const float4*>(reinterpret_cast<const char*>(wide) +
                                                               ((rec << 6) + (q << 5)));
            const float4 lo = at[0], hi = at[1];
            const uint32_t ref = __float_as_uint(lo.w);
            const float x1 = (lo.x - ray.o.x) * ray.r.x, x2 = (hi.x - ray.o.x) * ray.r.x;
            const float y1 = (lo.y - ray.o.y) * ray.r.y, y2 = (hi.y - ray.o.y) * ray.r.y;
            const float z1 = (lo.z - ray.o.z) * ray.r.z, z2 = (hi.z - ray.o.z) * ray.r.z;
            const float nx = fminf(x1, x2), ny = fminf(y1, y2), nz = fminf(z1, z2);
            const float tmin = fmaxf(fmaxf(nx, ny), nz);
            const float tmax = fminf(fminf(fmaxf(x1, x2), fmaxf(y1, y2)), fmaxf(z1, z2));
            // a pair's step takes its side only: in the lanes of the other side
            // its two bits differ from theirs in the side
            const uint64_t out = lanes_of(((cur >> kPackShift) ^ (pair_bits >> kPackShift)) == 1u);
            uint64_t hit = lanes_of(tmax >= tmin) & lanes_of(tmax > 0.0f) & ~out;
            // the child's key (meant only where it is hit); beside a leaf child
            // stands a box of NaNs, which fminf passes over
            float kp = fmaxf(fmaxf(fminf(nx, dpp_f<kXor1>(nx)), fminf(ny, dpp_f<kXor1>(ny))),
                             fminf(nz, dpp_f<kXor1>(nz)));
            if (degen) {
                kp = slab_key(make_float4(fminf(lo.x, dpp_f<kXor1>(lo.x)), fminf(lo.y, dpp_f<kXor1>(lo.y)),
                                          fminf(lo.z, dpp_f<kXor1>(lo.z)), 0.0f),
                              make_float4(fmaxf(hi.x, dpp_f<kXor1>(hi.x)), fmaxf(hi.y, dpp_f<kXor1>(hi.y)),
                                          fmaxf(hi.z, dpp_f<kXor1>(hi.z)), 0.0f),
                              ray);
                hit &= lanes_of(kp < closest) | lanes_of((cur & kPairRef) != 0);
            }
            const float key = lane_in(hit) ? tmin : kFltMax;
            // the side's nearer grandchild first, ties to the right one; then
            // the nearer side, ties to the right one
            const float kn = dpp_f<kXor1>(key), kpo = dpp_f<kXor2>(kp);
            const uint64_t first = (lanes_of(key < kn) & kEven) | (lanes_of(key <= kn) & ~kEven);
            const uint64_t below = lanes_of(key < closest);
            const uint64_t pass = below | mask_xor1(below), pass_o = mask_xor2(pass);
            const uint64_t near =
                pass & (~pass_o | (lanes_of(kp < kpo) & kLow2) | (lanes_of(kp <= kpo) & ~kLow2));
            const uint64_t both = pass & pass_o;
            const uint32_t rn = dpp_u<kXor1>(ref);
            const uint32_t ra = lane_in(first) ? ref : rn;
            const float ks = lane_in(first) ? kn : key;
            const uint32_t rao = dpp_u<kXor2>(ra);
            const float kso = dpp_f<kXor2>(ks);
            // the near side's second grandchild, and the far side: a leaf
            // child, or the pair
            const uint64_t second = lanes_of((lane_in(near) ? ks : kso) < closest) & (pass | pass_o);
            const uint64_t push = (below & near & ~first) | (both & first & ~near);
            if (lane_in(push)) {
                const uint64_t child = lanes_of(rn == kNoRef) & ~near;  // far leaf children
                const uint64_t leaf = lanes_of((int32_t)ref < 0);
                const uint32_t e = lane_in(near | child) ? ref : rec | pair_bits;
                const uint32_t k = __float_as_uint(lane_in((near & leaf) | child) ? neg_inf : key);
                st[(sp + (lane_in(near & both) ? 1u : 0u)) * 16] = (uint64_t)k << 32 | e;
            }
            wave_lds_fence();  // the pop's reads come after
            sp += (lane_in(both) ? 1u : 0u) + (lane_in(second) ? 1u : 0u);
            const uint32_t next = lane_in(near) ? ra : rao;
            cur = sp > kQuadSlots - 2 ? kFull : lane_in(pass | pass_o) ? next : kPop;
            if ((uint32_t)__popcll(lanes_of((int32_t)cur >= 0)) < kDescendMin)
                break;
        }
        if ((int32_t)cur < 0 && cur < kFull) {
            const uint32_t begin = cur & kPackMask, cnt = (cur >> kPackShift) & 63u;
            float bt = closest;
            uint32_t bi = BVHT_MISS;
            for (uint32_t k = q; k < cnt; k += 4) {
                float t, u, v;
                if (tri_test(tris + 9 * (size_t)(begin + k), ray, t, u, v) && t < bt) {
                    bt = t;
                    bi = begin + k;
                }
            }
            float ot = dpp_f<kXor1>(bt);
            uint32_t oi = dpp_u<kXor1>(bi);
            bool take = lane_in(lanes_of(ot < bt) | (lanes_of(ot == bt) & lanes_of(oi < bi)));
            bt = take ? ot : bt;
            bi = take ? oi : bi;
            ot = dpp_f<kXor2>(bt);
            oi = dpp_u<kXor2>(bi);
            take = lane_in(lanes_of(ot < bt) | (lanes_of(ot == bt) & lanes_of(oi < bi)));
            closest = take ? ot : bt;
            bi = take ? oi : bi;
            prim = bi != BVHT_MISS ? bi : prim;
            cur = kPop;
        }
        if (cur == kPop) {
            cur = kDone;
            while (sp > 0) {
                --sp;
                const uint64_t e = st[sp * 16];
                if (__uint_as_float((uint32_t)(e >> 32)) < closest) {
                    cur = (uint32_t)e;
                    break;
                }
            }
        }
        if (cur == kDone || cur == kFull)
            break;
        wave_lds_fence();                 // the next push's writes come after the pop's reads
        __builtin_amdgcn_wave_barrier();  // one loop latch for every lane (see traverse_blas)
    }
    overflow = cur == kFull;
    // the hit's t, u and v again from its triangle: the same arithmetic
    BlasResult res{0.0f, 0.0f, 0.0f, prim, false};
    if (prim != BVHT_MISS && closest < kFltMax)
        res.found = tri_test(tris + 9 * (size_t)prim, ray, res.t, res.u, res.v);
    return res;
}

// One ray of a quad: traverse_quad where the tree's records are unmarked and
// every ray of the wave allows it, else (and for a ray whose stack overflowed)
// the binary loop in the quad's first lane, with the quad's LDS as its stack.
// The result is the first lane's.  lds: kQuadLds words for each lane of the
// workgroup; each wave keeps to its own.
__device__ __forceinline__ BlasResult trace_quad(const float4* __restrict__ nodes, const float4* __restrict__ wide,
                                                 const float* __restrict__ tris, const DRay& ray, uint32_t* lds,
                                                 uint32_t* spill, size_t stride, uint32_t cap, uint32_t* status)
{
    lds_u32* wave = (lds_u32*)(lds + (threadIdx.x >> 6) * (64 * kQuadLds));
    const uint32_t lane = threadIdx.x & 63u;
    BlasResult r{0.0f, 0.0f, 0.0f, 0u, false};
    bool again = true;
    if (*reinterpret_cast<const uint32_t*>(wide) == 0 && __builtin_amdgcn_ballot_w64(!wide_ray(ray)) == 0)
        r = traverse_quad(nodes, wide, tris, ray, __builtin_amdgcn_ballot_w64(!finite_dir(ray)) != 0,
                          reinterpret_cast<lds_u64*>(wave) + (lane >> 2), again);
    // (the ballot keeps the binary loop behind the other for the whole wave:
    // both use its LDS)
    wave_lds_fence();
    if (__builtin_amdgcn_ballot_w64(again) != 0 && again && (lane & 3u) == 0) {
        Stack<kQuadStack, 16> st{wave + (lane >> 2), spill, stride, cap, status};
        uint32_t pairs = 0, tests = 0;
        r = traverse_blas<false, true, false>(nodes, tris, ray, st, 0u, pairs, tests);
    }
    return r;
}

// Per-BLAS device pointers used by the TLAS kernels.
struct BlasRef {
    const float4* nodes;
    const float* tris;
    uint64_t ntris;
};

// Object record as the TLAS kernels read it: the 3x4 row block of M^-1
// ({m[0][i], m[1][i], m[2][i], m[3][i]} for rows i = 0..2) and the BLAS id.
struct ObjRows {
    float4 r0, r1, r2;
    uint32_t blas;
    uint32_t pad[3];
};

// Whether a hit record is bounced off: a hit whose indices lie inside the
// structure (prim < prim_limit and inst < inst_limit; for TLAS hits, with
// rows/blases given, prim below the triangle count of the object's BLAS).
// Hits outside are skipped, never dereferenced.
__device__ __forceinline__ bool bounce_hit(const bvht_hit& h, uint32_t prim_limit, uint32_t inst_limit,
                                           const ObjRows* rows, const BlasRef* blases)
{
    if (h.prim == BVHT_MISS || h.inst >= inst_limit)
        return false;
    if (rows)
        return h.prim < blases[rows[h.inst].blas].ntris;
    return h.prim < prim_limit;
}

struct TlasResult {
    float t, u, v;
    uint32_t prim, inst;
    bool found;
};

// Tlas::intersect (tlas.rs:123-177): the TLAS node loop with
// SceneObject::intersect at the leaves (scene_object.rs:77-89).  Left child =
// high 16 bits of the LeftRightIndex word (tlas.rs:24-32).
//
// Both levels run in one loop: a lane is either in the TLAS (world ray) or in
// the BLAS of the object whose leaf it reached (object-space ray), and the
// node-pair steps of the two levels share one step body, so the lanes of a
// wave descend their instances' BLASes together instead of one instance
// visit at a time.  Each lane's sequence of TLAS steps, object visits (with
// the BLAS traversal of traverse_blas inside) and pops is that of the nested
// traversal; a visit's nearest hit is committed when its BLAS stack empties,
// under the same conditions as the nested form (found, t < FLT_MAX, t below
// the committed distance).
template <bool STATS, bool PACKED = false, bool FINITE = false, class StackT>
__device__ __forceinline__ TlasResult traverse_tlas(const float4* __restrict__ tnodes, const ObjRows* __restrict__ objs,
                                                    const BlasRef* __restrict__ blases, const DRay& ray,
                                                    StackT& st, uint32_t& pairs, uint32_t& tests,
                                                    uint32_t& tpairs, uint32_t& visits)
{
    TlasResult res{0.0f, 0.0f, 0.0f, 0u, 0u, false};
    float closest = ray.t;  // committed nearest distance (world)
    // Current level: in_blas = false -> TLAS with the world ray; true -> the
    // BLAS of object `obj` with the object-space ray cr.
    bool in_blas = false;
    DRay cr = ray;
    float cclosest = closest;  // culling distance of the current level
    const float4* bnodes = tnodes;
    const float* btris = nullptr;
    uint32_t obj = 0, sp = 0, sp_base = 0;
    float bt = 0.0f, bu = 0.0f, bv = 0.0f;
    uint32_t bprim = 0;
    bool bfound = false;
    // Current node: TLAS -> (left_right, object index), leaf when x == 0;
    // BLAS -> (left_first, count), leaf when y > 0.
    uint32_t x = __float_as_uint(tnodes[0].w);
    uint32_t y = __float_as_uint(tnodes[1].w);
    bool pend = false;
    while (true) {
        while (!pend && (in_blas ? y == 0 : x != 0)) {
            if (STATS) {
                if (in_blas)
                    ++pairs;
                else
                    ++tpairs;
            }
            const float4* pl;
            const float4* pr;
            if (in_blas) {
                pl = bnodes + 2 * (size_t)x;
                pr = pl + 2;
            } else {
                pl = tnodes + 2 * (size_t)((x & 0xFFFF0000u) >> 16);
                pr = tnodes + 2 * (size_t)(x & 0x0000FFFFu);
            }
            float4 a0 = pl[0], a1 = pl[1], b0 = pr[0], b1 = pr[1];
            bool left_near, near_hit, far_hit;
            if (FINITE) {
                float kl = slab_key(a0, a1, cr);
                float kr = slab_key(b0, b1, cr);
                left_near = kl < kr;
                near_hit = (left_near ? kl : kr) < cclosest;
                far_hit = (left_near ? kr : kl) < cclosest;
            } else {
                float dl, dr;
                bool hl = slab(a0, a1, cr, cclosest, dl);
                bool hr = slab(b0, b1, cr, cclosest, dr);
                float kl = hl ? dl : kFltMax;
                float kr = hr ? dr : kFltMax;
                left_near = kl < kr;
                near_hit = left_near ? hl : hr;
                far_hit = left_near ? hr : hl;
            }
            if (near_hit) {
                if (far_hit) {
                    uint32_t e;
                    if (in_blas) {
                        uint32_t flf = __float_as_uint(left_near ? b0.w : a0.w);
                        uint32_t fcnt = __float_as_uint(left_near ? b1.w : a1.w);
                        e = PACKED ? (kPackFlag | (fcnt << kPackShift) | flf)
                                   : pack_entry(left_near ? x + 1 : x, flf, fcnt);
                    } else
                        e = left_near ? (x & 0x0000FFFFu) : ((x & 0xFFFF0000u) >> 16);
                    st.push(sp, e);
                }
                uint32_t nx = __float_as_uint(left_near ? a0.w : b0.w);
                y = __float_as_uint(left_near ? a1.w : b1.w);
                x = nx;
            } else {
                pend = true;
            }
            if ((uint32_t)__popcll(__builtin_amdgcn_ballot_w64(!pend && (in_blas ? y == 0 : x != 0))) < kDescendMin)
                break;
        }
        if (!pend && in_blas && y > 0) {
            for (uint32_t k = 0; k < y; ++k) {
                float t, u, v;
                if (STATS)
                    ++tests;
                if (tri_test(btris + 9 * (size_t)(x + k), cr, t, u, v) && t < cclosest) {
                    cclosest = t;
                    bt = t;
                    bu = u;
                    bv = v;
                    bprim = x + k;
                    bfound = true;
                }
            }
            pend = true;
        }
        if (!pend && !in_blas && x == 0) {
            // object leaf: enter its BLAS with the object-space ray
            if (STATS)
                ++visits;
            const ObjRows* ob = objs + y;
            float4 q0 = ob->r0, q1 = ob->r1, q2 = ob->r2;
            uint32_t model = ob->blas;
            V3 om = rows_mul(q0, q1, q2, ray.o, 1.0f);
            V3 dm = rows_mul(q0, q1, q2, ray.d, 0.0f);
            cr = make_ray(om, dm, closest);
            BlasRef br = blases[model];
            bnodes = br.nodes;
            btris = br.tris;
            obj = y;
            sp_base = sp;
            cclosest = closest;
            bfound = false;
            in_blas = true;
            x = __float_as_uint(bnodes[0].w);
            y = __float_as_uint(bnodes[1].w);
        }
        if (pend) {
            if (in_blas && sp == sp_base) {
                // the object's BLAS traversal is over: commit its nearest hit
                if (bfound && cclosest < kFltMax && cclosest < closest) {
                    closest = cclosest;
                    res.t = bt;
                    res.u = bu;
                    res.v = bv;
                    res.prim = bprim;
                    res.inst = obj;
                    res.found = true;
                }
                in_blas = false;
                cr = ray;
                cclosest = closest;
            }
            if (!in_blas && sp == 0)
                break;
            uint32_t e = st.pop(sp);
            if (!in_blas) {
                x = __float_as_uint(tnodes[2 * (size_t)e].w);
                y = __float_as_uint(tnodes[2 * (size_t)e + 1].w);
            } else if (PACKED || (e & kPackFlag)) {
                x = e & kPackMask;
                y = (e >> kPackShift) & 63u;
            } else {
                x = __float_as_uint(bnodes[2 * (size_t)e].w);
                y = __float_as_uint(bnodes[2 * (size_t)e + 1].w);
            }
            pend = false;
        }
        // one loop latch for every lane (see traverse_blas)
        __builtin_amdgcn_wave_barrier();
    }
    if (!(closest < kFltMax))
        res.found = false;
    return res;
}

}  // namespace bvht
