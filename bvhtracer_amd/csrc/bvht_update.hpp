// bvht_update.hpp -- per-frame structure updates shared by the single-structure
// kernels and the batched multi-scene kernels: BLAS refit, object bounds and
// the TLAS rebuild.
#pragma once

#include "bvht_device.hpp"
#include "bvht_trace.hpp"

namespace bvht {

// Bvh::refit (bvh.rs:469-493) for node k, run one tree level at a time from
// the deepest level up (the levels are separate launches, so a node's
// children are final when it is processed): a leaf recomputes its box from
// its triangles starting at (+MAX, -MAX) (update_node_bounds, bvh.rs:317-330),
// a branch takes the union of its two children.  min/max are exact and every
// child has a larger index than its parent (bvh.rs:601-612), so the result
// equals the reference's reverse index sweep bit for bit.
// Leaves with more than kBigLeaf triangles (the reference builder makes
// leaves of thousands) are refit by a whole wave each (refit_big_leaf), before
// the level passes; refit_node leaves them alone.
constexpr uint32_t kBigLeaf = 64;

__device__ __forceinline__ void leaf_box(const float* __restrict__ tris, uint32_t first, uint32_t count, V3& lo, V3& hi)
{
    lo = mk3(kFltMax, kFltMax, kFltMax);
    hi = mk3(-kFltMax, -kFltMax, -kFltMax);
    for (uint32_t j = 0; j < count; ++j) {
        const float* t = tris + 9 * (size_t)(first + j);
        V3 v0 = mk3(t[0], t[1], t[2]), v1 = mk3(t[3], t[4], t[5]), v2 = mk3(t[6], t[7], t[8]);
        lo = min3(lo, v0);
        lo = min3(lo, v1);
        lo = min3(lo, v2);
        hi = max3(hi, v0);
        hi = max3(hi, v1);
        hi = max3(hi, v2);
    }
}

__device__ __forceinline__ void refit_node(bvht_node* __restrict__ nodes, const float* __restrict__ tris, uint32_t k)
{
    bvht_node nd = nodes[k];
    if (nd.count > kBigLeaf)
        return;
    V3 lo, hi;
    if (nd.count > 0) {
        leaf_box(tris, nd.left_first, nd.count, lo, hi);
    } else {
        bvht_node a = nodes[nd.left_first], c = nodes[nd.left_first + 1];
        lo = min3(mk3(a.bmin[0], a.bmin[1], a.bmin[2]), mk3(c.bmin[0], c.bmin[1], c.bmin[2]));
        hi = max3(mk3(a.bmax[0], a.bmax[1], a.bmax[2]), mk3(c.bmax[0], c.bmax[1], c.bmax[2]));
    }
    float4* o = reinterpret_cast<float4*>(nodes + k);
    o[0] = make_float4(lo.x, lo.y, lo.z, __uint_as_float(nd.left_first));
    o[1] = make_float4(hi.x, hi.y, hi.z, __uint_as_float(nd.count));
}

// Leaf k's box from its triangles by the 64 lanes of one wave: lanes take
// every 64th triangle, then min/max are combined across the wave (exact, so
// the order does not change the box; only the sign of a zero bound can
// differ from the sequential sweep).  Every lane of the wave must call it.
__device__ __forceinline__ void refit_big_leaf(bvht_node* __restrict__ nodes, const float* __restrict__ tris,
                                               uint32_t k, uint32_t lane)
{
    bvht_node nd = nodes[k];
    V3 lo = mk3(kFltMax, kFltMax, kFltMax);
    V3 hi = mk3(-kFltMax, -kFltMax, -kFltMax);
    for (uint32_t j = lane; j < nd.count; j += 64) {
        const float* t = tris + 9 * (size_t)(nd.left_first + j);
        V3 v0 = mk3(t[0], t[1], t[2]), v1 = mk3(t[3], t[4], t[5]), v2 = mk3(t[6], t[7], t[8]);
        lo = min3(min3(min3(lo, v0), v1), v2);
        hi = max3(max3(max3(hi, v0), v1), v2);
    }
    for (int m = 32; m >= 1; m >>= 1) {
        lo = min3(lo, mk3(__shfl_xor(lo.x, m, 64), __shfl_xor(lo.y, m, 64), __shfl_xor(lo.z, m, 64)));
        hi = max3(hi, mk3(__shfl_xor(hi.x, m, 64), __shfl_xor(hi.y, m, 64), __shfl_xor(hi.z, m, 64)));
    }
    if (lane == 0) {
        float4* o = reinterpret_cast<float4*>(nodes + k);
        o[0] = make_float4(lo.x, lo.y, lo.z, __uint_as_float(nd.left_first));
        o[1] = make_float4(hi.x, hi.y, hi.z, __uint_as_float(nd.count));
    }
}

// Refit of a chunk of consecutive nodes (at most kRefitChunk) by one workgroup,
// in LDS: every leaf, and every branch whose whole subtree lies in the chunk.
// Nodes are numbered depth first (a subtree's nodes are consecutive), so a
// boundary cuts the ancestors of the pair it stands at, and it is put at a
// pair of the least level in a window of kChunkWindow nodes (chunk_start): 691
// of the 163,840 nodes of an 81,920-triangle sphere, on 12 levels, are left for
// the level passes, where boundaries at every 1,024th node leave 2,004 on 19.
// Which branches are inside is a property of the tree, kept in bit 31 of
// `level` (mark_chunk).  Rounds go up the chunk's levels, deepest first, with a
// barrier between; a branch's children are one level below it.  A tree of at
// most kRefitChunk nodes is one chunk and has no pass after it (one chunk or
// chunks of 768: 160 triangles' nodes in 4.4 or 4.2 us, 1,440 in 9.4 or 11.0,
// 1,960 in 11.4 or 11.3; level passes of all nodes 6.3, 9.7 and 10.7).  Bound by
// latency and launches up to some 200k triangles (8.9 us for 81,920, the level
// passes after it 10.3), by HBM beyond (16 scenes of 0.9M triangles, 155 MB: 62
// us; 54 where no chunk has more than 1,024 nodes, with 512 threads).
constexpr uint32_t kRefitChunk = 2048;
constexpr uint32_t kChunkStride = 768, kChunkWindow = 256;
constexpr uint32_t kChunkWG = 1024;
constexpr uint32_t kChunkPer = kRefitChunk / kChunkWG;
constexpr uint32_t kInChunk = 0x80000000u;
inline uint32_t chunk_count(uint32_t nodes_used)
{
    return nodes_used <= kRefitChunk ? 1u : (nodes_used + kChunkStride - 1) / kChunkStride;
}

// First node of chunk `chunk`: of the pairs at [768 chunk, + 256) one of the
// least level (levels without bit 31), the first; by one wave, in every lane.
__device__ __forceinline__ uint32_t chunk_start(const uint32_t* __restrict__ level, uint32_t nodes_used,
                                                uint32_t chunk, uint32_t lane)
{
    const uint32_t from = chunk * kChunkStride;
    if (chunk == 0 || from >= nodes_used)
        return min(from, nodes_used);
    uint32_t best = 0xFFFFFFFFu;  // level << 8 | offset
    for (uint32_t o = 2 * lane; o < kChunkWindow; o += 128)
        if (from + o < nodes_used)
            best = min(best, level[from + o] << 8 | o);
    for (int m = 32; m >= 1; m >>= 1)
        best = min(best, (uint32_t)__shfl_xor((int)best, m, 64));
    return from + (best & 0xFFu);
}

// Levels of the chunk's branches: [lowest, highest], lowest > highest if none.
__device__ __forceinline__ void chunk_levels(const uint32_t (&lv)[kChunkPer], uint32_t& lowest, uint32_t& highest)
{
    __shared__ uint32_t s_lo, s_hi;
    if (threadIdx.x == 0) {
        s_lo = 0xFFFFFFFFu;
        s_hi = 0;
    }
    __syncthreads();
    uint32_t lo = 0xFFFFFFFFu, hi = 0;
    for (uint32_t j = 0; j < kChunkPer; ++j)
        if (lv[j] != BVHT_MISS) {
            lo = min(lo, lv[j]);
            hi = max(hi, lv[j]);
        }
    for (int m = 32; m >= 1; m >>= 1) {
        lo = min(lo, (uint32_t)__shfl_xor((int)lo, m, 64));
        hi = max(hi, (uint32_t)__shfl_xor((int)hi, m, 64));
    }
    if ((threadIdx.x & 63u) == 0) {
        atomicMin(&s_lo, lo);
        atomicMax(&s_hi, hi);
    }
    __syncthreads();
    lowest = s_lo;
    highest = s_hi;
}

// Sets bit 31 of `level` for the leaves among nodes [base, end) and for the
// branches whose subtrees lie there.  (Node 1 is no node.)
__device__ __forceinline__ void mark_chunk(const bvht_node* __restrict__ nodes, uint32_t base, uint32_t end,
                                           uint32_t* __restrict__ level)
{
    __shared__ uint8_t inside[kRefitChunk];
    uint32_t lv[kChunkPer], child[kChunkPer];
    for (uint32_t j = 0; j < kChunkPer; ++j) {
        const uint32_t i = j * kChunkWG + threadIdx.x, k = base + i;
        lv[j] = BVHT_MISS;
        child[j] = 0;
        bool leaf = false;
        if (k < end && k != 1) {
            leaf = nodes[k].count > 0;
            if (leaf) {
                level[k] |= kInChunk;
            } else {
                lv[j] = level[k];
                child[j] = nodes[k].left_first - base;  // children come after their parent
            }
        }
        inside[i] = leaf;
    }
    uint32_t lowest, highest;
    chunk_levels(lv, lowest, highest);
    for (uint32_t L = highest + 1; L-- > lowest;) {
        for (uint32_t j = 0; j < kChunkPer; ++j)
            if (lv[j] == L && child[j] + 1 < end - base && inside[child[j]] && inside[child[j] + 1]) {
                inside[j * kChunkWG + threadIdx.x] = 1;
                level[base + j * kChunkWG + threadIdx.x] = L | kInChunk;
            }
        __syncthreads();
    }
}

__device__ __forceinline__ void refit_chunk(bvht_node* __restrict__ nodes, const float* __restrict__ tris,
                                            const uint32_t* __restrict__ level, uint32_t base, uint32_t end,
                                            float4* __restrict__ wide, uint32_t stale)
{
    if (wide && base == 0 && threadIdx.x == 0)
        *reinterpret_cast<uint32_t*>(wide) = stale;  // the mark: 1, or 0 if the records are written after this
    __shared__ float box[6][kRefitChunk];
    uint32_t lv[kChunkPer], lf[kChunkPer];
    for (uint32_t j = 0; j < kChunkPer; ++j) {
        const uint32_t i = j * kChunkWG + threadIdx.x, k = base + i;
        lv[j] = BVHT_MISS;
        lf[j] = 0;
        if (k >= end || k == 1 || !(level[k] & kInChunk))
            continue;
        float4* b = reinterpret_cast<float4*>(nodes + k);
        const float4 a = b[0], c = b[1];
        const uint32_t cnt = __float_as_uint(c.w);
        lf[j] = __float_as_uint(a.w);
        if (cnt == 0) {
            lv[j] = level[k] & ~kInChunk;
            continue;
        }
        V3 lo = mk3(a.x, a.y, a.z), hi = mk3(c.x, c.y, c.z);  // a big leaf has its box by now
        if (cnt <= kBigLeaf) {
            leaf_box(tris, lf[j], cnt, lo, hi);
            b[0] = make_float4(lo.x, lo.y, lo.z, a.w);
            b[1] = make_float4(hi.x, hi.y, hi.z, c.w);
        }
        box[0][i] = lo.x;
        box[1][i] = lo.y;
        box[2][i] = lo.z;
        box[3][i] = hi.x;
        box[4][i] = hi.y;
        box[5][i] = hi.z;
    }
    uint32_t lowest, highest;
    chunk_levels(lv, lowest, highest);
    for (uint32_t L = highest + 1; L-- > lowest;) {
        for (uint32_t j = 0; j < kChunkPer; ++j) {
            if (lv[j] != L)
                continue;
            const uint32_t i = j * kChunkWG + threadIdx.x, c = lf[j] - base;
            const V3 lo = min3(mk3(box[0][c], box[1][c], box[2][c]), mk3(box[0][c + 1], box[1][c + 1], box[2][c + 1]));
            const V3 hi = max3(mk3(box[3][c], box[4][c], box[5][c]), mk3(box[3][c + 1], box[4][c + 1], box[5][c + 1]));
            box[0][i] = lo.x;
            box[1][i] = lo.y;
            box[2][i] = lo.z;
            box[3][i] = hi.x;
            box[4][i] = hi.y;
            box[5][i] = hi.z;
            float4* o = reinterpret_cast<float4*>(nodes + base + i);
            o[0] = make_float4(lo.x, lo.y, lo.z, __uint_as_float(lf[j]));
            o[1] = make_float4(hi.x, hi.y, hi.z, 0.0f);
        }
        __syncthreads();
    }
}

// SceneObject::set_transform (scene_object.rs:60-75) for object i: world box of
// the 8 corners of its BLAS root box under M, and the traced rows of M^-1.
__device__ __forceinline__ void object_bounds(const bvht_instance* __restrict__ objs,
                                              const BlasRef* __restrict__ blases, float* __restrict__ bounds,
                                              ObjRows* __restrict__ rows, uint32_t i)
{
    const bvht_instance& o = objs[i];
    const float4* bn = blases[o.blas].nodes;
    float4 a = bn[0], b = bn[1];
    V3 lo = mk3(kFltMax, kFltMax, kFltMax), hi = mk3(-kFltMax, -kFltMax, -kFltMax);
    for (int c = 0; c < 8; ++c) {
        V3 p = mk3((c & 1) ? b.x : a.x, (c & 2) ? b.y : a.y, (c & 4) ? b.z : a.z);
        V3 w = mat_mul4(o.m, p, 1.0f);
        lo = min3(lo, w);
        hi = max3(hi, w);
    }
    float* bo = bounds + 6 * (size_t)i;
    bo[0] = lo.x; bo[1] = lo.y; bo[2] = lo.z;
    bo[3] = hi.x; bo[4] = hi.y; bo[5] = hi.z;
    ObjRows r;
    r.r0 = make_float4(o.minv[0], o.minv[4], o.minv[8], o.minv[12]);
    r.r1 = make_float4(o.minv[1], o.minv[5], o.minv[9], o.minv[13]);
    r.r2 = make_float4(o.minv[2], o.minv[6], o.minv[10], o.minv[14]);
    r.blas = o.blas;
    r.pad[0] = r.pad[1] = r.pad[2] = 0;
    rows[i] = r;
}

constexpr uint32_t kRebuildWG = 256;

// Tlas::find_best_match (tlas.rs:179-202) as a block-wide argmin: the
// sequential scan keeps the first b whose area is strictly below the running
// minimum (starting at f32::MAX), i.e. the smallest index among the minimal
// areas that are < f32::MAX.
__device__ __forceinline__ int32_t block_best_match(const bvht_tnode* nodes, const int32_t* list, int32_t count, int32_t a,
                                    float* s_val, int32_t* s_idx)
{
    float best = kFltMax;
    int32_t bi = -1;
    const bvht_tnode& na = nodes[list[a]];
    for (int32_t b = threadIdx.x; b < count; b += kRebuildWG) {
        if (b == a)
            continue;
        const bvht_tnode& nb = nodes[list[b]];
        V3 mx = max3(mk3(na.bmax[0], na.bmax[1], na.bmax[2]), mk3(nb.bmax[0], nb.bmax[1], nb.bmax[2]));
        V3 mn = min3(mk3(na.bmin[0], na.bmin[1], na.bmin[2]), mk3(nb.bmin[0], nb.bmin[1], nb.bmin[2]));
        V3 e = sub3(mx, mn);
        float sa = e.x * e.y + e.y * e.z + e.z * e.x;
        if (sa < best) {
            best = sa;
            bi = b;
        }
    }
    s_val[threadIdx.x] = best;
    s_idx[threadIdx.x] = bi;
    __syncthreads();
    for (uint32_t off = kRebuildWG / 2; off > 0; off >>= 1) {
        if (threadIdx.x < off) {
            float v2 = s_val[threadIdx.x + off];
            int32_t i2 = s_idx[threadIdx.x + off];
            float v1 = s_val[threadIdx.x];
            int32_t i1 = s_idx[threadIdx.x];
            bool take = i2 >= 0 && (i1 < 0 || v2 < v1 || (!(v1 < v2) && i2 < i1));
            if (take) {
                s_val[threadIdx.x] = v2;
                s_idx[threadIdx.x] = i2;
            }
        }
        __syncthreads();
    }
    int32_t r = s_idx[0];
    __syncthreads();
    return r;
}

// The merge loop of Tlas::rebuild (tlas.rs:204-250) for 1 <= n <= 64 objects
// by one wave, without barriers.  Lane i holds list entry i in registers: the
// node index, its box, link field, object index and subtree height (entries
// past count keep their last values, as the reference's list does).
// find_best_match is a butterfly minimum over the areas < f32::MAX (as
// order-preserving unsigned keys) followed by a ballot for the first lane
// holding it: the sequential scan's first minimum.  Lane 0 writes the merged
// nodes, the root copy in node 0 and the results; the height of the root is
// the depth that walking the tree from node 0 gives.  The loop is capped (it
// ends after at most n merges and chain steps, far below the cap).
__device__ __forceinline__ float lane_f(float v, int32_t l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ int32_t lane_i(int32_t v, int32_t l) { return __builtin_amdgcn_readlane(v, l); }

__device__ void wave_rebuild_loop(const float* __restrict__ bounds, bvht_tnode* nodes, int32_t* list, int32_t n,
                                  int32_t* out_a, int32_t* out_used, int32_t* out_fail, uint32_t* out_depth)
{
    const int32_t lane = (int32_t)(threadIdx.x & 63u);
    int32_t li = 0, lr = 0, obj = 0, h = 1;
    V3 lo = mk3(0.0f, 0.0f, 0.0f), hi = lo;
    if (lane < n) {  // leaves 1..n in object order
        const float* bb = bounds + 6 * (size_t)lane;
        li = lane + 1;
        obj = lane;
        lo = mk3(bb[0], bb[1], bb[2]);
        hi = mk3(bb[3], bb[4], bb[5]);
    }
    auto best_match = [&](int32_t count, int32_t x) -> int32_t {
        V3 xl = mk3(lane_f(lo.x, x), lane_f(lo.y, x), lane_f(lo.z, x));
        V3 xh = mk3(lane_f(hi.x, x), lane_f(hi.y, x), lane_f(hi.z, x));
        // candidate areas as order-preserving unsigned keys (an area is
        // never -0, so equal areas give equal keys); no candidate: ~0
        uint32_t key = 0xFFFFFFFFu;
        if (lane < count && lane != x) {
            V3 e = sub3(max3(xh, hi), min3(xl, lo));
            float sa = e.x * e.y + e.y * e.z + e.z * e.x;
            if (sa < kFltMax) {
                uint32_t u = __float_as_uint(sa);
                key = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
            }
        }
        uint32_t mk = key, ul = (uint32_t)lane;  // butterfly minimum, VALU exchanges
        mk = min(mk, xor_lane<32>(mk, ul));
        mk = min(mk, xor_lane<16>(mk, ul));
        mk = min(mk, xor_lane<8>(mk, ul));
        mk = min(mk, xor_lane<4>(mk, ul));
        mk = min(mk, xor_lane<2>(mk, ul));
        mk = min(mk, xor_lane<1>(mk, ul));
        mk = __builtin_amdgcn_readfirstlane(mk);
        if (mk == 0xFFFFFFFFu)
            return -1;
        // the first lane holding the minimum: the sequential scan's choice
        return (int32_t)__ffsll((long long)__ballot(key == mk)) - 1;
    };
    int32_t count = n, used = n + 1, a = 0, fail = 0;
    int32_t b = best_match(count, a);
    for (int32_t guard = 0; count > 1; ++guard) {
        if (b < 0 || guard > 8 * 64 * 64) {  // every area >= f32::MAX (the reference panics)
            fail = 1;
            break;
        }
        int32_t c = best_match(count, b);
        if (a == c) {
            int32_t ia = lane_i(li, a), ib = lane_i(li, b);
            V3 mn = min3(mk3(lane_f(lo.x, a), lane_f(lo.y, a), lane_f(lo.z, a)),
                         mk3(lane_f(lo.x, b), lane_f(lo.y, b), lane_f(lo.z, b)));
            V3 mx = max3(mk3(lane_f(hi.x, a), lane_f(hi.y, a), lane_f(hi.z, a)),
                         mk3(lane_f(hi.x, b), lane_f(hi.y, b), lane_f(hi.z, b)));
            int32_t hn = 1 + max(lane_i(h, a), lane_i(h, b));
            int32_t lrn = (int32_t)((uint32_t)ia + ((uint32_t)ib << 16));
            if (lane == 0) {
                bvht_tnode nn;
                nn.left_right = (uint32_t)lrn;
                nn.bmin[0] = mn.x; nn.bmin[1] = mn.y; nn.bmin[2] = mn.z;
                nn.bmax[0] = mx.x; nn.bmax[1] = mx.y; nn.bmax[2] = mx.z;
                nn.blas = 0;
                nodes[used] = nn;
            }
            // list[a] = used, then list[b] = list[count - 1] (which is the new
            // entry when a == count - 1)
            if (lane == a) {
                li = used;
                lo = mn;
                hi = mx;
                lr = lrn;
                obj = 0;
                h = hn;
            }
            int32_t t = count - 1;
            int32_t tli = lane_i(li, t), tlr = lane_i(lr, t), tobj = lane_i(obj, t), th_ = lane_i(h, t);
            V3 tlo = mk3(lane_f(lo.x, t), lane_f(lo.y, t), lane_f(lo.z, t));
            V3 thi = mk3(lane_f(hi.x, t), lane_f(hi.y, t), lane_f(hi.z, t));
            if (lane == b) {
                li = tli;
                lr = tlr;
                obj = tobj;
                h = th_;
                lo = tlo;
                hi = thi;
            }
            used += 1;
            count -= 1;
            b = best_match(count, a);
        } else {
            a = b;
            b = c;
        }
    }
    if (lane < n)
        list[lane] = li;
    // the root (entry a) copied to node 0, and its height
    V3 rl = mk3(lane_f(lo.x, a), lane_f(lo.y, a), lane_f(lo.z, a));
    V3 rh = mk3(lane_f(hi.x, a), lane_f(hi.y, a), lane_f(hi.z, a));
    int32_t rlr = lane_i(lr, a), robj = lane_i(obj, a), rh_ = lane_i(h, a);
    if (lane == 0) {
        if (!fail) {
            bvht_tnode r;
            r.bmin[0] = rl.x; r.bmin[1] = rl.y; r.bmin[2] = rl.z;
            r.bmax[0] = rh.x; r.bmax[1] = rh.y; r.bmax[2] = rh.z;
            r.left_right = (uint32_t)rlr;
            r.blas = (uint32_t)robj;
            nodes[0] = r;
        }
        *out_a = a;
        *out_used = used;
        *out_fail = fail;
        *out_depth = (uint32_t)rh_;
    }
}

__device__ __forceinline__ void meta_out(uint32_t* meta, uint32_t used, uint32_t depth, uint32_t status)
{
    meta[0] = used;
    meta[1] = depth;
    meta[2] = status;
}

// The merge loop of Tlas::rebuild for 64 < n <= kRebuildLds objects by one
// workgroup, with the list in LDS: entry i is seven arrays of n words (bmin,
// bmax, node index | subtree height << 16) at sh + 0, n, ... 6 n.  Every thread
// follows the loop (a, b, count) on its own from the same results.
// find_best_match: each thread scans every kRebuildWG-th entry, keeping its
// first minimum; a wave combines by DPP minima of the areas as
// order-preserving keys, then its lowest entry among those holding the
// minimum; the waves' {key, entry} words are read back by all after one
// barrier (two sets of words in turn, so the next scan cannot overtake the
// reading).  The height of the root is the depth that walking the tree from
// node 0 gives.  Bound by the latency of n dependent rounds of scan, exchange
// and barrier: 400 objects 2543 -> 977 us against the list in global memory with
// a nine-barrier exchange and a walk for the depth.
constexpr uint32_t kRebuildLds = 2048;
inline size_t rebuild_lds_bytes(uint32_t n) { return n > 64 && n <= kRebuildLds ? 7 * sizeof(float) * (size_t)n : 0; }

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v, uint32_t lane)
{
    v = min(v, xor_lane<32>(v, lane));
    v = min(v, xor_lane<16>(v, lane));
    v = min(v, xor_lane<8>(v, lane));
    v = min(v, xor_lane<4>(v, lane));
    v = min(v, xor_lane<2>(v, lane));
    v = min(v, xor_lane<1>(v, lane));
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}

__device__ void block_rebuild_loop(const float* __restrict__ bounds, bvht_tnode* nodes, uint32_t* meta, int32_t n,
                                   float* sh)
{
    __shared__ uint64_t slots[2][kRebuildWG / 64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    uint32_t* const info = reinterpret_cast<uint32_t*>(sh + 6 * n);
    for (int32_t i = (int32_t)tid; i < n; i += kRebuildWG) {  // leaves 1..n in object order
        for (int32_t k = 0; k < 6; ++k)
            sh[k * n + i] = bounds[6 * (size_t)i + k];
        info[i] = (uint32_t)(i + 1) | 1u << 16;
    }
    __syncthreads();
    uint32_t turn = 0;
    auto best_match = [&](int32_t count, int32_t x) -> int32_t {
        const V3 xl = mk3(sh[x], sh[n + x], sh[2 * n + x]);
        const V3 xh = mk3(sh[3 * n + x], sh[4 * n + x], sh[5 * n + x]);
        float best = kFltMax;
        uint32_t bi = 0xFFFFFFFFu;
        for (int32_t i = (int32_t)tid; i < count; i += kRebuildWG) {
            const V3 e = sub3(max3(xh, mk3(sh[3 * n + i], sh[4 * n + i], sh[5 * n + i])),
                              min3(xl, mk3(sh[i], sh[n + i], sh[2 * n + i])));
            const float sa = e.x * e.y + e.y * e.z + e.z * e.x;
            if (i != x && sa < best) {
                best = sa;
                bi = (uint32_t)i;
            }
        }
        // (an area is never -0, so equal areas give equal keys)
        const uint32_t key = bi == 0xFFFFFFFFu ? bi : f2key(best);
        const uint32_t mk = wave_min_u32(key, lane);
        const uint64_t holders = __ballot(key == mk);
        const uint32_t mi = (holders & (holders - 1)) == 0
                                ? (uint32_t)__builtin_amdgcn_readlane((int)bi, (int)__ffsll((long long)holders) - 1)
                                : wave_min_u32(key == mk ? bi : 0xFFFFFFFFu, lane);
        if (lane == 0)
            slots[turn][tid >> 6] = (uint64_t)mk << 32 | mi;
        __syncthreads();
        uint64_t m = slots[turn][0];
        for (uint32_t w = 1; w < kRebuildWG / 64; ++w)
            m = min(m, slots[turn][w]);
        turn ^= 1u;
        return (m >> 32) == 0xFFFFFFFFu ? -1 : (int32_t)(uint32_t)m;
    };
    int32_t count = n, used = n + 1, a = 0;
    int32_t b = best_match(count, a);
    bool fail = false;
    while (count > 1) {
        if (b < 0) {  // every candidate area was >= f32::MAX (the reference panics)
            fail = true;
            break;
        }
        const int32_t c = best_match(count, b);
        if (a != c) {
            a = b;
            b = c;
            continue;
        }
        // merge; list[a] = the new node, then list[b] = list[count - 1].  All
        // scans of the list are behind the barrier in best_match.
        if (tid == 0) {
            const uint32_t ia = info[a], ib = info[b];
            float box[6];
            for (int32_t k = 0; k < 3; ++k) {
                box[k] = fminf(sh[k * n + a], sh[k * n + b]);
                box[3 + k] = fmaxf(sh[(3 + k) * n + a], sh[(3 + k) * n + b]);
            }
            bvht_tnode nn;
            nn.left_right = (ia & 0xFFFFu) + ((ib & 0xFFFFu) << 16);
            nn.blas = 0;
            for (int32_t k = 0; k < 3; ++k) {
                nn.bmin[k] = box[k];
                nn.bmax[k] = box[3 + k];
            }
            nodes[used] = nn;
            for (int32_t k = 0; k < 6; ++k)
                sh[k * n + a] = box[k];
            info[a] = (uint32_t)used | (1u + max(ia >> 16, ib >> 16)) << 16;
            for (int32_t k = 0; k < 6; ++k)
                sh[k * n + b] = sh[k * n + count - 1];
            info[b] = info[count - 1];
        }
        used += 1;
        count -= 1;
        __syncthreads();
        b = best_match(count, a);
    }
    if (tid == 0) {
        if (!fail)
            nodes[0] = nodes[info[a] & 0xFFFFu];
        meta_out(meta, (uint32_t)used, fail ? 0u : info[a] >> 16, fail ? 1u : 0u);
    }
}

// Tlas::rebuild (tlas.rs:204-250) + TlasBuilder::build_for (tlas.rs:273-279):
// 2n default nodes (empty box), leaves 1..n in object order, mutual-best-match
// merges with LeftRightIndex::new(a, b) = a + (b << 16), root = copy of the
// last node.  meta = {nodes_used, depth, status}.
// `lds`: rebuild_lds_bytes(n) of dynamic LDS.  WAVE: n is at most 64, and the
// kernel holds nothing but that loop (64 objects 66.9 us; 70.1 in a kernel that
// holds the other two as well).
template <bool WAVE>
__device__ void tlas_rebuild_block(const float* __restrict__ bounds, uint32_t n, bvht_tnode* nodes, int32_t* list,
                                   uint32_t* meta, float* lds)
{
    __shared__ float s_val[kRebuildWG];
    __shared__ int32_t s_idx[kRebuildWG];
    __shared__ int32_t sh_a, sh_b, sh_count, sh_used, sh_merged, sh_fail;
    __shared__ uint32_t sh_depth;
    for (uint32_t i = threadIdx.x; i < 2 * n; i += kRebuildWG) {
        bvht_tnode d;
        d.bmin[0] = d.bmin[1] = d.bmin[2] = kFltMax;
        d.bmax[0] = d.bmax[1] = d.bmax[2] = -kFltMax;
        d.left_right = 0;
        d.blas = 0;
        nodes[i] = d;
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += kRebuildWG) {
        list[i] = (int32_t)(i + 1);
        bvht_tnode l;
        const float* b = bounds + 6 * (size_t)i;
        l.bmin[0] = b[0]; l.bmin[1] = b[1]; l.bmin[2] = b[2];
        l.bmax[0] = b[3]; l.bmax[1] = b[4]; l.bmax[2] = b[5];
        l.left_right = 0;
        l.blas = i;
        nodes[i + 1] = l;
    }
    if (threadIdx.x == 0) {
        sh_a = 0;
        sh_count = (int32_t)n;
        sh_used = (int32_t)n + 1;
        sh_fail = 0;
    }
    __syncthreads();
    if (WAVE || (n >= 1 && n <= 64)) {
        if (threadIdx.x < 64)
            wave_rebuild_loop(bounds, nodes, list, (int32_t)n, &sh_a, &sh_used, &sh_fail, &sh_depth);
        __syncthreads();
        if (threadIdx.x == 0)
            meta_out(meta, (uint32_t)sh_used, sh_fail ? 0u : sh_depth, sh_fail ? 1u : 0u);
        return;
    }
    if constexpr (!WAVE) {
    if (n <= kRebuildLds) {
        block_rebuild_loop(bounds, nodes, meta, (int32_t)n, lds);
        return;
    }
    int32_t b0 = block_best_match(nodes, list, sh_count, sh_a, s_val, s_idx);
    if (threadIdx.x == 0)
        sh_b = b0;
    __syncthreads();
    while (sh_count > 1) {
        if (sh_b < 0) {  // every candidate area was >= f32::MAX (the reference panics)
            if (threadIdx.x == 0)
                sh_fail = 1;
            __syncthreads();
            break;
        }
        int32_t c = block_best_match(nodes, list, sh_count, sh_b, s_val, s_idx);
        if (threadIdx.x == 0) {
            int32_t a = sh_a, b = sh_b;
            if (a == c) {
                int32_t ia = list[a], ib = list[b];
                bvht_tnode na = nodes[ia], nb = nodes[ib];
                bvht_tnode nn;
                nn.left_right = (uint32_t)ia + ((uint32_t)ib << 16);
                V3 mn = min3(mk3(na.bmin[0], na.bmin[1], na.bmin[2]), mk3(nb.bmin[0], nb.bmin[1], nb.bmin[2]));
                V3 mx = max3(mk3(na.bmax[0], na.bmax[1], na.bmax[2]), mk3(nb.bmax[0], nb.bmax[1], nb.bmax[2]));
                nn.bmin[0] = mn.x; nn.bmin[1] = mn.y; nn.bmin[2] = mn.z;
                nn.bmax[0] = mx.x; nn.bmax[1] = mx.y; nn.bmax[2] = mx.z;
                nn.blas = 0;
                nodes[sh_used] = nn;
                list[a] = sh_used;
                sh_used += 1;
                list[b] = list[sh_count - 1];
                sh_count -= 1;
                sh_merged = 1;
            } else {
                sh_a = b;
                sh_b = c;
                sh_merged = 0;
            }
        }
        __syncthreads();
        if (sh_merged) {
            int32_t nb = block_best_match(nodes, list, sh_count, sh_a, s_val, s_idx);
            if (threadIdx.x == 0)
                sh_b = nb;
            __syncthreads();
        }
    }
    // more than kRebuildLds objects
    if (threadIdx.x == 0) {
        if (!sh_fail) {
            nodes[0] = nodes[list[sh_a]];
            // depth: iterative walk, list[] reused as (node, level) stack
            uint32_t best = 0, sp = 0;
            uint32_t* st = reinterpret_cast<uint32_t*>(list);
            st[sp++] = 0;
            st[sp++] = 1;
            while (sp) {
                uint32_t lvl = st[--sp], ni = st[--sp];
                best = max(best, lvl);
                uint32_t lr = nodes[ni].left_right;
                if (lr != 0 && sp + 4 <= 2 * max(n, 4u) + 4) {  // the list holds 2 max(n, 4) + 4 words
                    st[sp++] = lr >> 16;
                    st[sp++] = lvl + 1;
                    st[sp++] = lr & 0xFFFFu;
                    st[sp++] = lvl + 1;
                }
            }
            meta[0] = (uint32_t)sh_used;
            meta[1] = best;
            meta[2] = 0;
        } else {
            meta[0] = (uint32_t)sh_used;
            meta[1] = 0;
            meta[2] = 1;
        }
    }
    }
}


}  // namespace bvht
