// GPU BVH build: scene bounds -> circumscribed cube -> Morton codes -> stable
// radix sort -> PLOC passes -> pre-order flatten -> traversal layout.
//
// Float arithmetic follows the reference's evaluation order exactly (built with
// -ffp-contract=off, std::min/std::max written as the same compares), so codes,
// cluster boxes and the flattened node array are bit-identical to a serial run
// of bvh.cpp / scene.cpp on the same input.
#include <cmath>
#include <cstring>

#include "rtq_internal.hpp"

namespace rtq {
namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ float smin(float a, float b) { return (b < a) ? b : a; }
__device__ __forceinline__ float smax(float a, float b) { return (a < b) ? b : a; }
__host__ __device__ __forceinline__ float canon0(float x) { return x == 0.0f ? 0.0f : x; }

// glm mat4 * vec4 as evaluated at bvh.cpp:238-240 / triangle.cpp:33:
// (m0*x + m1*y) + (m2*z + m3*w), column-major m.
__device__ __forceinline__ void mat_vec(const float* m, float x, float y, float z, float w,
                                        float* out) {
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        float a0 = m[0 + r] * x + m[4 + r] * y;
        float a1 = m[8 + r] * z + m[12 + r] * w;
        out[r] = a0 + a1;
    }
}

__device__ __forceinline__ void world_vertex(const DevModel& md, const rtq_vec4& p, float* out) {
    float m[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) m[i] = md.m[i];
    mat_vec(m, p.x, p.y, p.z, p.w, out);
}

// Triangle box, bvh.cpp:383-399.
__device__ __forceinline__ void tri_box(const rtq_triangle& t, const DevModel& md, float* lo, float* hi) {
    float p0[3], p1[3], p2[3];
    world_vertex(md, t.p0, p0);
    world_vertex(md, t.p1, p1);
    world_vertex(md, t.p2, p2);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        lo[k] = smin(p0[k], smin(p1[k], p2[k]));
        hi[k] = smax(p0[k], smax(p1[k], p2[k]));
    }
}

// ------------------------------------------------------------- refit

// Leaf cluster c < N keeps its triangle; its box is the triangle's box for the
// current vertices (bvh.cpp:383-399), as k_leaf_init computes it.
__global__ __launch_bounds__(kThreads) void k_refit_leaves(const rtq_triangle* __restrict__ tris,
                                                           const DevModel* __restrict__ models,
                                                           const uint32_t* __restrict__ ctri, uint32_t n,
                                                           rtq_aabb* __restrict__ cbox) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const rtq_triangle t = tris[ctri[i]];
    float lo[3], hi[3];
    tri_box(t, models[t.model_id], lo, hi);
    rtq_aabb a{};
    for (int k = 0; k < 3; ++k) { a.min[k] = lo[k]; a.max[k] = hi[k]; }
    cbox[i] = a;
}

// A merged cluster's box: the merge of the children's (left operand first, as
// k_ploc_merge).
__device__ __forceinline__ rtq_aabb merged_box(const rtq_aabb& l, const rtq_aabb& r) {
    rtq_aabb a{};
    for (int k = 0; k < 3; ++k) {
        a.min[k] = smin(l.min[k], r.min[k]);
        a.max[k] = smax(l.max[k], r.max[k]);
    }
    return a;
}

// Merged clusters [first, first + count) of one PLOC pass.
__global__ __launch_bounds__(kThreads) void k_refit_merge(uint32_t first, uint32_t count,
                                                          const uint32_t* __restrict__ cleft,
                                                          const uint32_t* __restrict__ cright,
                                                          rtq_aabb* __restrict__ cbox) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i < count) cbox[first + i] = merged_box(cbox[cleft[first + i]], cbox[cright[first + i]]);
}

// The boxes of one middle subtree per workgroup (one wave), the deepest level
// first, from the list its placement left.  260,642 triangles with 17 passes
// below the top ones: a refit and its rays 292 us with a launch per pass, 263 us
// now.
__global__ __launch_bounds__(kSubThreads) void k_refit_subtrees(const uint2* __restrict__ roots,
                                                                const uint32_t* __restrict__ list,
                                                                const uint4* __restrict__ placed,
                                                                const uint32_t* __restrict__ cleft,
                                                                const uint32_t* __restrict__ cright, rtq_aabb* cbox) {
    if (blockIdx.x >= roots[0].x) return;
    const uint2 root = roots[1 + blockIdx.x];
    levels_up(list + placed[root.x].y, root.y,
              [&](uint32_t c) { cbox[c] = merged_box(cbox[cleft[c]], cbox[cright[c]]); });
}

// The passes at the top of the tree in one workgroup, in build order,
// with the boxes of their clusters [c_lo, nc) in LDS (a child from an earlier
// pass gives its box from global memory); a barrier between passes, and the
// range's boxes written back at the end.  nc - c_lo <= kLdsClusters.
__global__ __launch_bounds__(kLdsThreads) void k_refit_merge_lds(TopPasses passes, uint32_t c_lo, uint32_t nc,
                                                                 const uint32_t* __restrict__ cleft,
                                                                 const uint32_t* __restrict__ cright,
                                                                 rtq_aabb* __restrict__ cbox) {
    constexpr int kSlots = kLdsClusters / kLdsThreads;
    __shared__ rtq_aabb s_box[kLdsClusters];
    const uint32_t t = threadIdx.x;
    const uint32_t R = nc - c_lo;
    uint32_t L[kSlots], Rc[kSlots];
#pragma unroll
    for (int q = 0; q < kSlots; ++q) {
        const uint32_t idx = t + kLdsThreads * q;
        L[q] = idx < R ? cleft[c_lo + idx] : 0u;
        Rc[q] = idx < R ? cright[c_lo + idx] : 0u;
    }
    for (uint32_t k = 0; k < passes.n; ++k) {
        const uint2 p = passes[k];
#pragma unroll
        for (int q = 0; q < kSlots; ++q) {
            const uint32_t idx = t + kLdsThreads * q, c = c_lo + idx;
            if (idx >= R || c < p.x || c >= p.x + p.y) continue;
            const rtq_aabb l = L[q] >= c_lo ? s_box[L[q] - c_lo] : cbox[L[q]];
            const rtq_aabb r = Rc[q] >= c_lo ? s_box[Rc[q] - c_lo] : cbox[Rc[q]];
            s_box[idx] = merged_box(l, r);
        }
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < kSlots; ++q) {
        const uint32_t idx = t + kLdsThreads * q;
        if (idx < R) cbox[c_lo + idx] = s_box[idx];
    }
}

// ------------------------------------------------------------- top of the tree

// One thread: BFS from the root over internal-node refs, at most kTopNodes
// nodes.  A child's slot is its position in the BFS queue, known when it is
// appended, so each node is read once and written with its refs into the set
// already rewritten to kTopBit | slot (leaf refs and refs leaving the set
// unchanged).
// One wave, level by level: lane l holds BFS slot l.  A level's lanes load
// their nodes together, then number their internal children in (slot, left
// before right) order with a wave prefix sum, which is the order a FIFO
// breadth-first walk appends them; children past kTopNodes keep their refs.
static_assert(kTopNodes <= 64, "one lane per top-of-tree slot");
// A second workgroup, if launched, writes the host's words: the scene's box, and
// after a build (n_blocks > 0) the maximum of block_depth.
struct BuildReport {
    rtq_aabb box;
    uint32_t depth;
};
constexpr int kTopThreads = 1024;
__global__ __launch_bounds__(kTopThreads) void k_top_nodes(const float4* __restrict__ nodes, float4* __restrict__ top,
                                                           const uint32_t* __restrict__ block_depth, uint32_t n_blocks,
                                                           const rtq_aabb* __restrict__ bounds,
                                                           BuildReport* __restrict__ host) {
    if (blockIdx.x == 1) {
        __shared__ uint32_t s_max[kTopThreads / 64];
        uint32_t m = 0;
        for (uint32_t i = threadIdx.x; i < n_blocks; i += kTopThreads) m = max(m, block_depth[i]);
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) m = max(m, (uint32_t)__shfl_xor(m, d, 64));
        if ((threadIdx.x & 63) == 0) s_max[threadIdx.x / 64] = m;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (uint32_t w = 1; w < kTopThreads / 64; ++w) m = max(m, s_max[w]);
            host->box = bounds[0];
            host->depth = m;
        }
        return;
    }
    if (threadIdx.x >= 64) return;
    __shared__ uint32_t s_q[64];
    const uint32_t lane = threadIdx.x;
    uint32_t node = 0;                 // node index of slot `lane` once its level is reached
    uint32_t begin = 0, end = 1;       // the current level's slots
    while (begin < end) {
        const bool mine = lane >= begin && lane < end;
        float4 a{}, b{}, c{}, w{};
        uint32_t r0 = kLeafBit, r1 = kLeafBit;
        if (mine) {
            const float4* src = nodes + 4ull * node;
            a = src[0];
            b = src[1];
            c = src[2];
            w = src[3];
            r0 = __float_as_uint(w.x);
            r1 = __float_as_uint(w.y);
        }
        const uint32_t k0 = (r0 & kLeafBit) ? 0u : 1u, k1 = (r1 & kLeafBit) ? 0u : 1u;
        uint32_t incl = k0 + k1;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(incl, d, 64);
            if (lane >= (uint32_t)d) incl += o;
        }
        const uint32_t total = __shfl(incl, 63, 64);
        const uint32_t s0 = end + incl - (k0 + k1), s1 = s0 + k0;
        if (k0 && s0 < kTopNodes) {
            s_q[s0] = r0;
            r0 = kTopBit | s0;
        }
        if (k1 && s1 < kTopNodes) {
            s_q[s1] = r1;
            r1 = kTopBit | s1;
        }
        if (mine) {
            w.x = __uint_as_float(r0);
            w.y = __uint_as_float(r1);
            float4* dst = top + 4ull * lane;
            dst[0] = a;
            dst[1] = b;
            dst[2] = c;
            dst[3] = w;
        }
        __syncthreads();
        const uint32_t next = min(end + total, kTopNodes);
        if (lane >= end && lane < next) node = s_q[lane];
        __syncthreads();
        begin = end;
        end = next;
    }
}

// ------------------------------------------------------------- scene bounds

__global__ __launch_bounds__(kThreads) void k_bounds_partial(const rtq_triangle* __restrict__ tris,
                                                             const DevModel* __restrict__ models,
                                                             uint32_t n, float* __restrict__ partial) {
    __shared__ float s[6][kThreads];
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < n; i += gridDim.x * kThreads) {
        float a[3], b[3];
        tri_box(tris[i], models[tris[i].model_id], a, b);
#pragma unroll
        for (int k = 0; k < 3; ++k) { lo[k] = smin(lo[k], a[k]); hi[k] = smax(hi[k], b[k]); }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) { s[k][threadIdx.x] = lo[k]; s[3 + k][threadIdx.x] = hi[k]; }
    __syncthreads();
    for (int w = kThreads / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                s[k][threadIdx.x] = smin(s[k][threadIdx.x], s[k][threadIdx.x + w]);
                s[3 + k][threadIdx.x] = smax(s[3 + k][threadIdx.x], s[3 + k][threadIdx.x + w]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) partial[blockIdx.x * 6 + threadIdx.x] = s[threadIdx.x][0];
}

// Reduces the partial boxes, then (one thread) the circumscribed cube of
// bvh.cpp:253-303.  out[0] = scene box, out[1] = cube.
__global__ __launch_bounds__(kThreads) void k_bounds_final(const float* __restrict__ partial, uint32_t nb,
                                                           uint32_t n, uint32_t pad_origin,
                                                           rtq_aabb* __restrict__ out) {
    __shared__ float s[6][kThreads];
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t b = threadIdx.x; b < nb; b += kThreads) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lo[k] = smin(lo[k], partial[b * 6 + k]);
            hi[k] = smax(hi[k], partial[b * 6 + 3 + k]);
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) { s[k][threadIdx.x] = lo[k]; s[3 + k][threadIdx.x] = hi[k]; }
    __syncthreads();
    for (int w = kThreads / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                s[k][threadIdx.x] = smin(s[k][threadIdx.x], s[k][threadIdx.x + w]);
                s[3 + k][threadIdx.x] = smax(s[3 + k][threadIdx.x], s[3 + k][threadIdx.x + w]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    rtq_aabb b{};
    for (int k = 0; k < 3; ++k) { b.min[k] = s[k][0]; b.max[k] = s[3 + k][0]; }
    if (pad_origin && n < 65536u) {
        for (int k = 0; k < 3; ++k) { b.max[k] = smax(b.max[k], 0.0f); b.min[k] = smin(b.min[k], 0.0f); }
    }
    for (int k = 0; k < 3; ++k) { b.min[k] = canon0(b.min[k]); b.max[k] = canon0(b.max[k]); }
    out[0] = b;
    rtq_aabb c = b;
    float dist_x = b.max[0] - b.min[0];
    float dist_y = b.max[1] - b.min[1];
    float dist_z = b.max[2] - b.min[2];
    float max_dist = 0.0f;
    int axis;
    if (dist_x > max_dist) { max_dist = dist_x; axis = 0; }
    else if (dist_y > max_dist) { max_dist = dist_y; axis = 1; }
    else { max_dist = dist_z; axis = 2; }
    float delta;
    if (axis == 0) {
        delta = (max_dist - dist_y) / 2.0f; c.max[1] += delta; c.min[1] -= delta;
        delta = (max_dist - dist_z) / 2.0f; c.max[2] += delta; c.min[2] -= delta;
    } else if (axis == 1) {
        delta = (max_dist - dist_x) / 2.0f; c.max[0] += delta; c.min[0] -= delta;
        delta = (max_dist - dist_z) / 2.0f; c.max[2] += delta; c.min[2] -= delta;
    } else {
        delta = (max_dist - dist_x) / 2.0f; c.max[0] += delta; c.min[0] -= delta;
        delta = (max_dist - dist_y) / 2.0f; c.max[1] += delta; c.min[1] -= delta;
    }
    out[1] = c;
}

// ------------------------------------------------------------- Morton codes

__device__ __forceinline__ uint32_t expand_bits(uint32_t v) {
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

__device__ __forceinline__ uint32_t quantize10(float x) {
    x = smin(smax(x * 1024.0f, 0.0f), 1023.0f);
    if (x != x) return 0u;   // zero-extent axis: the reference cast is undefined
    return (uint32_t)x;
}

// bvh.cpp:305-372 for one triangle.
__global__ __launch_bounds__(kThreads) void k_morton(const rtq_triangle* __restrict__ tris,
                                                     const DevModel* __restrict__ models, uint32_t n,
                                                     const rtq_aabb* __restrict__ bounds,
                                                     uint32_t* __restrict__ codes,
                                                     uint32_t* __restrict__ idx) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const rtq_aabb cube = bounds[1];
    const rtq_triangle t = tris[i];
    const DevModel& md = models[t.model_id];
    const float third = 1.0f / 3.0f;
    float ms[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) ms[k] = third * md.m[k];
    float sx = (t.p0.x + t.p1.x) + t.p2.x;
    float sy = (t.p0.y + t.p1.y) + t.p2.y;
    float sz = (t.p0.z + t.p1.z) + t.p2.z;
    float sw = (t.p0.w + t.p1.w) + t.p2.w;
    float c[3];
    mat_vec(ms, sx, sy, sz, sw, c);
    uint32_t q[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float len = cube.max[k] - cube.min[k];
        q[k] = quantize10((c[k] - cube.min[k]) / len);
    }
    codes[i] = (expand_bits(q[0]) << 2) | (expand_bits(q[1]) << 1) | expand_bits(q[2]);
    if (idx) idx[i] = i;
}

// --------------------------------------------------------------------- PLOC

struct alignas(8) Box6 {   // three 8-B words, so LDS reads take 8 B at a time
    float lo[3], hi[3];
};

__device__ __forceinline__ float merged_sa(const Box6& a, const Box6& b) {
    // AABB::merge then AABB::getSurfaceArea (bvh.cpp:378-381, 401-413)
    float dx = smax(a.hi[0], b.hi[0]) - smin(a.lo[0], b.lo[0]);
    float dy = smax(a.hi[1], b.hi[1]) - smin(a.lo[1], b.lo[1]);
    float dz = smax(a.hi[2], b.hi[2]) - smin(a.lo[2], b.lo[2]);
    return 2.0f * ((dx * dy + dy * dz) + dz * dx);
}

// Half of merged_sa for the comparisons of the neighbour search: the doubling
// is exact, and the minimum and maximum instructions differ from the compares
// of smin / smax in the sign of a zero only, so the order of two clusters is
// the same (vertices are finite).  17 instead of 34 instructions per neighbour
// with the search's loop unrolled (the first pass of 2M clusters spends 35 us
// in it, close to the rate of its instructions; 27 us wait in the look-back).
__device__ __forceinline__ float vmin(float a, float b) {
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float vmax(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float merge_cost(const Box6& a, const Box6& b) {
    const float dx = vmax(a.hi[0], b.hi[0]) - vmin(a.lo[0], b.lo[0]);
    const float dy = vmax(a.hi[1], b.hi[1]) - vmin(a.lo[1], b.lo[1]);
    const float dz = vmax(a.hi[2], b.hi[2]) - vmin(a.lo[2], b.lo[2]);
    return (dx * dy + dy * dz) + dz * dx;
}

// A box past the ends of a list: its merge cost with any box is infinite, so
// the search never takes it.
__device__ __forceinline__ Box6 far_box() {
    constexpr float f = 3.0e38f;
    return Box6{{-f, -f, -f}, {f, f, f}};
}

// The nearer of (best, arg) and the N boxes from w on, whose list positions are
// j, j + 1, ...; the first one on ties.
template <int N>
__device__ __forceinline__ void nearest_of(const Box6& b, const Box6* w, int j, float& best, uint32_t& arg) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const float d = merge_cost(b, w[k]);
        const bool take = d < best;
        best = take ? d : best;
        arg = take ? (uint32_t)(j + k) : arg;
    }
}

// Search radius of the reference (bvh.hpp:66): its window is unrolled.
constexpr int kRefRadius = 16;

// Nearest neighbour in the window [i - r, i + r] of list position i, the
// lowest one on ties (bvh.cpp:193-210); w is the box at i - r, with far boxes
// beside the list's ends when r is kRefRadius, else the list is [lo, hi).
__device__ __forceinline__ uint32_t nearest_in_window(const Box6* w, int i, int r, int lo, int hi) {
    float best = INFINITY;
    uint32_t arg = kNone;
    if (r == kRefRadius) {
        const Box6 b = w[kRefRadius];
        nearest_of<kRefRadius>(b, w, i - kRefRadius, best, arg);
        nearest_of<kRefRadius>(b, w + kRefRadius + 1, i + 1, best, arg);
    } else {
        const Box6 b = w[r];
        const int start = max(i - r, lo), end = min(i + r + 1, hi);
        for (int j = start; j < end; ++j) {
            const float d = merge_cost(b, w[j - i + r]);
            const bool take = j != i && d < best;
            best = take ? d : best;
            arg = take ? (uint32_t)j : arg;
        }
    }
    return arg;
}

// plocPreprocessing, bvh.cpp:26-46: the clusters of one triangle each (the merges
// write everything of the others but the root's parent), the list they start as
// and, unless null, the fused passes' state (kPlocHeadWords words).
constexpr uint32_t kPlocBatch = 16;
constexpr uint32_t kPlocErrWord = 8, kTailCountWord = 9;   // errors and tail pass count, after the state
constexpr uint32_t kPlocHeadWords = 16 + 4 * kPlocBatch;   // state (8), those two (8), pass log, then the tail's log
constexpr uint32_t kTailPeek = 128;                        // tail log entries that reach the host with them
constexpr uint32_t kPlocReportWords = kPlocHeadWords + 4 * kTailPeek;
static_assert(kPlocReportWords <= kReportWords && kPlocReportWords <= 1024, "one word per thread of the tail");

__global__ __launch_bounds__(kThreads) void k_leaf_init(const rtq_triangle* __restrict__ tris,
                                                        const DevModel* __restrict__ models,
                                                        const uint32_t* __restrict__ sorted_idx,
                                                        uint32_t n, rtq_aabb* __restrict__ cbox,
                                                        uint32_t* __restrict__ ctri,
                                                        uint32_t* __restrict__ ccount,
                                                        uint32_t* __restrict__ cleft,
                                                        uint32_t* __restrict__ cright,
                                                        uint32_t* __restrict__ cparent,
                                                        uint32_t* __restrict__ c_in,
                                                        Box6* __restrict__ b_in, uint32_t* __restrict__ state) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i == 0) cparent[2 * n - 2] = kNone;
    if (state && i < 16) state[i] = i < 2 ? n : 0u;
    if (i >= n) return;
    const uint32_t ti = sorted_idx[i];
    const rtq_triangle t = tris[ti];
    Box6 b;
    tri_box(t, models[t.model_id], b.lo, b.hi);
    rtq_aabb a{};
    for (int k = 0; k < 3; ++k) { a.min[k] = b.lo[k]; a.max[k] = b.hi[k]; }
    cbox[i] = a;
    ctri[i] = ti;
    ccount[i] = 1;
    cleft[i] = kNone;
    cright[i] = kNone;
    c_in[i] = i;
    b_in[i] = b;
}

// plocNearestNeighborSearch, bvh.cpp:193-210: window [i-r, i+r] of the active
// cluster list staged through LDS; strict '<' keeps the lowest j on ties.
// PLOC state on the device, so passes can be queued without reading the
// cluster count back: state[0] = clusters this pass, state[1] = clusters
// made so far (the next merge id).  Kernels are launched for an upper bound.
__global__ __launch_bounds__(kThreads) void k_ploc_nn(const Box6* __restrict__ b_in,
                                                      const uint32_t* __restrict__ state, uint32_t radius,
                                                      uint32_t* __restrict__ nn) {
    __shared__ Box6 s_box[kThreads + 64];
    const uint32_t iter = state[0];
    const uint32_t base = blockIdx.x * kThreads;
    const uint32_t lo = base > radius ? base - radius : 0u;
    const uint32_t hi = min(iter, base + kThreads + radius);
    for (uint32_t j = lo + threadIdx.x; j < hi; j += kThreads) s_box[j - lo] = b_in[j];
    __syncthreads();
    const uint32_t i = base + threadIdx.x;
    if (i >= iter) return;
    const Box6 bi = s_box[i - lo];
    const uint32_t start = i > radius ? i - radius : 0u;
    const uint32_t end = min(i + radius + 1, iter);
    float best = INFINITY;
    uint32_t arg = kNone;
    for (uint32_t j = start; j < end; ++j) {
        if (j == i) continue;
        float d = merged_sa(bi, s_box[j - lo]);
        if (d < best) { best = d; arg = j; }
    }
    if (arg != kNone) nn[i] = arg;
}

// Per position: x = 1 if this position starts a merge (mutual pair, lower
// index), y = 1 if a cluster stays at this position after merging.
__global__ __launch_bounds__(kThreads) void k_ploc_flags(const uint32_t* __restrict__ nn,
                                                         const uint32_t* __restrict__ state, uint32_t bound,
                                                         uint2* __restrict__ flags) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    const uint32_t iter = state[0];
    if (i >= bound) return;
    if (i >= iter) {
        flags[i] = make_uint2(0u, 0u);  // past this pass's clusters: counted as nothing
        return;
    }
    const uint32_t j = nn[i];
    const bool mutual = (j < iter) && (j != i) && nn[j] == i;
    flags[i] = make_uint2((mutual && i < j) ? 1u : 0u, (mutual && j < i) ? 0u : 1u);
}

// plocMerging + plocCompaction (bvh.cpp:150-191): merged cluster ids are
// n_total + (number of merges at lower positions), deterministic.
__global__ __launch_bounds__(kThreads) void k_ploc_merge(
    const uint32_t* __restrict__ state, const uint32_t* __restrict__ nn, const uint2* __restrict__ flags,
    const uint2* __restrict__ offs, const uint32_t* __restrict__ c_in, const Box6* __restrict__ b_in,
    uint32_t* __restrict__ c_out, Box6* __restrict__ b_out, rtq_aabb* __restrict__ cbox,
    uint32_t* __restrict__ cleft, uint32_t* __restrict__ cright, uint32_t* __restrict__ cparent,
    uint32_t* __restrict__ ccount, uint32_t* __restrict__ ctri, uint32_t* __restrict__ ctrav, uint32_t nt,
    uint32_t max_leaf) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    const uint32_t iter = state[0], n_total = state[1];
    if (i >= iter) return;
    const uint2 f = flags[i];
    if (!f.y) return;
    const uint2 o = offs[i];
    uint32_t cid = c_in[i];
    Box6 b = b_in[i];
    if (f.x) {
        const uint32_t j = nn[i];
        const uint32_t cj = c_in[j];
        const Box6 bj = b_in[j];
        const uint32_t id = n_total + o.x;
        Box6 m;
        rtq_aabb a{};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            m.lo[k] = smin(b.lo[k], bj.lo[k]);
            m.hi[k] = smax(b.hi[k], bj.hi[k]);
            a.min[k] = m.lo[k];
            a.max[k] = m.hi[k];
        }
        cbox[id] = a;
        cleft[id] = cid;
        cright[id] = cj;
        cparent[cid] = id;
        cparent[cj] = id;
        const uint32_t count = ccount[cid] + ccount[cj];
        ccount[id] = count;
        ctrav[id] = (cid < nt ? 0u : ctrav[cid]) + (cj < nt ? 0u : ctrav[cj]) + (count > max_leaf ? 1u : 0u);
        ctri[id] = 0;
        cid = id;
        b = m;
    }
    c_out[o.y] = cid;
    b_out[o.y] = b;
}

// --------------------------------------------------------------- flattening

// End of a pass: log (first merge id, merges, clusters) and move the state on.
__global__ void k_ploc_advance(const uint2* __restrict__ tot, uint32_t* __restrict__ state,
                               uint4* __restrict__ pass_log, uint32_t slot) {
    const uint2 t = *tot;
    pass_log[slot] = make_uint4(state[1], t.x, state[0], 0u);
    state[1] += t.x;
    state[0] = t.y;
}

// ------------------------------------------------------- fused PLOC passes
//
// The single-launch PLOC iteration of PLOC++ (Benthin, Meister, Barczak,
// Mohanty & Wald, HPG 2022), replacing the neighbour search, flag, scan (two
// or three launches), merge and state-update launches of a pass.  Workgroup w
// owns the T = kPassThreads - 2r positions [wT, wT + T) of the active list. It
// stages the boxes of [wT - 2r, wT + T + 2r) in LDS and finds the nearest
// neighbour of every position of [wT - r, wT + T + r), so the partner of each
// owned position has its own neighbour at hand.  It then sets the merge and
// stay flags of its positions, scans them inside the workgroup and gets the
// counts before its tile by decoupled look-back over per-tile status words
// (Merrill & Garland, "Single-pass Parallel Prefix Scan with Decoupled
// Look-back", 2016).  Tiles are numbered by take_tile; a tile that has published
// nothing for long (kTilePatience) is counted by the wave that waits for it
// (ploc_tile_counts).  A status word carries its counts, so it is stored
// and loaded with relaxed device-scope atomics: acquire / release would add an
// L2 write-back or invalidate per poll.  Each position goes through the arithmetic of
// k_ploc_nn, k_ploc_flags and k_ploc_merge, so the clusters are identical.
//
// Passes with at most kTailMax clusters (33 of the 61 passes of a 2M-triangle
// terrain) run in one workgroup, k_ploc_tail, the whole list held in LDS.
//
// Device state per pass slot: {clusters, next merge id, list buffer 0/1, 0};
// a pass reads slot k & 1 and writes slot (k + 1) & 1, so no workgroup reads
// a word another one writes.

constexpr int kPassThreads = 512;
constexpr int kTailThreads = 1024;
constexpr uint32_t kTailMax = 4 * kTailThreads;   // 4 positions per tail thread
constexpr uint64_t kTileAgg = 1ull << 62;         // tile status: own counts published
constexpr uint64_t kTilePre = 2ull << 62;         // tile status: counts through this tile
constexpr uint64_t kTileState = 3ull << 62;

enum : uint32_t { kPlocErrNoNeighbour = 1, kPlocErrBound = 2, kPlocErrNoMerge = 4 };

struct PlocLists {
    uint32_t* c[2];
    Box6* b[2];
};

struct PlocClusters {
    rtq_aabb* box;
    uint32_t *left, *right, *parent, *count, *tri, *trav;
    uint32_t n_tris, max_leaf;
};

// Triangles and binary traversal nodes below a cluster.
__device__ __forceinline__ uint2 ploc_below(const PlocClusters& cl, uint32_t c) {
    return make_uint2(cl.count[c], c < cl.n_tris ? 0u : cl.trav[c]);
}
__device__ __forceinline__ uint2 ploc_below_merged(const PlocClusters& cl, uint2 a, uint2 b) {
    const uint32_t count = a.x + b.x;
    return make_uint2(count, a.y + b.y + (count > cl.max_leaf ? 1u : 0u));
}

__device__ __forceinline__ uint64_t tile_word(uint64_t st, uint32_t merges, uint32_t stays) {
    return st | ((uint64_t)merges << 32) | stays;
}

// Exclusive sum over the workgroup; `total` is the workgroup's sum.  Every
// thread calls it; s_w holds one word per wave.
template <int THREADS>
__device__ __forceinline__ uint32_t block_exclusive_sum(uint32_t v, uint32_t* s_w, uint32_t& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(incl, d, 64);
        if (lane >= d) incl += o;
    }
    if (lane == 63) s_w[wave] = incl;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < THREADS / 64; ++w) {
        const uint32_t x = s_w[w];
        before += (w < wave) ? x : 0u;
        all += x;
    }
    total = all;
    return before + incl - v;
}

// Merge of clusters cid (box b) and cj (box bj) into cluster id, as
// k_ploc_merge writes it; b becomes the merged box.
// `below`: what lies below it (ploc_below_merged).
__device__ __forceinline__ void ploc_merge_store(const PlocClusters& cl, uint32_t id, uint32_t cid, uint32_t cj,
                                                 uint2 below, Box6& b, const Box6& bj) {
    Box6 m;
    rtq_aabb a{};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        m.lo[k] = smin(b.lo[k], bj.lo[k]);
        m.hi[k] = smax(b.hi[k], bj.hi[k]);
        a.min[k] = m.lo[k];
        a.max[k] = m.hi[k];
    }
    cl.box[id] = a;
    cl.left[id] = cid;
    cl.right[id] = cj;
    cl.parent[cid] = id;
    cl.parent[cj] = id;
    cl.count[id] = below.x;
    cl.trav[id] = below.y;
    cl.tri[id] = 0;
    b = m;
}

__device__ __forceinline__ void ploc_merge_write(const PlocClusters& cl, uint32_t id, uint32_t cid, uint32_t cj,
                                                 Box6& b, const Box6& bj) {
    // the counts are read before any store: the arrays may alias as far as
    // the compiler knows, and a load after a store waits for the store
    const uint2 below = ploc_below_merged(cl, ploc_below(cl, cid), ploc_below(cl, cj));
    ploc_merge_store(cl, id, cid, cj, below, b, bj);
}

struct PlocPassArgs {
    const uint32_t* st_in;
    uint32_t* st_out;
    uint32_t bound;       // clusters at the start of the batch: the grid covers them
    uint32_t radius;
    uint32_t* tile_ctr;   // kTicketWords words, zeroed before the pass
    uint64_t* tile_status;// one word per tile, zeroed before the pass
    uint32_t* err;
    uint4* log;           // (first merge id, merges, clusters, 1 if left to the tail)
    PlocLists lists;
    PlocClusters cl;
};

// Merges and stays of the list's positions [first, end), by one wave, from the
// list itself: the counts that the tile which owns them publishes.
__device__ uint2 ploc_tile_counts(const Box6* __restrict__ list, int first, int end, int r, int n) {
    const auto nearest = [&](int i) {
        const Box6 b = list[i];
        float best = INFINITY;
        uint32_t arg = kNone;
        for (int j = max(i - r, 0); j < min(i + r + 1, n); ++j) {
            const float d = merge_cost(b, list[j]);
            const bool take = j != i && d < best;
            best = take ? d : best;
            arg = take ? (uint32_t)j : arg;
        }
        return arg;
    };
    uint2 counts = make_uint2(0u, 0u);
    for (int i0 = first; i0 < end; i0 += 64) {
        const int i = i0 + ((int)threadIdx.x & 63);
        const uint32_t j = i < end ? nearest(i) : kNone;
        const bool mutual = j != kNone && nearest((int)j) == (uint32_t)i;
        counts.x += (uint32_t)__popcll(__ballot(mutual && (uint32_t)i < j));
        counts.y += (uint32_t)__popcll(__ballot(i < end && !(mutual && j < (uint32_t)i)));
    }
    return counts;
}

__global__ __launch_bounds__(kPassThreads) void k_ploc_pass(PlocPassArgs a) {
    __shared__ Box6 s_box[kPassThreads + 64];
    __shared__ uint32_t s_nn[kPassThreads];
    __shared__ uint32_t s_w[kPassThreads / 64];
    __shared__ uint32_t s_hdr[5];  // tile, clusters, next merge id, list buffer, skip
    __shared__ uint32_t s_excl[2]; // merges and stays before the tile
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = (int)a.radius;
    const uint32_t T = (uint32_t)(kPassThreads - 2 * r);
    if (tid == 0) {
        const uint32_t iter = a.st_in[0], n_total = a.st_in[1], cur = a.st_in[2] & 1u;
        uint32_t skip = 0;
        if (__hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 || iter <= kTailMax) {
            skip = 1;
        } else if (iter > a.bound) {
            atomicOr(a.err, kPlocErrBound);
            skip = 1;
        }
        if (skip && blockIdx.x == 0) {  // left to the tail kernel (or stopped): carry the state over
            a.st_out[0] = iter;
            a.st_out[1] = n_total;
            a.st_out[2] = cur;
            *a.log = make_uint4(n_total, 0u, iter, 1u);
        }
        // the grid covers the batch's first pass: only as many workgroups as
        // this pass has tiles take one (the others leave without touching the
        // counter, whose atomics serialise), so the tiles are 0 .. need - 1
        const uint32_t need = (iter + T - 1) / T;
        if (!skip && blockIdx.x >= need) skip = 1;
        const uint32_t tile = skip ? 0u : take_tile(a.tile_ctr);
        s_hdr[0] = tile;
        s_hdr[1] = iter;
        s_hdr[2] = n_total;
        s_hdr[3] = cur;
        s_hdr[4] = skip;
    }
    __syncthreads();
    if (s_hdr[4]) return;
    const uint32_t tile = s_hdr[0], iter = s_hdr[1], n_total = s_hdr[2], cur = s_hdr[3];
    const uint32_t* __restrict__ c_in = a.lists.c[cur];
    const Box6* __restrict__ b_in = a.lists.b[cur];
    const int base = (int)(tile * T);
    const int lo = base - 2 * r;
    for (int q = tid; q < kPassThreads + 2 * r; q += kPassThreads) {
        const int p = lo + q;
        s_box[q] = p >= 0 && p < (int)iter ? b_in[p] : far_box();
    }
    __syncthreads();

    // nearest neighbour of position i = base - r + tid (k_ploc_nn); its box
    // is s_box[tid + r] and the window [i - r, i + r] is s_box[tid .. tid + 2r]
    const int i = base - r + tid;
    {
        uint32_t arg = kNone;
        if (i >= 0 && i < (int)iter) {
            arg = nearest_in_window(s_box + tid, i, r, 0, (int)iter);
            if (arg == kNone) atomicOr(a.err, kPlocErrNoNeighbour);
        }
        s_nn[tid] = arg;
    }
    __syncthreads();

    // flags of the owned positions (k_ploc_flags): the partner j lies in
    // [i - r, i + r], so its neighbour is s_nn[tid + (j - i)]
    const bool owned = tid >= r && tid < r + (int)T && i < (int)iter;
    uint32_t fx = 0, fy = 0, j = kNone;
    if (owned) {
        j = s_nn[tid];
        const bool mutual = j != kNone && s_nn[tid + ((int)j - i)] == (uint32_t)i;
        fx = (mutual && (uint32_t)i < j) ? 1u : 0u;
        fy = (mutual && j < (uint32_t)i) ? 0u : 1u;
    }
    uint32_t total = 0;
    const uint32_t v = (fx << 16) | fy;  // at most kPassThreads of each per tile
    const uint32_t local = block_exclusive_sum<kPassThreads>(v, s_w, total);

    // counts before this tile: decoupled look-back by wave 0
    if (wave == 0) {
        const uint32_t ax = total >> 16, ay = total & 0xFFFFu;
        uint32_t ex = 0, ey = 0;
        if (tile == 0) {
            if (lane == 0)
                __hip_atomic_store(&a.tile_status[0], tile_word(kTilePre, ax, ay), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        } else {
            if (lane == 0)
                __hip_atomic_store(&a.tile_status[tile], tile_word(kTileAgg, ax, ay), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            int64_t top = (int64_t)tile - 1;
            uint32_t polls = 0;
            for (;;) {
                const int64_t idx = top - lane;  // lane 0 = nearest tile
                uint64_t w = kTilePre;           // before tile 0: an empty prefix
                if (idx >= 0)
                    w = __hip_atomic_load(&a.tile_status[idx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                for (uint64_t missing; (missing = __ballot((w & kTileState) == 0)) != 0;) {
                    if (++polls > kTilePatience) {
                        const int m = __ffsll((long long)missing) - 1;
                        const int first = (int)((top - m) * T);   // a whole tile: only the last may be short
                        const uint2 c = ploc_tile_counts(b_in, first, first + (int)T, r, (int)iter);
                        if (lane == m) w = publish_for(&a.tile_status[idx], tile_word(kTileAgg, c.x, c.y));
                    } else {
                        __builtin_amdgcn_s_sleep(1);
                    }
                    if ((w & kTileState) == 0)
                        w = __hip_atomic_load(&a.tile_status[idx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                // nearest tile with counts through it
                const unsigned long long pre = __ballot((w & kTileState) == kTilePre);
                const int stop = pre ? __ffsll((long long)pre) - 1 : 63;
                uint32_t cx = lane <= stop ? (uint32_t)(w >> 32) & 0x3FFFFFFFu : 0u;
                uint32_t cy = lane <= stop ? (uint32_t)w : 0u;
#pragma unroll
                for (int d = 32; d >= 1; d >>= 1) {
                    cx += __shfl_xor(cx, d, 64);
                    cy += __shfl_xor(cy, d, 64);
                }
                ex += cx;
                ey += cy;
                if (pre) break;
                top -= 64;
            }
            if (lane == 0)
                __hip_atomic_store(&a.tile_status[tile], tile_word(kTilePre, ex + ax, ey + ay), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        if (lane == 0) {
            s_excl[0] = ex;
            s_excl[1] = ey;
            if (tile == (iter - 1) / T) {  // the tile holding the last position ends the pass
                a.st_out[0] = ey + ay;
                a.st_out[1] = n_total + ex + ax;
                a.st_out[2] = cur ^ 1u;
                *a.log = make_uint4(n_total, ex + ax, iter, 0u);
            }
        }
    }
    __syncthreads();
    if (!owned || !fy) return;

    // merge and compaction (k_ploc_merge)
    const uint32_t ox = s_excl[0] + (local >> 16), oy = s_excl[1] + (local & 0xFFFFu);
    uint32_t cid = c_in[i];
    Box6 b = s_box[tid + r];
    if (fx) {
        ploc_merge_write(a.cl, n_total + ox, cid, c_in[j], b, s_box[(int)j - lo]);
        cid = n_total + ox;
    }
    a.lists.c[cur ^ 1u][oy] = cid;
    a.lists.b[cur ^ 1u][oy] = b;
}

// Lane l's value from lane l ^ X of its group of four.
template <int X>
__device__ __forceinline__ uint32_t quad_xor(uint32_t v) {
    constexpr int ctrl = X == 1 ? 0xB1 : 0x4E;   // quad_perm [1 0 3 2] or [2 3 0 1]
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xF, 0xF, true);
}

// kRefRadius search of position i by P = 2 or 4 neighbouring lanes, each with a
// part of the window (lane part q before lane part q + 1 in list order).
template <int P>
__device__ __forceinline__ uint32_t nearest_by_lanes(const Box6* w, int i, int q) {
    constexpr int kPart = 2 * kRefRadius / P;
    // the parts before the box, then (one further) those after it
    const int k = -kRefRadius + q * kPart + (q >= P / 2 ? 1 : 0);
    float best = INFINITY;
    uint32_t arg = kNone;
    nearest_of<kPart>(*w, w + k, i + k, best, arg);
#pragma unroll
    for (int x = 1; x < P; x *= 2) {
        const float d = __uint_as_float(x == 1 ? quad_xor<1>(__float_as_uint(best)) : quad_xor<2>(__float_as_uint(best)));
        const uint32_t j = x == 1 ? quad_xor<1>(arg) : quad_xor<2>(arg);
        const bool take = d < best || (d == best && j < arg);
        best = take ? d : best;
        arg = take ? j : arg;
    }
    return arg;
}

// The tail's list in LDS, with its triangle and node counts (no global loads
// between the passes' barriers) and nearest neighbours.
struct TailLists {
    Box6 list[kTailMax + 2 * kRefRadius];   // kRefRadius far boxes, the list's boxes, kRefRadius far boxes
    uint32_t c[kTailMax];
    uint2 n[kTailMax];
    uint16_t nn[kTailMax];
    uint32_t w[64];
};

// Flags, scan, merge and compaction of a list of m clusters whose neighbours
// are found: thread t owns positions t, t + W, .., of W threads, so that
// neighbouring lanes read and write neighbouring entries (four positions in a row
// per thread lie 96 B apart: 4,095 passes of a list that loses one cluster each
// 58.7 ms, 54.8 so).  Returns merges << 16 |
// clusters left.  ONE_WAVE: the first wave alone (m <= 64 K), else every thread
// (two barriers).  A position's own state is read before anything depends on
// it, and by one wave its partner's too, so that a pass waits for LDS three
// times, not once per position and step.
template <int K, bool ONE_WAVE>
__device__ __forceinline__ uint32_t tail_merge(TailLists& L, int tid, uint32_t m, uint32_t n_total,
                                               const PlocClusters& cl) {
    constexpr int W = ONE_WAVE ? 64 : kTailThreads;
    Box6* const s_box = L.list + kRefRadius;
    uint32_t j[K], back[K], f[K], run[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t i = (uint32_t)(tid + W * k);
        j[k] = L.nn[min(i, m - 1)];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        j[k] = min(j[k], m - 1);   // in range also where the search found none (which fails the build)
        back[k] = L.nn[j[k]];
    }
    Box6 ob[K], pb[K];
    uint32_t oc[K], pc[K], opos[K];
    uint2 on[K], pn[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t i = min((uint32_t)(tid + W * k), m - 1);
        ob[k] = s_box[i];
        oc[k] = L.c[i];
        on[k] = L.n[i];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t i = (uint32_t)(tid + W * k);
        const bool mutual = back[k] == i && j[k] != i;
        f[k] = i < m ? ((mutual && i < j[k]) ? 1u << 16 : 0u) | ((mutual && j[k] < i) ? 0u : 1u) : 0u;
    }
#pragma unroll
    for (int k = 0; k < K; ++k)
        if (ONE_WAVE || f[k] >> 16) {
            pb[k] = s_box[j[k]];
            pc[k] = L.c[j[k]];
            pn[k] = L.n[j[k]];
        }
    // flags before each position, and of all
    uint32_t total = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) run[k] = wave_inclusive_sum(f[k]);
    if constexpr (ONE_WAVE) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t here = (uint32_t)__builtin_amdgcn_readlane((int)run[k], 63);
            run[k] += total - f[k];
            total += here;
        }
    } else {
        // the sums of the waves, a lane for each wave's of each k
        constexpr int kWaves = kTailThreads / 64;
        static_assert(K * kWaves == 64, "one lane per sum");
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        if ((tid & 63) == 63)
#pragma unroll
            for (int k = 0; k < K; ++k) L.w[kWaves * k + wave] = run[k];
        __syncthreads();
        const uint32_t w = L.w[tid & 63], through = wave_inclusive_sum(w);
        total = (uint32_t)__builtin_amdgcn_readlane((int)through, 63);
#pragma unroll
        for (int k = 0; k < K; ++k)
            run[k] += (uint32_t)__builtin_amdgcn_readlane((int)(through - w), kWaves * k + wave) - f[k];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        opos[k] = (f[k] & 0xFFFFu) ? run[k] & 0xFFFFu : kNone;
        if (f[k] >> 16) {
            const uint32_t id = n_total + (run[k] >> 16);
            on[k] = ploc_below_merged(cl, on[k], pn[k]);
            ploc_merge_store(cl, id, oc[k], pc[k], on[k], ob[k], pb[k]);
            oc[k] = id;
        }
    }
    // every read of this pass's list is done: by the barrier above, or because
    // one wave's instructions keep their order
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < K; ++k)
        if (opos[k] != kNone) {
            s_box[opos[k]] = ob[k];
            L.c[opos[k]] = oc[k];
            L.n[opos[k]] = on[k];
        }
    if (tid < kRefRadius) s_box[(total & 0xFFFFu) + tid] = far_box();
    return total;
}

// All remaining passes once at most kTailMax clusters are left, in one
// workgroup with the list in LDS (same arithmetic as k_ploc_pass).  Does nothing
// unless 1 < clusters <= kTailMax.
// One CU runs it, so its long passes are bound by the search's instructions
// (merge_cost), its short ones (half of them have under 130 clusters) by a
// pass's chain of dependent steps: up to 512 or 256 clusters a position's window
// is shared by 2 or 4 lanes, and up to 256 the first wave alone flags, scans
// and merges, so that a pass has two barriers.  960 clusters (19 passes): 112
// us before these and the shorter search, 60 now; the last 33 passes of a
// 2M-triangle terrain, whose first ones are long, 228 and 182.
__global__ __launch_bounds__(kTailThreads) void k_ploc_tail(uint32_t* state, uint32_t radius, PlocLists lists,
                                                            PlocClusters cl, uint32_t* host) {
    __shared__ TailLists L;
    __shared__ uint32_t s_hdr[4];
    uint32_t* const err = state + kPlocErrWord;
    uint32_t* const log_count = state + kTailCountWord;
    uint4* const log = reinterpret_cast<uint4*>(state + kPlocHeadWords);
    Box6* const s_box = L.list + kRefRadius;
    const int tid = threadIdx.x;
    const int r = (int)radius;
    if (tid == 0) {
        const uint32_t m0 = state[0];
        s_hdr[0] = m0;
        s_hdr[1] = state[1];
        s_hdr[2] = state[2] & 1u;
        s_hdr[3] = (*err != 0 || m0 <= 1 || m0 > kTailMax) ? 1u : 0u;
        if (s_hdr[3]) *log_count = 0;
    }
    __syncthreads();
    // at the end, the head words and the log's first entries for the host: earlier
    // launches and this workgroup wrote them, so the barrier orders the reads (a
    // device-scope fence writes the L2 back: 4 us of a rebuild of 960 triangles);
    // at device scope, where the error bits are set
    const auto tell = [&]() {
        __syncthreads();
        if (tid < (int)kPlocReportWords)
            host[tid] = __hip_atomic_load(state + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    if (s_hdr[3]) {
        tell();
        return;
    }
    uint32_t m = s_hdr[0], n_total = s_hdr[1];
    const uint32_t cur = s_hdr[2];
    for (uint32_t q = tid; q < m; q += kTailThreads) {
        s_box[q] = lists.b[cur][q];
        const uint32_t c = lists.c[cur][q];
        L.c[q] = c;
        L.n[q] = ploc_below(cl, c);
    }
    if (tid < kRefRadius) {
        L.list[tid] = far_box();
        s_box[m + tid] = far_box();
    }
    __syncthreads();
    uint32_t passes = 0;
    while (m > 1) {
        const bool shared = r == kRefRadius;   // window parts need the unrolled search
        const int split = shared && m <= 256 ? 2 : shared && m <= 512 ? 1 : 0;   // log2 of the lanes per window
        for (int t = tid; t < (int)m << split; t += kTailThreads) {
            const int i = t >> split, q = t & ((1 << split) - 1);
            const uint32_t arg = split == 2   ? nearest_by_lanes<4>(s_box + i, i, q)
                                 : split == 1 ? nearest_by_lanes<2>(s_box + i, i, q)
                                              : nearest_in_window(s_box + i - r, i, r, 0, (int)m);
            if (arg == kNone) atomicOr(err, kPlocErrNoNeighbour);
            if (q == 0) L.nn[i] = (uint16_t)arg;
        }
        __syncthreads();
        const bool one_wave = m <= 256;
        uint32_t total = 0;
        if (m <= 64) {
            if (tid < 64) total = tail_merge<1, true>(L, tid, m, n_total, cl);
        } else if (one_wave) {
            if (tid < 64) total = tail_merge<4, true>(L, tid, m, n_total, cl);
        } else {
            total = tail_merge<4, false>(L, tid, m, n_total, cl);
        }
        if (tid == 0) {
            s_hdr[0] = total;
            log[passes] = make_uint4(n_total, total >> 16, m, 0u);
        }
        __syncthreads();
        total = s_hdr[0];
        const uint32_t merges = total >> 16, stays = total & 0xFFFFu;
        if (merges == 0) {  // uniform: no progress, the build reports it
            if (tid == 0) atomicOr(err, kPlocErrNoMerge);
            break;
        }
        n_total += merges;
        m = stays;
        ++passes;
    }
    if (tid == 0) {
        state[0] = m;
        state[1] = n_total;
        state[3] = L.n[0].y;   // the root's, once one cluster is left
        *log_count = passes;
    }
    tell();
}

// Clusters of one PLOC pass give their children's places (their own are known:
// their parents were created in later passes).
__global__ __launch_bounds__(kThreads) void k_place_pass(uint32_t first, uint32_t count, uint32_t nt,
                                                         const uint32_t* __restrict__ cleft,
                                                         const uint32_t* __restrict__ cright,
                                                         const uint32_t* __restrict__ ccount,
                                                         const uint32_t* __restrict__ ctrav,
                                                         uint4* __restrict__ placed) {
    const uint32_t k = blockIdx.x * kThreads + threadIdx.x;
    if (k >= count) return;
    const uint32_t l = cleft[first + k], r = cright[first + k];
    const Place p = place_of(placed[first + k]);
    const uint32_t lc = ccount[l], lt = l < nt ? 0u : ctrav[l];
    placed[l] = left_place(p);
    placed[r] = right_place(p, lc, lt);
}

// The middle subtrees' clusters (from c_mid on), level by level from the root,
// one subtree per workgroup (one wave).  A level's clusters come with their state
// from the lanes that placed them, through LDS while they fit, else from the
// list and the arrays.  A subtree's list of clusters takes its first-leaf range
// of `list`; the order within a level is free, no result depends on it.
constexpr uint32_t kFront = 256;

__global__ __launch_bounds__(kSubThreads) void k_place_subtrees(uint2* roots, uint32_t c_mid, uint32_t nt,
                                                                const uint32_t* __restrict__ cleft,
                                                                const uint32_t* __restrict__ cright,
                                                                const uint32_t* __restrict__ ccount,
                                                                const uint32_t* __restrict__ ctrav, uint4* placed,
                                                                uint32_t* list_base) {
    __shared__ uint32_t s_id[2][kFront];
    __shared__ uint4 s_at[2][kFront];
    if (blockIdx.x >= roots[0].x) return;
    const uint32_t lane = threadIdx.x;
    const uint32_t root = roots[1 + blockIdx.x].x;
    const uint4 at = placed[root];
    uint32_t* const list = list_base + at.y;
    if (lane == 0) {
        s_id[0][0] = root;
        s_at[0][0] = at;
        list[0] = root | kLevelStart;
    }
    __syncthreads();
    uint32_t begin = 0, end = 1;
    for (uint32_t k = 0; begin < end; ++k) {
        const uint32_t cur = k & 1u, nxt = cur ^ 1u;
        uint32_t n_next = 0;
        for (uint32_t e0 = begin; e0 < end; e0 += kSubThreads) {
            const uint32_t e = e0 + lane;
            uint32_t l = 0, r = 0;
            uint4 lp{}, rp{};
            if (e < end) {
                uint32_t c;
                Place p;
                if (e - begin < kFront) {
                    c = s_id[cur][e - begin];
                    p = place_of(s_at[cur][e - begin]);
                } else {
                    c = list[e] & ~kLevelStart;
                    p = place_of(placed[c]);
                }
                l = cleft[c];
                r = cright[c];
                lp = left_place(p);
                rp = right_place(p, ccount[l], l < nt ? 0u : ctrav[l]);
                placed[l] = lp;
                placed[r] = rp;
            }
            // children of the middle passes to the next level
            const bool bl = l >= c_mid, br = r >= c_mid;
            const uint64_t ml = __ballot(bl), mr = __ballot(br);
            const uint64_t below = (1ull << lane) - 1u;
            const auto put = [&](uint32_t i, uint32_t c, const uint4& v) {
                list[end + i] = i == 0 ? c | kLevelStart : c;
                if (i < kFront) {
                    s_id[nxt][i] = c;
                    s_at[nxt][i] = v;
                }
            };
            if (bl) put(n_next + (uint32_t)__popcll(ml & below), l, lp);
            n_next += (uint32_t)__popcll(ml);
            if (br) put(n_next + (uint32_t)__popcll(mr & below), r, rp);
            n_next += (uint32_t)__popcll(mr);
        }
        __syncthreads();
        begin = end;
        end += n_next;
    }
    if (lane == 0) roots[1 + blockIdx.x].y = end;
}

// The passes at the top of the tree in one workgroup, last pass
// first, with the places of their clusters [c_lo, nc) in LDS: a pass reads and
// writes LDS only, a barrier between passes.  Children from earlier passes get
// their places in global memory, and those from c_mid on are the roots of the
// middle subtrees, listed in roots; the clusters of the range write theirs back
// at the end.  Each thread keeps the child ids and the left child's counts of
// its clusters c_lo + t + kLdsThreads * s in registers.  1 <= nc - c_lo <=
// kLdsClusters.
__global__ __launch_bounds__(kLdsThreads) void k_place_lds(TopPasses passes, uint32_t c_lo, uint32_t nc,
                                                           uint32_t c_mid, uint32_t nt,
                                                           const uint32_t* __restrict__ cleft,
                                                           const uint32_t* __restrict__ cright,
                                                           const uint32_t* __restrict__ ccount,
                                                           const uint32_t* __restrict__ ctrav,
                                                           uint4* __restrict__ placed, uint2* __restrict__ roots) {
    constexpr int kSlots = kLdsClusters / kLdsThreads;
    __shared__ uint4 s_at[kLdsClusters];
    __shared__ uint32_t s_roots;
    const uint32_t t = threadIdx.x;
    const uint32_t R = nc - c_lo;
    uint32_t L[kSlots], Rc[kSlots], LC[kSlots], LT[kSlots];
#pragma unroll
    for (int q = 0; q < kSlots; ++q) {
        const uint32_t idx = t + kLdsThreads * q;
        L[q] = idx < R ? cleft[c_lo + idx] : 0u;
        Rc[q] = idx < R ? cright[c_lo + idx] : 0u;
    }
#pragma unroll
    for (int q = 0; q < kSlots; ++q) {
        // a scene of one triangle has no child
        const bool in = L[q] < nc && t + kLdsThreads * q < R;
        LC[q] = in ? ccount[L[q]] : 0u;
        LT[q] = in && L[q] >= nt ? ctrav[L[q]] : 0u;
    }
    if (t == 0) {  // the root, the last cluster
        s_at[R - 1] = make_uint4(0, 0, 0, 0);
        s_roots = 0;
    }
    __syncthreads();
    for (uint32_t k = passes.n; k > 0; --k) {
        const uint2 p = passes[k - 1];
#pragma unroll
        for (int q = 0; q < kSlots; ++q) {
            const uint32_t idx = t + kLdsThreads * q, c = c_lo + idx;
            if (idx >= R || c < p.x || c >= p.x + p.y) continue;
            const Place at = place_of(s_at[idx]);
            const uint32_t l = L[q], r = Rc[q];
            const uint4 lp = left_place(at), rp = right_place(at, LC[q], LT[q]);
            if (l >= c_lo) s_at[l - c_lo] = lp;
            else placed[l] = lp;
            if (r >= c_lo) s_at[r - c_lo] = rp;
            else placed[r] = rp;
        }
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < kSlots; ++q) {
        const uint32_t idx = t + kLdsThreads * q;
        const bool in = idx < R;
        if (in) placed[c_lo + idx] = s_at[idx];
        const bool bl = in && L[q] >= c_mid && L[q] < c_lo, br = in && Rc[q] >= c_mid && Rc[q] < c_lo;
        const uint64_t ml = __ballot(bl), mr = __ballot(br);
        uint32_t at = 0;
        if ((t & 63u) == 0 && (ml | mr)) at = atomicAdd(&s_roots, (uint32_t)(__popcll(ml) + __popcll(mr)));
        at = 1u + (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
        const uint64_t below = (1ull << (t & 63u)) - 1u;
        if (bl) roots[at + __popcll(ml & below)] = make_uint2(L[q], 0u);
        if (br) roots[at + __popcll(ml) + __popcll(mr & below)] = make_uint2(Rc[q], 0u);
    }
    __syncthreads();
    if (t == 0) roots[0] = make_uint2(s_roots, 0u);
}

// Leaf-ordered traversal triangles, and the depth of each workgroup's deepest
// leaf in block_depth[blockIdx.x] (k_top_nodes takes the maximum: atomics of
// every wave on one word would serialise, tens of thousands of them).
__device__ __forceinline__ void write_leaves(uint32_t n, const uint32_t* __restrict__ ctri,
                                             const uint4* __restrict__ placed, const float4* __restrict__ tri_world,
                                             float4* __restrict__ tris, uint32_t* __restrict__ block_depth) {
    __shared__ uint32_t s_max[kThreads / 64];
    const uint32_t c = blockIdx.x * kThreads + threadIdx.x;
    uint32_t depth = 0;
    if (c < n) {   // the clusters of one triangle
        const uint32_t t = ctri[c];
        const Place p = place_of(placed[c]);
        const uint64_t dst = 3ull * p.first;
        tris[dst + 0] = tri_world[3ull * t + 0];
        tris[dst + 1] = tri_world[3ull * t + 1];
        tris[dst + 2] = tri_world[3ull * t + 2];
        depth = p.depth;
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) depth = max(depth, (uint32_t)__shfl_xor(depth, d, 64));
    if ((threadIdx.x & 63) == 0) s_max[threadIdx.x / 64] = depth;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t m = 0;
        for (uint32_t w = 0; w < kThreads / 64; ++w) m = max(m, s_max[w]);
        block_depth[blockIdx.x] = m;
    }
}

// Reference node array (scene.cpp:189-208): cluster c at its pre-order
// position, children as positions, leaves with their triangle.
__global__ __launch_bounds__(kThreads) void k_write_ref(
    uint32_t n_clusters, const rtq_aabb* __restrict__ cbox, const uint32_t* __restrict__ ctri,
    const uint32_t* __restrict__ cleft, const uint32_t* __restrict__ cright, const uint4* __restrict__ placed,
    rtq_bvh_node* __restrict__ ref) {
    const uint32_t c = blockIdx.x * kThreads + threadIdx.x;
    if (c >= n_clusters) return;
    rtq_bvh_node nd{};
    nd.box = cbox[c];
    nd.box.pad0_ = 0.0f;
    nd.box.pad1_ = 0.0f;
    const bool leaf = cleft[c] == kNone;
    nd.triangle_id = leaf ? ctri[c] : 0u;
    nd.left_child = leaf ? 0u : placed[cleft[c]].x;
    nd.right_child = leaf ? 0u : placed[cright[c]].x;
    nd.pad_ = 0u;
    ref[placed[c].x] = nd;
}

// Traversal node (64 B): child boxes widened outward by the box margin, interleaved as
//   [c0.lo.x c0.hi.x c0.lo.y c0.hi.y] [c0.lo.z c0.hi.z c1.lo.x c1.hi.x]
//   [c1.lo.y c1.hi.y c1.lo.z c1.hi.z] [ref0 ref1 order 0]
// where `order` holds the learned child-order bits (zero until a model is applied).
// One thread per merged cluster c; what a child needs besides its box follows
// from the node's own place and the counts below the children.  2,093,058
// triangles: 150 us when a child's index came from a scan over marks in
// pre-order, 61 us with the counts that PLOC's merges keep (they cost its passes
// nothing).
__device__ __forceinline__ void write_trav(uint32_t c, uint32_t nt, uint32_t nc, uint32_t max_leaf, float pad,
                                           const rtq_aabb* __restrict__ cbox, const uint32_t* __restrict__ cleft,
                                           const uint32_t* __restrict__ cright, const uint32_t* __restrict__ ccount,
                                           const uint32_t* __restrict__ ctrav, const uint4* __restrict__ placed,
                                           float4* __restrict__ nodes, uint4* __restrict__ aux) {
    if (!(ccount[c] > max_leaf || c == nc - 1)) return;
    const uint32_t l = cleft[c], r = cright[c];
    const Place p = place_of(placed[c]);
    const rtq_aabb bl = cbox[l], br = cbox[r];
    const uint32_t lc = ccount[l], rc = ccount[r], lt = l < nt ? 0u : ctrav[l];
    const uint32_t middle = p.first + lc;
    const uint32_t r0 = l >= nt && lc > max_leaf ? p.trav + 1 : leaf_ref(p.first, lc);
    const uint32_t r1 = r >= nt && rc > max_leaf ? p.trav + 1 + lt : leaf_ref(middle, rc);
    float4* o = nodes + 4ull * p.trav;
    o[0] = make_float4(bl.min[0] - pad, bl.max[0] + pad, bl.min[1] - pad, bl.max[1] + pad);
    o[1] = make_float4(bl.min[2] - pad, bl.max[2] + pad, br.min[0] - pad, br.max[0] + pad);
    o[2] = make_float4(br.min[1] - pad, br.max[1] + pad, br.min[2] - pad, br.max[2] + pad);
    // .z holds the learned child-order bits (none until an order model is applied)
    o[3] = make_float4(__uint_as_float(r0), __uint_as_float(r1), 0.0f, 0.0f);
    // leaf-order ranges of the children, [A, B) and [B, C), and the binary depth
    aux[p.trav] = make_uint4(p.first, middle, middle + rc, p.depth);
}

// Single-triangle scene: one node whose two children are the same leaf.
__device__ __forceinline__ void write_single(const rtq_aabb& a, float pad, float4* __restrict__ nodes,
                                             uint4* __restrict__ aux) {
    float lo[3], hi[3];
    for (int k = 0; k < 3; ++k) { lo[k] = a.min[k] - pad; hi[k] = a.max[k] + pad; }
    const uint32_t r = leaf_ref(0, 1);
    nodes[0] = make_float4(lo[0], hi[0], lo[1], hi[1]);
    nodes[1] = make_float4(lo[2], hi[2], lo[0], hi[0]);
    nodes[2] = make_float4(lo[1], hi[1], lo[2], hi[2]);
    nodes[3] = make_float4(__uint_as_float(r), __uint_as_float(r), 0.0f, 0.0f);
    aux[0] = make_uint4(0u, 1u, 1u, 0u);
}

// The traversal triangles (the first leaf_blocks workgroups) and the binary
// traversal nodes (the others) in one launch: neither reads what the other
// writes.
__global__ __launch_bounds__(kThreads) void k_write_layout(
    uint32_t leaf_blocks, uint32_t nt, uint32_t nc, uint32_t max_leaf, const rtq_aabb* __restrict__ bounds,
    const uint32_t* __restrict__ ctri, const float4* __restrict__ tri_world, const rtq_aabb* __restrict__ cbox,
    const uint32_t* __restrict__ cleft, const uint32_t* __restrict__ cright, const uint32_t* __restrict__ ccount,
    const uint32_t* __restrict__ ctrav, const uint4* __restrict__ placed, float4* __restrict__ tris,
    uint32_t* __restrict__ block_depth, float4* __restrict__ nodes, uint4* __restrict__ aux) {
    if (blockIdx.x < leaf_blocks) {
        write_leaves(nt, ctri, placed, tri_world, tris, block_depth);
        return;
    }
    const uint32_t i = (blockIdx.x - leaf_blocks) * kThreads + threadIdx.x;
    const float pad = box_pad_of(bounds[0]);
    if (nc == 1) {
        if (i == 0) write_single(cbox[0], pad, nodes, aux);
    } else if (nt + i < nc) {
        write_trav(nt + i, nt, nc, max_leaf, pad, cbox, cleft, cright, ccount, ctrav, placed, nodes, aux);
    }
}

inline uint32_t blocks_for(uint64_t n) { return (uint32_t)((n + kThreads - 1) / kThreads); }

// Shared front half of the build and of rtq_morton_codes: scene box + cube.
// d_bounds holds 2 boxes followed by 6 floats per partial block (at most
// kBoundsPartials): kBoundsBoxes boxes of 32 B.
constexpr uint32_t kBoundsPartials = 1024;
constexpr uint32_t kBoundsBoxes = 2 + (6 * kBoundsPartials + 7) / 8;
rtq_status compute_bounds(rtq_ctx* ctx, Scene* s, uint32_t pad_origin, rtq_aabb* d_bounds,
                          hipStream_t st) {
    const uint32_t nb = std::min<uint32_t>(blocks_for(s->n_tris), kBoundsPartials);
    float* partial = reinterpret_cast<float*>(d_bounds + 2);
    hipLaunchKernelGGL(k_bounds_partial, dim3(nb), dim3(kThreads), 0, st, s->tris_ref, s->models,
                       s->n_tris, partial);
    RTQ_HIP(ctx, hipGetLastError());
    hipLaunchKernelGGL(k_bounds_final, dim3(1), dim3(kThreads), 0, st, partial, nb, s->n_tris,
                       pad_origin, d_bounds);
    RTQ_HIP(ctx, hipGetLastError());
    return RTQ_OK;
}


// PLOC with fused passes: batches of kPlocBatch k_ploc_pass launches (each a
// no-op once at most kTailMax clusters are left) and one k_ploc_tail launch
// (a no-op until then), then one read of the state and the pass logs.  The
// active list starts in (c0, b0); c1, b1 are the other buffers.  state: the
// kPlocHeadWords words that k_leaf_init set, then room for the tail's log.  A batch's
// passes all take the grid of its first pass; 16 passes per batch bring a
// 2M-triangle terrain (61 passes) to the tail in two host round trips.
// root_trav: the traversal nodes in the whole tree (Scene::ctrav of the root).
rtq_status ploc_fused(rtq_ctx* ctx, Scene* s, uint32_t radius, Temps& tmp, uint32_t* state, uint32_t* c0, uint32_t* c1,
                      Box6* b0, Box6* b1, std::vector<std::pair<uint32_t, uint32_t>>& passes, uint32_t* root_trav,
                      hipStream_t st) {
    const uint32_t n = s->n_tris;
    const uint32_t T = kPassThreads - 2 * radius;
    const uint32_t max_tiles = (n + T - 1) / T;
    // ctl: kPlocBatch tile counters, then kPlocBatch x max_tiles status words
    constexpr size_t kCtrWords = (size_t)kPlocBatch * kTicketWords;
    const size_t ctl_words = kCtrWords + (size_t)kPlocBatch * max_tiles * 2;
    uint32_t* ctl = nullptr;
    if (n > kTailMax) RTQ_HIP(ctx, tmp.get(&ctl, ctl_words));
    uint32_t* const err = state + kPlocErrWord;
    uint4* const log = reinterpret_cast<uint4*>(state + 16);
    uint4* const tail_log = reinterpret_cast<uint4*>(state + kPlocHeadWords);
    PlocLists lists{{c0, c1}, {b0, b1}};
    PlocClusters cl{s->cbox, s->cleft,  s->cright, s->cparent, s->ccount,
                    s->ctri, s->ctrav, n,         s->params.max_leaf_size};
    uint32_t iter = n, n_total = n;
    std::vector<uint4> h_tail;
    while (iter > 1) {
        const uint32_t bound = iter;
        if (iter > kTailMax) {
            const uint32_t tiles = (bound + T - 1) / T;
            RTQ_HIP(ctx, hipMemsetAsync(ctl, 0, sizeof(uint32_t) * (kCtrWords + 2ull * kPlocBatch * tiles), st));
            uint64_t* status = reinterpret_cast<uint64_t*>(ctl + kCtrWords);
            for (uint32_t k = 0; k < kPlocBatch; ++k) {
                PlocPassArgs a{state + 4 * (k & 1), state + 4 * ((k + 1) & 1), bound, radius, ctl + k * kTicketWords,
                               status + (size_t)k * tiles, err, log + k, lists, cl};
                hipLaunchKernelGGL(k_ploc_pass, dim3(tiles), dim3(kPassThreads), 0, st, a);
                RTQ_HIP(ctx, hipGetLastError());
            }
        }
        // the state of the batch's last pass is in slot 0 (kPlocBatch is even)
        hipLaunchKernelGGL(k_ploc_tail, dim3(1), dim3(kTailThreads), 0, st, state, radius, lists, cl, report(ctx));
        RTQ_HIP(ctx, hipGetLastError());
        // the head block and the first tail log entries (those past the tail's
        // pass count are not used)
        RTQ_HIP(ctx, hipStreamSynchronize(st));
        uint32_t h_head[kPlocReportWords];
        std::memcpy(h_head, report(ctx), sizeof h_head);
        const uint32_t* h_state = h_head;
        const uint32_t* h_err = h_head + kPlocErrWord;
        uint4 h_log[kPlocBatch];
        memcpy(h_log, h_head + 16, sizeof h_log);
        if (h_err[0] & kPlocErrNoMerge) return fail(ctx, RTQ_EINTERNAL, "PLOC pass made no merge");
        if (h_err[0])
            return fail(ctx, RTQ_EINTERNAL, "fused PLOC pass failed (error bits 0x%x)", h_err[0]);
        if (iter > kTailMax)
            for (uint32_t k = 0; k < kPlocBatch; ++k) {
                const uint4 e = h_log[k];  // (first merge id, merges, clusters at the pass, left to the tail)
                if (e.w) break;
                if (e.y == 0) return fail(ctx, RTQ_EINTERNAL, "PLOC pass with %u clusters made no merge", e.z);
                passes.emplace_back(e.x, e.y);
            }
        const uint32_t nt = h_head[kTailCountWord];
        if (nt > kTailMax) return fail(ctx, RTQ_EINTERNAL, "PLOC tail ran %u passes", nt);
        if (nt) {
            h_tail.resize(nt);
            if (nt <= kTailPeek) {
                memcpy(h_tail.data(), h_head + kPlocHeadWords, sizeof(uint4) * nt);
            } else {
                HostReads rd(ctx, st);
                RTQ_HIP(ctx, rd.add(h_tail.data(), tail_log, sizeof(uint4) * nt));
                RTQ_HIP(ctx, rd.wait());
            }
            for (const uint4& e : h_tail) passes.emplace_back(e.x, e.y);
        }
        if (h_state[0] >= iter && h_state[0] > 1)
            return fail(ctx, RTQ_EINTERNAL, "PLOC made no progress at %u clusters", iter);
        iter = h_state[0];
        n_total = h_state[1];
        *root_trav = h_state[3];
    }
    if (n_total != 2 * n - 1) return fail(ctx, RTQ_EINTERNAL, "PLOC produced %u clusters, expected %u", n_total, 2 * n - 1);
    return RTQ_OK;
}

// PLOC with one launch per step of a pass: neighbour search, flags, scan,
// merge and state update (RTQ_BUILD_PLOC_SPLIT).  Passes are queued kPlocBatch
// at a time against a device-side cluster count; the host reads the count and
// the pass log once per batch (passes queued after the last merge find one
// cluster and change nothing).
rtq_status ploc_split(rtq_ctx* ctx, Scene* s, uint32_t radius, Temps& tmp, uint32_t* c_in, uint32_t* c_out,
                      Box6* b_in, Box6* b_out, std::vector<std::pair<uint32_t, uint32_t>>& pass_ranges,
                      uint32_t* root_trav, hipStream_t st) {
    constexpr uint32_t kPlocBatch = 8;
    const uint32_t n = s->n_tris;
    uint32_t *nn = nullptr, *state = nullptr;
    uint2 *flags = nullptr, *offs = nullptr, *tot = nullptr, *scan_ws = nullptr;
    uint4* pass_log = nullptr;
    RTQ_HIP(ctx, tmp.get(&nn, n));
    RTQ_HIP(ctx, tmp.get(&flags, n));
    RTQ_HIP(ctx, tmp.get(&offs, n));
    RTQ_HIP(ctx, tmp.get(&tot, 1));
    RTQ_HIP(ctx, tmp.get(&state, 2));
    RTQ_HIP(ctx, tmp.get(&pass_log, kPlocBatch));
    RTQ_HIP(ctx, tmp.get(&scan_ws, std::max<uint64_t>(scan_u32x2_workspace(n), 1)));
    RTQ_HIP(ctx, hipMemsetAsync(nn, 0, sizeof(uint32_t) * n, st));
    const uint32_t h_state0[2] = {n, n};
    RTQ_HIP(ctx, hipMemcpyAsync(state, h_state0, sizeof h_state0, hipMemcpyHostToDevice, st));
    uint32_t iter = n, n_total = n;
    while (iter > 1) {
        const uint32_t bound = iter;
        for (uint32_t k = 0; k < kPlocBatch; ++k) {
            hipLaunchKernelGGL(k_ploc_nn, dim3(blocks_for(bound)), dim3(kThreads), 0, st, b_in, state,
                               radius, nn);
            RTQ_HIP(ctx, hipGetLastError());
            hipLaunchKernelGGL(k_ploc_flags, dim3(blocks_for(bound)), dim3(kThreads), 0, st, nn, state, bound, flags);
            RTQ_HIP(ctx, hipGetLastError());
            const rtq_status rs = scan_u32x2_ws(ctx, flags, offs, bound, tot, scan_ws, st);
            if (rs != RTQ_OK) return rs;
            hipLaunchKernelGGL(k_ploc_merge, dim3(blocks_for(bound)), dim3(kThreads), 0, st, state, nn, flags, offs,
                               c_in, b_in, c_out, b_out, s->cbox, s->cleft, s->cright, s->cparent, s->ccount,
                               s->ctri, s->ctrav, n, s->params.max_leaf_size);
            RTQ_HIP(ctx, hipGetLastError());
            hipLaunchKernelGGL(k_ploc_advance, dim3(1), dim3(1), 0, st, tot, state, pass_log, k);
            RTQ_HIP(ctx, hipGetLastError());
            std::swap(c_in, c_out);
            std::swap(b_in, b_out);
        }
        uint4 h_log[kPlocBatch];
        uint32_t h_state[2];
        HostReads rd(ctx, st);
        RTQ_HIP(ctx, rd.add(h_log, pass_log, sizeof h_log));
        RTQ_HIP(ctx, rd.add(h_state, state, sizeof h_state));
        RTQ_HIP(ctx, rd.wait());
        for (uint32_t k = 0; k < kPlocBatch; ++k) {
            const uint4 e = h_log[k];  // (first merge id, merges, clusters at the pass)
            if (e.z <= 1) break;
            if (e.y == 0) return fail(ctx, RTQ_EINTERNAL, "PLOC pass with %u clusters made no merge", e.z);
            pass_ranges.emplace_back(e.x, e.y);
        }
        iter = h_state[0];
        n_total = h_state[1];
    }
    if (n_total != 2 * n - 1)
        return fail(ctx, RTQ_EINTERNAL, "PLOC produced %u clusters, expected %u", n_total, 2 * n - 1);
    if (n > 1) {
        HostReads rd(ctx, st);
        RTQ_HIP(ctx, rd.add(root_trav, s->ctrav + (n_total - 1), sizeof(uint32_t)));
        RTQ_HIP(ctx, rd.wait());
    }
    return RTQ_OK;
}

// Steps after PLOC, shared by the build and the refit: pre-order placement,
// the reference node array and leaf-ordered triangles, the box pad from the
// scene extent, the binary traversal nodes and (node_width 8) the compressed
// wide nodes.  Buffers that exist already are written in place (a refit keeps
// their addresses, so captured batch graphs stay valid).
// Work queued on the context's second stream: fork(st) makes it wait for
// what st has queued, join(st) makes st wait for it.  Forked work that is
// never joined (an early return) is waited for on the host when the guard
// goes out of scope, before the temporaries it uses are given back.
class SideWork {
public:
    explicit SideWork(rtq_ctx* ctx) : ctx_(ctx) {}
    SideWork(const SideWork&) = delete;
    SideWork& operator=(const SideWork&) = delete;
    ~SideWork() {
        if (forked_ && !joined_) (void)hipStreamSynchronize(ctx_->side);
    }
    hipError_t fork(hipStream_t st) {
        hipError_t e = hipEventRecord(ctx_->fork, st);
        if (e == hipSuccess) e = hipStreamWaitEvent(ctx_->side, ctx_->fork, 0);
        forked_ = true;  // even on an error: the destructor then waits for the side stream
        return e;
    }
    hipError_t join(hipStream_t st) {
        if (!forked_ || joined_) return hipSuccess;
        hipError_t e = hipEventRecord(ctx_->join, ctx_->side);
        if (e == hipSuccess) e = hipStreamWaitEvent(st, ctx_->join, 0);
        if (e == hipSuccess) joined_ = true;
        return e;
    }

private:
    rtq_ctx* ctx_;
    bool forked_ = false, joined_ = false;
};

// refit: the tree is the one the last build wrote the layouts for, with new
// boxes: its placement is kept and the 8-wide nodes keep their children.
// d_bounds: the scene's box and cube (compute_bounds), after a refit the
// root cluster's box.
rtq_status write_layouts(rtq_ctx* ctx, Scene* s, const rtq_aabb* d_bounds, hipStream_t st, bool refit) {
    const uint32_t n = s->n_tris;
    const uint32_t nc = s->n_clusters;
    Temps tmp(ctx);
    // the places stay with the scene: the reference node array is written from
    // them on demand (ensure_ref_nodes), and a refit keeps them
    if (!s->placed) RTQ_HIP(ctx, dev_alloc(&s->placed, nc));
    if (!s->sub_roots) RTQ_HIP(ctx, dev_alloc(&s->sub_roots, kLdsClusters + 2));
    if (!s->sub_list) RTQ_HIP(ctx, dev_alloc(&s->sub_list, n));
    if (!s->nodes) RTQ_HIP(ctx, take(s->kept_nodes, &s->nodes, 4ull * s->n_trav));
    if (!s->node_aux) RTQ_HIP(ctx, take(s->kept_aux, &s->node_aux, s->n_trav));
    s->ref_ready = false;
    uint32_t* bdep = nullptr;
    RTQ_HIP(ctx, tmp.get(&bdep, blocks_for(n)));
    float* wcost = nullptr;
    uint32_t* wchoice = nullptr;
    SideWork side(ctx);
    rtq_status rs = RTQ_OK;
    if (!refit) {
        const uint32_t n_passes = (uint32_t)s->passes.size();
        const bool cost = s->params.node_width == 8 && n > 1;
        if (cost) {
            RTQ_HIP(ctx, tmp.get(&wcost, (size_t)(nc - n) * 8));
            RTQ_HIP(ctx, tmp.get(&wchoice, nc - n));
        }
        // the passes at the top of the tree in one launch (their clusters'
        // state in LDS), then the middle subtrees, then the larger passes, last
        // pass first; the collapse's cost table the other way round on the
        // second stream, where it waits for the subtrees' lists
        const uint32_t c_lo = n_passes ? s->passes[s->lds_from].first : nc - 1;
        const uint32_t c_mid = s->sub_from < s->lds_from ? s->passes[s->sub_from].first : c_lo;
        if (cost) RTQ_HIP(ctx, side.fork(st));
        hipLaunchKernelGGL(k_place_lds, dim3(1), dim3(kLdsThreads), 0, st, top_passes(s), c_lo, nc, c_mid, n,
                           s->cleft, s->cright, s->ccount, s->ctrav, s->placed, s->sub_roots);
        RTQ_HIP(ctx, hipGetLastError());
        if (cost) {
            rs = wide_cost_bottom(ctx, s, wcost, wchoice, ctx->side);
            if (rs != RTQ_OK) return rs;
        }
        if (c_mid < c_lo) {
            hipLaunchKernelGGL(k_place_subtrees, dim3(nc - c_lo + 1), dim3(kSubThreads), 0, st, s->sub_roots, c_mid,
                               n, s->cleft, s->cright, s->ccount, s->ctrav, s->placed, s->sub_list);
            RTQ_HIP(ctx, hipGetLastError());
        }
        if (cost) {
            RTQ_HIP(ctx, side.fork(st));
            rs = wide_cost_top(ctx, s, wcost, wchoice, ctx->side);
            if (rs != RTQ_OK) return rs;
        }
        for (uint32_t k = s->sub_from; k > 0; --k) {
            const auto& pr = s->passes[k - 1];
            hipLaunchKernelGGL(k_place_pass, dim3(blocks_for(pr.second)), dim3(kThreads), 0, st, pr.first, pr.second,
                               n, s->cleft, s->cright, s->ccount, s->ctrav, s->placed);
            RTQ_HIP(ctx, hipGetLastError());
        }
    }
    const uint32_t leaf_blocks = blocks_for(n);
    hipLaunchKernelGGL(k_write_layout, dim3(leaf_blocks + blocks_for(std::max(nc - n, 1u))), dim3(kThreads), 0, st,
                       leaf_blocks, n, nc, s->params.max_leaf_size, d_bounds, s->ctri, s->tri_world, s->cbox, s->cleft,
                       s->cright, s->ccount, s->ctrav, s->placed, s->tris, bdep, s->nodes, s->node_aux);
    RTQ_HIP(ctx, hipGetLastError());
    // the depth depends on the topology only: a refit keeps it
    rs = write_top(ctx, s, bdep, refit ? 0u : leaf_blocks, d_bounds, st);
    if (rs != RTQ_OK) return rs;
    if (s->params.node_width == 8) {
        if (refit) {
            rs = refit_wide(ctx, s, st);
        } else {
            RTQ_HIP(ctx, side.join(st));
            rs = build_wide(ctx, s, wchoice, d_bounds, st);
        }
        if (rs != RTQ_OK) return rs;
    }
    if (!refit) RTQ_HIP(ctx, hipEventRecord(ctx->build_end, st));
    RTQ_HIP(ctx, hipStreamSynchronize(st));
    BuildReport h;
    std::memcpy(&h, report(ctx), sizeof h);
    if (!refit) s->depth = h.depth;
    s->box_pad = box_pad_of(h.box);
    return RTQ_OK;
}

}  // namespace

rtq_status ensure_ref_nodes(rtq_ctx* ctx, Scene* s, hipStream_t st) {
    if (s->ref_ready) return RTQ_OK;
    const uint32_t nc = s->n_clusters;
    if (!s->built || !s->placed || nc == 0)
        return fail(ctx, RTQ_EINTERNAL, "reference nodes: scene has no placed tree");
    if (!s->ref_nodes) RTQ_HIP(ctx, dev_alloc(&s->ref_nodes, nc));
    if (!s->ref_nodes) return fail(ctx, RTQ_ENOMEM, "reference nodes: allocation failed");
    hipLaunchKernelGGL(k_write_ref, dim3(blocks_for(nc)), dim3(kThreads), 0, st, nc, s->cbox, s->ctri, s->cleft,
                       s->cright, s->placed, s->ref_nodes);
    RTQ_HIP(ctx, hipGetLastError());
    s->ref_ready = true;
    return RTQ_OK;
}

TopPasses top_passes(const Scene* s) {
    TopPasses t{};
    t.n = (uint32_t)s->passes.size() - s->lds_from;
    for (uint32_t k = 0; k < std::min(t.n, kInlinePasses); ++k)
        t.inline_passes[k] = make_uint2(s->passes[s->lds_from + k].first, s->passes[s->lds_from + k].second);
    t.rest = s->d_passes;
    return t;
}

rtq_status build_scene(rtq_ctx* ctx, Scene* s, const rtq_build_params& prm) {
    hipStream_t st = ctx->stream;
    const uint32_t n = s->n_tris;
    const uint32_t nc = 2 * n - 1;
    // work queued earlier may still read the buffers a rebuild overwrites
    RTQ_HIP(ctx, hipDeviceSynchronize());
    reset_build(s);
    s->params = prm;
    s->n_clusters = nc;
    // size the context's scratch for this build's temporaries up front, so a
    // first build does not allocate them one by one.  Alive together, per
    // triangle: sort keys and values and the PLOC lists 64 B; with 8-wide nodes
    // also the collapse cost table 36 B and the collapse's two level lists 8 B
    // per binary traversal node (one per triangle with leaves of one triangle);
    // the fused PLOC passes' tile status words (16 passes x 8 B per tile of 480),
    // each leaf workgroup's deepest leaf and the collapse's tile status words,
    // under n / 2 B; 1 MiB for scans and 256-B rounding
    const size_t per_tri = prm.node_width == 8 ? 64 + 36 + 8 : 64;
    ctx->arena.peak = std::max<size_t>(ctx->arena.peak, per_tri * n + n / 2 + ((size_t)1 << 20));
    rtq_status rs = arena_reserve(ctx);
    if (rs != RTQ_OK) return rs;

    RTQ_HIP(ctx, hipEventRecord(ctx->build_begin, st));

    // persistent products, sized by the triangle count: a rebuild rewrites them
    if (!s->cbox) RTQ_HIP(ctx, dev_alloc(&s->cbox, nc));
    if (!s->ctri) RTQ_HIP(ctx, dev_alloc(&s->ctri, nc));
    if (!s->cleft) RTQ_HIP(ctx, dev_alloc(&s->cleft, nc));
    if (!s->cright) RTQ_HIP(ctx, dev_alloc(&s->cright, nc));
    if (!s->cparent) RTQ_HIP(ctx, dev_alloc(&s->cparent, nc));
    if (!s->ccount) RTQ_HIP(ctx, dev_alloc(&s->ccount, nc));
    if (!s->ctrav) RTQ_HIP(ctx, dev_alloc(&s->ctrav, nc));
    if (!s->sorted_idx) RTQ_HIP(ctx, dev_alloc(&s->sorted_idx, n));
    if (!s->sorted_codes) RTQ_HIP(ctx, dev_alloc(&s->sorted_codes, n));
    if (!s->tris) RTQ_HIP(ctx, dev_alloc(&s->tris, 3ull * n));

    Temps tmp(ctx);
    rtq_aabb* d_bounds = nullptr;
    uint32_t *tk = nullptr, *tv = nullptr, *c_in = nullptr, *c_out = nullptr;
    Box6 *b_in = nullptr, *b_out = nullptr;
    RTQ_HIP(ctx, tmp.get(&d_bounds, kBoundsBoxes));
    RTQ_HIP(ctx, tmp.get(&tk, n));
    RTQ_HIP(ctx, tmp.get(&tv, n));
    RTQ_HIP(ctx, tmp.get(&c_in, n));
    RTQ_HIP(ctx, tmp.get(&c_out, n));
    RTQ_HIP(ctx, tmp.get(&b_in, n));
    RTQ_HIP(ctx, tmp.get(&b_out, n));

    // 1. bounds, cube, Morton codes, sort
    rs = compute_bounds(ctx, s, prm.flags & RTQ_BUILD_REF_PADDED_BOUNDS, d_bounds, st);
    if (rs != RTQ_OK) return rs;
    hipLaunchKernelGGL(k_morton, dim3(blocks_for(n)), dim3(kThreads), 0, st, s->tris_ref, s->models, n,
                       d_bounds, s->sorted_codes, s->sorted_idx);
    RTQ_HIP(ctx, hipGetLastError());
    rs = radix_sort_pairs(ctx, s->sorted_codes, s->sorted_idx, tk, tv, n, 30, st);
    if (rs != RTQ_OK) return rs;

    // 2. PLOC
    uint32_t* head = nullptr;
    RTQ_HIP(ctx, tmp.get(&head, kPlocHeadWords + 4 * kTailMax));
    hipLaunchKernelGGL(k_leaf_init, dim3(blocks_for(n)), dim3(kThreads), 0, st, s->tris_ref, s->models,
                       s->sorted_idx, n, s->cbox, s->ctri, s->ccount, s->cleft, s->cright, s->cparent, c_in, b_in,
                       head);
    RTQ_HIP(ctx, hipGetLastError());
    std::vector<std::pair<uint32_t, uint32_t>> pass_ranges;
    uint32_t root_trav = 0;
    rs = (prm.flags & RTQ_BUILD_PLOC_SPLIT)
             ? ploc_split(ctx, s, prm.search_radius, tmp, c_in, c_out, b_in, b_out, pass_ranges, &root_trav, st)
             : ploc_fused(ctx, s, prm.search_radius, tmp, head, c_in, c_out, b_in, b_out, pass_ranges, &root_trav, st);
    if (rs != RTQ_OK) return rs;
    s->n_trav = std::max(root_trav, 1u);   // the root always has a node
    s->ploc_passes = (uint32_t)pass_ranges.size();
    s->passes = pass_ranges;
    // the passes of the single-workgroup launches (placement, collapse costs,
    // refit merges): those from lds_from on create at most kLdsClusters clusters
    s->lds_from = s->ploc_passes;
    while (s->lds_from > 0 && nc - s->passes[s->lds_from - 1].first <= kLdsClusters) --s->lds_from;
    s->sub_from = s->lds_from;
    while (s->sub_from > 0 && s->passes[s->sub_from - 1].second <= kSubPass) --s->sub_from;
    if (s->ploc_passes - s->lds_from > kInlinePasses) {
        const uint32_t from = s->lds_from + kInlinePasses, rest = s->ploc_passes - from;
        s->h_passes.resize(rest);
        for (uint32_t k = 0; k < rest; ++k)
            s->h_passes[k] = make_uint2(s->passes[from + k].first, s->passes[from + k].second);
        RTQ_HIP(ctx, take(s->kept_passes, &s->d_passes, rest));
        RTQ_HIP(ctx, hipMemcpyAsync(s->d_passes, s->h_passes.data(), sizeof(uint2) * rest, hipMemcpyHostToDevice, st));
    }

    // 3-4. node arrays of every layout
    rs = write_layouts(ctx, s, d_bounds, st, false);
    if (rs != RTQ_OK) return rs;
    float ms = 0.0f;
    RTQ_HIP(ctx, hipEventElapsedTime(&ms, ctx->build_begin, ctx->build_end));
    s->build_ms = ms;
    s->built = true;
    s->generation = ++ctx->builds;
    // temporaries that did not fit the scratch reserved above raised its peak
    s->scratch_spill = ctx->arena.peak > ctx->arena.cap ? ctx->arena.peak - ctx->arena.cap : 0;
    return RTQ_OK;
}

rtq_status write_top(rtq_ctx* ctx, Scene* s, const uint32_t* block_depth, uint32_t n_blocks, const rtq_aabb* bounds,
                     hipStream_t st) {
    if (kTopNodes == 0 && !bounds) return RTQ_OK;
    // the set depends on the topology only, so a refit or an order update
    // rewrites the same buffer with the same node count
    if (!s->top) RTQ_HIP(ctx, dev_alloc(&s->top, 4ull * std::max(kTopNodes, 1u)));
    hipLaunchKernelGGL(k_top_nodes, dim3(bounds ? 2 : 1), dim3(kTopThreads), 0, st, s->nodes, s->top, block_depth,
                       n_blocks, bounds, reinterpret_cast<BuildReport*>(report(ctx)));
    RTQ_HIP(ctx, hipGetLastError());
    s->n_top = std::min(kTopNodes, s->n_trav);   // every traversal node can be reached from the root
    return RTQ_OK;
}

// New boxes for the kept cluster tree (rtq_bvh_refit): leaf boxes from the
// current vertices, then the merges of each PLOC pass in build order (a
// merge's children come from earlier passes), then the leaf triangles and the
// binary nodes again and new boxes in the kept 8-wide nodes, written into the
// buffers they already have.
rtq_status refit_scene(rtq_ctx* ctx, Scene* s) {
    hipStream_t st = ctx->stream;
    const uint32_t n = s->n_tris;
    const rtq_status ra = arena_reserve(ctx);
    if (ra != RTQ_OK) return ra;
    hipLaunchKernelGGL(k_refit_leaves, dim3(blocks_for(n)), dim3(kThreads), 0, st, s->tris_ref, s->models, s->ctri,
                       n, s->cbox);
    RTQ_HIP(ctx, hipGetLastError());
    const uint32_t n_passes = (uint32_t)s->passes.size();
    for (uint32_t k = 0; k < s->sub_from; ++k) {
        const auto& pr = s->passes[k];
        hipLaunchKernelGGL(k_refit_merge, dim3(blocks_for(pr.second)), dim3(kThreads), 0, st, pr.first, pr.second,
                           s->cleft, s->cright, s->cbox);
        RTQ_HIP(ctx, hipGetLastError());
    }
    if (s->sub_from < s->lds_from) {
        const uint32_t blocks = s->n_clusters - s->passes[s->lds_from].first + 1;
        hipLaunchKernelGGL(k_refit_subtrees, dim3(blocks), dim3(kSubThreads), 0, st, s->sub_roots, s->sub_list,
                           s->placed, s->cleft, s->cright, s->cbox);
        RTQ_HIP(ctx, hipGetLastError());
    }
    if (s->lds_from < n_passes) {
        hipLaunchKernelGGL(k_refit_merge_lds, dim3(1), dim3(kLdsThreads), 0, st, top_passes(s),
                           s->passes[s->lds_from].first, s->n_clusters, s->cleft, s->cright, s->cbox);
        RTQ_HIP(ctx, hipGetLastError());
    }
    // the box pad needs the largest coordinate magnitude of the scene bounds:
    // the root cluster's new box holds the same minima and maxima (merges are
    // exact), and the reference quirk of adding the origin cannot raise it
    return write_layouts(ctx, s, s->cbox + (s->n_clusters - 1), st, true);
}

rtq_status morton_codes(rtq_ctx* ctx, Scene* s, uint32_t flags, uint32_t* host_codes) {
    hipStream_t st = ctx->stream;
    RTQ_HIP(ctx, hipDeviceSynchronize());  // nothing queued still uses the arena
    const rtq_status ra = arena_reserve(ctx);
    if (ra != RTQ_OK) return ra;
    Temps tmp(ctx);
    rtq_aabb* d_bounds = nullptr;
    uint32_t* codes = nullptr;
    RTQ_HIP(ctx, tmp.get(&d_bounds, kBoundsBoxes));
    RTQ_HIP(ctx, tmp.get(&codes, s->n_tris));
    rtq_status rs = compute_bounds(ctx, s, flags & RTQ_BUILD_REF_PADDED_BOUNDS, d_bounds, st);
    if (rs != RTQ_OK) return rs;
    hipLaunchKernelGGL(k_morton, dim3(blocks_for(s->n_tris)), dim3(kThreads), 0, st, s->tris_ref, s->models,
                       s->n_tris, d_bounds, codes, (uint32_t*)nullptr);
    RTQ_HIP(ctx, hipGetLastError());
    RTQ_HIP(ctx, hipMemcpyAsync(host_codes, codes, sizeof(uint32_t) * s->n_tris, hipMemcpyDeviceToHost, st));
    RTQ_HIP(ctx, hipStreamSynchronize(st));
    return RTQ_OK;
}

}  // namespace rtq
