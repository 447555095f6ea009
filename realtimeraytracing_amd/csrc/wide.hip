// Compressed 8-wide traversal nodes built from the binary PLOC tree.
//
// Collapse: top-down, one level per launch.  Each internal cluster's 8 slots
// are given out as an SAH cost table says (see k_dp_pass below): a child that
// is internal with more than max_leaf triangles becomes a wide node of the
// next level, any other child a leaf (the subtree's triangles are already
// contiguous in leaf order).  Next-level node indices come from a scan, so
// numbering is deterministic and the children of a node are contiguous.
//
// Node (128 B, 8 float4; the plain traversal reads the first 96 B):
//   [ox oy oz meta] meta = ex | ey << 8 | ez << 16 | valid << 24
//   [qlo_x[0..7] qhi_x[0..7]] [qlo_y.. qhi_y..] [qlo_z.. qhi_z..]   (bytes)
//   [ref0..ref3] [ref4..ref7]
//   [learned first child: 16 x 4 bits, lo hi 0 0]  (zero until an order model
//       is applied; entry octant + 8 * any_hit = 8 | slot when decided)
//   [0 0 0 0]
// A child box is o + q * 2^(e - 127) per axis.  Boxes are widened by the scene
// pad and quantised outward in exact (double) arithmetic, so the decoded box
// always contains the padded child box: no hit is lost to quantisation
// (Ylitie, Karras & Laine, "Efficient Incoherent Ray Traversal on GPUs Through
// Compressed Wide BVHs", HPG 2017, for the quantised-box idea).
#include <cmath>
#include <type_traits>

#include "rtq_internal.hpp"

namespace rtq {
namespace {

constexpr int kThreads = 256;
constexpr int kWidth = 8;
// a level's tile: kLevelNodes nodes of 8 lanes each
constexpr int kLevelThreads = 512;
constexpr uint32_t kLevelNodes = kLevelThreads / kWidth;

__device__ __forceinline__ float box_area(const rtq_aabb& b) {
    const float dx = b.max[0] - b.min[0], dy = b.max[1] - b.min[1], dz = b.max[2] - b.min[2];
    return 2.0f * ((dx * dy + dy * dz) + dz * dx);
}

// SAH-optimal collapse (Ylitie, Karras & Laine, "Efficient incoherent ray
// traversal on GPUs through compressed wide BVHs", HPG 2017), restricted to
// this layout: cost[x][j-1] is the least SAH cost of cluster x's subtree when
// it may fill j slots of its parent: a cluster of more than max_leaf triangles
// given one slot is an 8-wide node (node cost + the best split of 8 slots
// between its children), a smaller one a leaf (triangle cost x count); j > 1
// slots go either to the cluster with fewer slots or split between its
// children.  choice[x] keeps, per j = 2..8, 0 (fewer slots) or the left
// child's share (bits 3(j-2)), and the node's own split (bits 21..23).
// Rows are computed bottom-up: the large PLOC passes one at a time (a merge's
// children come from earlier passes), the middle subtrees in one launch, the
// top's in another; single triangles have a constant row.
constexpr float kNodeCost = 1.0f;
constexpr float kTriCost = 0.6f;  // best of 0.15-4 on the 2M-triangle terrain

__device__ __forceinline__ void dp_row(uint32_t x, uint32_t nt, const float* cost,
                                       const rtq_aabb* __restrict__ cbox, float* row) {
    if (x < nt) {
        const float a = kTriCost * box_area(cbox[x]);
#pragma unroll
        for (int j = 0; j < kWidth; ++j) row[j] = a;
    } else {
#pragma unroll
        for (int j = 0; j < kWidth; ++j) row[j] = cost[(size_t)(x - nt) * kWidth + j];
    }
}

// Row and choice word of a cluster of `cnt` triangles and box area a from its
// children's rows dl, dr.
__device__ __forceinline__ uint32_t dp_combine(const float* dl, const float* dr, float a, uint32_t cnt,
                                               uint32_t max_leaf, float* row) {
    float bn = INFINITY;
    uint32_t kn = 1;
    for (uint32_t k = 1; k < kWidth; ++k) {
        const float v = dl[k - 1] + dr[kWidth - k - 1];
        if (v < bn) { bn = v; kn = k; }
    }
    row[0] = cnt <= max_leaf ? kTriCost * a * (float)cnt : kNodeCost * a + bn;
    uint32_t ch = (kn - 1) << 21;
    for (uint32_t j = 2; j <= kWidth; ++j) {
        float best = row[j - 2];
        uint32_t pick = 0;
        for (uint32_t k = 1; k < j; ++k) {
            const float v = dl[k - 1] + dr[j - k - 1];
            if (v < best) { best = v; pick = k; }
        }
        row[j - 1] = best;
        ch |= pick << (3 * (j - 2));
    }
    return ch;
}

__device__ __forceinline__ void dp_cluster(uint32_t c, uint32_t nt, uint32_t max_leaf,
                                           const uint32_t* __restrict__ cleft, const uint32_t* __restrict__ cright,
                                           const uint32_t* __restrict__ ccount, const rtq_aabb* __restrict__ cbox,
                                           float* cost, uint32_t* __restrict__ choice) {
    float dl[kWidth], dr[kWidth], row[kWidth];
    dp_row(cleft[c], nt, cost, cbox, dl);
    dp_row(cright[c], nt, cost, cbox, dr);
    const uint32_t ch = dp_combine(dl, dr, box_area(cbox[c]), ccount[c], max_leaf, row);
    float* out = cost + (size_t)(c - nt) * kWidth;
#pragma unroll
    for (int j = 0; j < kWidth; ++j) out[j] = row[j];
    choice[c - nt] = ch;
}

__global__ __launch_bounds__(kThreads) void k_dp_pass(uint32_t first, uint32_t count, uint32_t nt, uint32_t max_leaf,
                                                      const uint32_t* __restrict__ cleft,
                                                      const uint32_t* __restrict__ cright,
                                                      const uint32_t* __restrict__ ccount,
                                                      const rtq_aabb* __restrict__ cbox, float* __restrict__ cost,
                                                      uint32_t* __restrict__ choice) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i < count) dp_cluster(first + i, nt, max_leaf, cleft, cright, ccount, cbox, cost, choice);
}

// The cost rows of one middle subtree per workgroup (one wave), the deepest
// level first.
__global__ __launch_bounds__(kSubThreads) void k_dp_subtrees(const uint2* __restrict__ roots,
                                                             const uint32_t* __restrict__ list,
                                                             const uint4* __restrict__ placed, uint32_t nt,
                                                             uint32_t max_leaf, const uint32_t* __restrict__ cleft,
                                                             const uint32_t* __restrict__ cright,
                                                             const uint32_t* __restrict__ ccount,
                                                             const rtq_aabb* __restrict__ cbox, float* cost,
                                                             uint32_t* __restrict__ choice) {
    if (blockIdx.x >= roots[0].x) return;
    const uint2 root = roots[1 + blockIdx.x];
    levels_up(list + placed[root.x].y, root.y,
              [&](uint32_t c) { dp_cluster(c, nt, max_leaf, cleft, cright, ccount, cbox, cost, choice); });
}

// The passes at the top of the tree in one workgroup, bottom-up, with
// the cost rows of their clusters [c_lo, nc) in LDS (a child from an earlier
// pass gives its row from global memory); a barrier between passes.  Each
// thread keeps the child ids, box area and triangle count of its clusters
// c_lo + t + kLdsThreads * s in registers.  nc - c_lo <= kLdsClusters.
__global__ __launch_bounds__(kLdsThreads) void k_dp_lds(TopPasses passes, uint32_t c_lo, uint32_t nc, uint32_t nt, uint32_t max_leaf,
                                                        const uint32_t* __restrict__ cleft,
                                                        const uint32_t* __restrict__ cright,
                                                        const uint32_t* __restrict__ ccount,
                                                        const rtq_aabb* __restrict__ cbox, const float* __restrict__ cost,
                                                        uint32_t* __restrict__ choice) {
    constexpr int kSlots = kLdsClusters / kLdsThreads;
    __shared__ float s_row[kLdsClusters * kWidth];
    const uint32_t t = threadIdx.x;
    const uint32_t R = nc - c_lo;
    uint32_t L[kSlots], Rc[kSlots], N[kSlots];
    float A[kSlots];
#pragma unroll
    for (int q = 0; q < kSlots; ++q) {
        const uint32_t idx = t + kLdsThreads * q;
        const bool in = idx < R;
        L[q] = in ? cleft[c_lo + idx] : 0u;
        Rc[q] = in ? cright[c_lo + idx] : 0u;
        N[q] = in ? ccount[c_lo + idx] : 0u;
        A[q] = in ? box_area(cbox[c_lo + idx]) : 0.0f;
    }
    for (uint32_t k = 0; k < passes.n; ++k) {
        const uint2 p = passes[k];
#pragma unroll
        for (int q = 0; q < kSlots; ++q) {
            const uint32_t idx = t + kLdsThreads * q, c = c_lo + idx;
            if (idx >= R || c < p.x || c >= p.x + p.y) continue;
            float dl[kWidth], dr[kWidth], row[kWidth];
            if (L[q] >= c_lo) {
#pragma unroll
                for (int j = 0; j < kWidth; ++j) dl[j] = s_row[(L[q] - c_lo) * kWidth + j];
            } else {
                dp_row(L[q], nt, cost, cbox, dl);
            }
            if (Rc[q] >= c_lo) {
#pragma unroll
                for (int j = 0; j < kWidth; ++j) dr[j] = s_row[(Rc[q] - c_lo) * kWidth + j];
            } else {
                dp_row(Rc[q], nt, cost, cbox, dr);
            }
            choice[c - nt] = dp_combine(dl, dr, A[q], N[q], max_leaf, row);
#pragma unroll
            for (int j = 0; j < kWidth; ++j) s_row[idx * kWidth + j] = row[j];
        }
        __syncthreads();
    }
}

// Eight lanes per 8-wide node, one per slot.  A lane's walk from the node's
// cluster c to the child in slot `slot`, as the cost table splits the slots
// (children left to right); false if the split leaves the slot empty.  The
// lanes of one node load the same words, and no lane waits for another: the
// walk takes as many steps as the slot's child lies below c, where one thread
// per node takes a step for each cluster opened.
__device__ __forceinline__ bool slot_child(uint32_t c, uint32_t slot, const uint32_t* __restrict__ cleft,
                                           const uint32_t* __restrict__ cright, uint32_t nt,
                                           const uint32_t* __restrict__ choice, uint32_t* child) {
    uint32_t x = c, j = kWidth, o = slot;   // cluster x fills j slots, this lane's is number o of them
    bool root = true;
    while (j > 1 && x >= nt) {
        const uint32_t cw = choice[x - nt], l = cleft[x], r = cright[x];
        uint32_t pick;
        if (root) {
            pick = ((cw >> 21) & 7u) + 1u;
            root = false;
        } else {
            while (j > 1 && (pick = (cw >> (3 * (j - 2))) & 7u) == 0) --j;   // fewer slots: the last ones stay empty
            if (j == 1) break;
            if (o >= j) return false;
        }
        if (o < pick) {
            x = l;
            j = pick;
        } else {
            x = r;
            j -= pick;
            o -= pick;
        }
    }
    *child = x;
    return o == 0;
}

// Minimum of a value over each 8 lanes, in all of them.
__device__ __forceinline__ float min_of_8(float x) {
    const auto dpp = [](float v, auto ctrl) {
        return __int_as_float(
            __builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctrl)::value, 0xF, 0xF, false));
    };
    x = fminf(x, dpp(x, std::integral_constant<int, 0xB1>{}));    // lanes 1 0 3 2 of each quad
    x = fminf(x, dpp(x, std::integral_constant<int, 0x4E>{}));    // lanes 2 3 0 1
    return fminf(x, dpp(x, std::integral_constant<int, 0x141>{}));   // the other quad
}

// Smallest e with 255 * 2^e >= extent, in [-126, 127]: for an extent of
// m 2^k, 1 <= m < 2, k - 7 if m <= 255 / 128, else k - 6.
__device__ __forceinline__ int exponent_for(double extent) {
    if (!(extent > 0.0)) return -126;
    const uint64_t b = (uint64_t)__double_as_longlong(extent);
    const int k = (int)(b >> 52) - 1023;
    const int e = (b & ((1ull << 52) - 1)) <= (127ull << 45) ? k - 7 : k - 6;
    return e < -126 ? -126 : e > 127 ? 127 : e;
}

// Words of a node in LDS: 32, and 4 more to spread the nodes over the banks.
constexpr uint32_t kImageWords = 36;

// The first 16 words of an 8-wide node (origin and meta: exponents and valid
// mask; then the x, y and z planes) into img, by the node's 8 lanes.  A lane
// with a child (`has`) gives its slot and box; the others have the slots past
// the last child, in any order.  Every lane of the wave calls it; live: the
// lane's node exists.  Child boxes are widened by pad and quantised outward in
// exact (double) arithmetic, so the decoded box contains the padded child box.
__device__ __forceinline__ void wide_boxes(bool live, bool has, uint32_t slot, uint32_t n, const rtq_aabb& box,
                                           float pad, uint32_t* img) {
    uint8_t* const bytes = reinterpret_cast<uint8_t*>(img);
    uint32_t meta = n ? ((1u << n) - 1u) << 24 : 0u;
    float org[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const float lo = has ? box.min[q] - pad : INFINITY;
        const float hi = has ? box.max[q] + pad : -INFINITY;
        org[q] = min_of_8(lo);
        const float top = -min_of_8(-hi);
        const int e = exponent_for((double)top - (double)org[q]);
        meta |= (uint32_t)(e + 127) << (8 * q);
        // exact: float differences and products with a power of two (2^-e is a
        // normal double) are exact in double
        const double inv = __longlong_as_double((int64_t)(1023 - e) << 52);
        const double l = fmin(fmax(floor(((double)lo - (double)org[q]) * inv), 0.0), 255.0);
        const double h = fmin(fmax(ceil(((double)hi - (double)org[q]) * inv), 0.0), 255.0);
        // empty slots: an inverted box (lower planes 255, upper 0) that a ray
        // misses on every axis unless its origin lies more than 2^19 node
        // extents away; their child ref is then harmless (one triangle test,
        // see the level kernel), so traversal needs no test of the valid bits
        if (live) {
            bytes[16 * (q + 1) + slot] = has ? (uint8_t)(uint32_t)l : (uint8_t)0xFF;
            bytes[16 * (q + 1) + 8 + slot] = has ? (uint8_t)(uint32_t)h : (uint8_t)0;
        }
    }
    if (live && slot == 0) {
#pragma unroll
        for (int q = 0; q < 3; ++q) img[q] = __float_as_uint(org[q]);
        img[3] = meta;
    }
}

// Float4 i of a node's image, after the wave's writes to it.
__device__ __forceinline__ float4 image_part(const uint32_t* img, uint32_t i) {
    const uint4 w = reinterpret_cast<const uint4*>(img)[i];
    return make_float4(__uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), __uint_as_float(w.w));
}

// Tile status of the level scan: value in the low 32 bits, state on top.
constexpr uint64_t kLvAgg = 1ull << 62;     // the tile's own count
constexpr uint64_t kLvPre = 2ull << 62;     // the counts through the tile
constexpr uint64_t kLvState = 3ull << 62;

struct LevelArgs {
    uint32_t* lv;              // this level's words: count, first node, first status word, errors; then the next one's
    uint32_t* tickets;         // tile counters of this level, zero before it
    uint32_t* next_tickets;    // of the next one
    uint64_t* status;          // tile status words, n_status of them, zero before the first level
    uint32_t n_status;
    uint32_t cap;              // node capacity
    uint32_t max_leaf;
    uint32_t nt;
    const rtq_aabb* bounds;    // the scene's, for the box margin
    const uint32_t* items;     // this level's node clusters
    uint32_t* next_items;      // the next level's
    const uint32_t* cleft;
    const uint32_t* cright;
    const uint32_t* ccount;
    const rtq_aabb* cbox;
    const uint32_t* choice;
    const uint4* placed;
    float4* nodes;
    uint32_t* wide_trav;
    uint32_t* kids;            // 8 child clusters per node (kNone past the last)
};

// A child that becomes an 8-wide node of the next level: a merged cluster (ids
// from nt on) of more than max_leaf triangles.
__device__ __forceinline__ bool expandable(const LevelArgs& a, uint32_t c, uint32_t count) {
    return c >= a.nt && count > a.max_leaf;
}

// Expandable children of a whole tile's nodes, by one wave: the count that the
// tile publishes.
__device__ uint32_t expandable_of_tile(const LevelArgs& a, uint32_t tile) {
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t total = 0;
    for (uint32_t i = 0; i < kLevelNodes; i += 64 / kWidth) {
        uint32_t c = 0;
        const bool has = slot_child(a.items[tile * kLevelNodes + i + lane / kWidth], lane % kWidth, a.cleft, a.cright,
                                    a.nt, a.choice, &c);
        total += (uint32_t)__popcll(__ballot(has && expandable(a, c, a.ccount[c])));
    }
    return total;
}

// One level of the collapse in one launch, eight lanes per node of the level:
// each lane finds its slot's child; the next level's nodes are numbered by an
// exclusive scan of the nodes' expandable children in node order, across
// workgroups by decoupled look-back (a tile that has published nothing for long
// is counted by the wave that waits for it, see take_tile); then each lane
// quantises its child's box and the lanes of a node write its 128 B together.
// The last tile writes the next level's words (lv[4..6]).  The grid covers an
// upper bound of the level's count; workgroups past the count, and every
// workgroup of an empty level, return at once.
// The chain of dependent loads down to a slot's child bounds small levels, the
// children's scattered boxes large ones.  2,093,058 triangles, 12 levels: 354 us
// with one thread per node (its walk, boxes and quantisation one child after
// another), 171 us now; a level of a few nodes 20 us and 6 us.
__global__ __launch_bounds__(kLevelThreads) void k_wide_level(LevelArgs a) {
    constexpr uint32_t kWaves = kLevelThreads / 64;
    __shared__ uint32_t s_tile, s_excl, s_w[kWaves];
    __shared__ __align__(16) uint32_t s_img[kLevelNodes * kImageWords];
    const uint32_t count = a.lv[0];
    const uint32_t tiles = (count + kLevelNodes - 1) / kLevelNodes;
    if (blockIdx.x >= tiles) return;
    if ((uint64_t)a.lv[2] + tiles > a.n_status) {   // more tiles than the levels can have: a broken invariant
        if (threadIdx.x == 0) atomicOr(a.lv + 3, 1u);
        return;
    }
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    if (tid == 0) s_tile = take_tile(a.tickets);
    if (blockIdx.x == 0 && tid >= 64 && tid < 72) a.next_tickets[(tid - 64) * kTicketStride] = 0;
    __syncthreads();
    const uint32_t tile = s_tile;
    const uint32_t k = tile * kLevelNodes + tid / kWidth;
    const uint32_t level_base = a.lv[1], sbase = a.lv[2];
    const bool live = k < count;

    // the children take the slots 0..n-1 in order, the lanes without one the rest
    const uint32_t c0 = live ? a.items[k] : 0u;
    uint32_t c = 0;
    const bool has = live && slot_child(c0, tid % kWidth, a.cleft, a.cright, a.nt, a.choice, &c);
    const uint32_t group = lane & ~(kWidth - 1u);
    const uint32_t mask = (uint32_t)(__ballot(has) >> group) & 0xFFu;
    const uint32_t below = (1u << (lane - group)) - 1u;
    const uint32_t n = __popc(mask);
    const uint32_t slot = has ? __popc(mask & below) : n + __popc(~mask & below);
    const uint32_t cnt = has ? a.ccount[c] : 0u;
    const rtq_aabb box = a.cbox[c];
    const uint32_t first = has ? a.placed[c].y : 0u;
    const bool expand = has && expandable(a, c, cnt);
    // exclusive sum of the expandable children over the workgroup
    const uint64_t em = __ballot(expand);
    const uint32_t in_wave = __builtin_amdgcn_mbcnt_hi((uint32_t)(em >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)em, 0u));
    if (lane == 0) s_w[wave] = (uint32_t)__popcll(em);
    __syncthreads();
    uint32_t wave_off = 0, total = 0;
#pragma unroll
    for (uint32_t w = 0; w < kWaves; ++w) {
        if (w < wave) wave_off += s_w[w];
        total += s_w[w];
    }

    uint64_t* const st = a.status + sbase;
    if (tid == 0)
        __hip_atomic_store(&st[tile], (tile == 0 ? kLvPre : kLvAgg) | total, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    // (before the look-back: a box in registers through it costs waves per SIMD)
    uint32_t* const img = s_img + (tid / kWidth) * kImageWords;
    wide_boxes(live, has, slot, n, box, box_pad_of(a.bounds[0]), img);

    // counts before this tile: decoupled look-back by wave 0
    if (wave == 0) {
        uint32_t excl = 0;
        if (tile > 0) {
            int64_t top = (int64_t)tile - 1;
            uint32_t polls = 0;
            for (;;) {
                const int64_t idx = top - (int64_t)lane;  // lane 0 = nearest tile
                uint64_t w = kLvPre;                       // before tile 0: an empty prefix
                if (idx >= 0) w = __hip_atomic_load(&st[idx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                for (uint64_t missing; (missing = __ballot((w & kLvState) == 0)) != 0;) {
                    if (++polls > kTilePatience) {
                        const uint32_t m = (uint32_t)__builtin_ctzll(missing);
                        const uint32_t c = expandable_of_tile(a, (uint32_t)top - m);
                        if (lane == m) w = publish_for(&st[idx], kLvAgg | c);
                    } else {
                        __builtin_amdgcn_s_sleep(1);
                    }
                    if ((w & kLvState) == 0)
                        w = __hip_atomic_load(&st[idx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                // nearest tile with counts through it
                const unsigned long long pre = __ballot((w & kLvState) == kLvPre);
                const int stop = pre ? __ffsll((long long)pre) - 1 : 63;
                uint32_t c = (int)lane <= stop ? (uint32_t)w : 0u;
#pragma unroll
                for (int d = 32; d >= 1; d >>= 1) c += __shfl_xor(c, d, 64);
                excl += c;
                if (pre) break;
                top -= 64;
            }
            if (lane == 0)
                __hip_atomic_store(&st[tile], kLvPre | (uint64_t)(excl + total), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        if (lane == 0) s_excl = excl;
    }
    __syncthreads();
    const uint32_t excl = s_excl;
    const uint32_t next_base = level_base + count;
    if (tile == tiles - 1 && tid == 0) {
        uint32_t next_count = excl + total;
        if ((uint64_t)next_base + next_count > a.cap) {
            atomicOr(a.lv + 3, 1u);   // more wide nodes than binary ones: a broken invariant
            next_count = 0;
        }
        a.lv[4] = next_count;
        a.lv[5] = next_base;
        a.lv[6] = sbase + tiles;
    }

    // an empty slot's box is inverted (wide_boxes); should a far ray still enter
    // it, its ref is the leaf of traversal triangle 0 alone: a real triangle, so
    // whatever that test reports is a genuine hit
    uint32_t ref = leaf_ref(0u, 1u);
    if (expand) {
        const uint32_t to = excl + wave_off + in_wave;
        ref = next_base + to;
        if ((uint64_t)next_base + to < a.cap) {
            a.next_items[to] = c;
        } else {
            atomicOr(a.lv + 3, 1u);
        }
    } else if (has) {
        ref = leaf_ref(first, cnt);
    }
    if (live) {
        img[16 + slot] = ref;
        img[24 + slot] = 0;
        // the node's child clusters, for a refit
        a.kids[8ull * (level_base + k) + slot] = has ? c : kNone;
        // the binary traversal node of this node's root cluster (learned order;
        // a scene of one triangle has none)
        if (slot == 0) a.wide_trav[level_base + k] = c0 >= a.nt ? a.placed[c0].w : kNone;
    }
    wave_lds_fence();
    if (live)
        a.nodes[8ull * (level_base + k) + tid % kWidth] = image_part(img, tid % kWidth);
}

// New boxes for the kept 8-wide nodes after a refit: each node's child
// clusters (kids, kNone past the last) quantised again from their refitted
// boxes; child refs stay, learned tables are cleared.
__global__ __launch_bounds__(kThreads) void k_wide_refit(uint32_t n_wide, const uint32_t* __restrict__ kids,
                                                         const rtq_aabb* __restrict__ cbox, uint32_t root,
                                                         float4* __restrict__ nodes) {
    __shared__ __align__(16) uint32_t s_img[kThreads / kWidth * kImageWords];
    const uint32_t tid = threadIdx.x, slot = tid % kWidth;
    const uint32_t k = blockIdx.x * (kThreads / kWidth) + tid / kWidth;
    const bool live = k < n_wide;
    const uint32_t c = live ? kids[8ull * k + slot] : kNone;
    const bool has = c != kNone;
    const uint32_t group = tid & 63u & ~(kWidth - 1u);
    const uint32_t n = __popc((uint32_t)(__ballot(has) >> group) & 0xFFu);
    const rtq_aabb box = cbox[has ? c : 0u];
    uint32_t* const img = s_img + (tid / kWidth) * kImageWords;
    wide_boxes(live, has, slot, n, box, box_pad_of(cbox[root]), img);
    if (live) img[24 + slot] = 0;
    wave_lds_fence();
    if (live && (slot < 4 || slot == 6))
        nodes[8ull * k + slot] = image_part(img, slot);
}

// Before the first level: n_clear words zero from `clear` on (the tile counters
// and status words, then the levels' words), the first level's one node, and
// that node's cluster.
__global__ __launch_bounds__(kThreads) void k_level_init(uint32_t* __restrict__ clear, uint32_t n_clear, uint32_t lv,
                                                         uint32_t* __restrict__ items, uint32_t root) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i < n_clear) clear[i] = i == lv ? 1u : 0u;
    if (i == 0) items[0] = root;
}

inline uint32_t blocks_for(uint64_t n) { return (uint32_t)((n + kThreads - 1) / kThreads); }

}  // namespace

rtq_status wide_cost_bottom(rtq_ctx* ctx, const Scene* s, float* cost, uint32_t* choice, hipStream_t st) {
    for (uint32_t k = 0; k < s->sub_from; ++k) {
        const auto& pr = s->passes[k];
        hipLaunchKernelGGL(k_dp_pass, dim3(blocks_for(pr.second)), dim3(kThreads), 0, st, pr.first, pr.second,
                           s->n_tris, s->params.max_leaf_size, s->cleft, s->cright, s->ccount, s->cbox, cost, choice);
        RTQ_HIP(ctx, hipGetLastError());
    }
    return RTQ_OK;
}

rtq_status wide_cost_top(rtq_ctx* ctx, const Scene* s, float* cost, uint32_t* choice, hipStream_t st) {
    const uint32_t nt = s->n_tris, max_leaf = s->params.max_leaf_size, c_lo = s->passes[s->lds_from].first;
    if (s->sub_from < s->lds_from) {
        hipLaunchKernelGGL(k_dp_subtrees, dim3(s->n_clusters - c_lo + 1), dim3(kSubThreads), 0, st, s->sub_roots,
                           s->sub_list, s->placed, nt, max_leaf, s->cleft, s->cright, s->ccount, s->cbox, cost,
                           choice);
        RTQ_HIP(ctx, hipGetLastError());
    }
    hipLaunchKernelGGL(k_dp_lds, dim3(1), dim3(kLdsThreads), 0, st, top_passes(s), c_lo, s->n_clusters, nt,
                       max_leaf, s->cleft, s->cright, s->ccount, s->cbox, cost, choice);
    RTQ_HIP(ctx, hipGetLastError());
    return RTQ_OK;
}

// Builds s->wide (s->n_wide nodes, s->wide_depth levels) from the cluster
// arrays and the cost table's choices.
rtq_status build_wide(rtq_ctx* ctx, Scene* s, const uint32_t* choice, const rtq_aabb* bounds, hipStream_t st) {
    const uint32_t nc = s->n_clusters;
    const uint32_t root = nc - 1;
    const uint32_t cap = std::max<uint32_t>(s->n_trav, 1);  // wide nodes are a subset of the binary ones
    if (nc > s->n_tris && !choice) return fail(ctx, RTQ_EINTERNAL, "wide collapse without a cost table");
    uint32_t *items = nullptr, *next = nullptr;
    Temps tmp(ctx);
    RTQ_HIP(ctx, tmp.get(&items, cap));
    RTQ_HIP(ctx, tmp.get(&next, cap));
    // tile status words of every level's scan: a level of c nodes takes
    // ceil(c / kLevelNodes) of them, and there are at most depth + 1 levels,
    // the depth no more than the PLOC passes
    const uint32_t max_levels = s->ploc_passes + 1;
    const uint32_t n_status = cap / kLevelNodes + max_levels + 1;
    // two sets of tile counters (a level clears the next one's), the status
    // words, and each level's words (and those of the one after the last)
    constexpr uint32_t kTickets = 2 * kTicketWords, kLvWords = 4;
    const uint32_t lv0 = kTickets + 2 * n_status;
    const uint32_t n_words = lv0 + kLvWords * (max_levels + 1);
    uint32_t* words = nullptr;
    RTQ_HIP(ctx, tmp.get(&words, n_words));
    uint32_t* const tickets = words;
    uint32_t* const lvl = words + lv0;
    // a refit writes the same buffer again (its size depends on the topology only)
    if (!s->wide) RTQ_HIP(ctx, take(s->kept_wide, &s->wide, 8ull * cap));
    if (!s->wide_trav) RTQ_HIP(ctx, take(s->kept_wide_trav, &s->wide_trav, cap));
    if (!s->wide_kids) RTQ_HIP(ctx, take(s->kept_wide_kids, &s->wide_kids, 8ull * cap));
    s->wide_ordered = false;   // the nodes are rewritten with empty tables
    hipLaunchKernelGGL(k_level_init, dim3(blocks_for(n_words)), dim3(kThreads), 0, st, words, n_words, lv0, items,
                       root);
    RTQ_HIP(ctx, hipGetLastError());
    LevelArgs la{};
    la.status = reinterpret_cast<uint64_t*>(words + kTickets);
    la.n_status = n_status;
    la.cap = cap;
    la.max_leaf = s->params.max_leaf_size;
    la.nt = s->n_tris;
    la.bounds = bounds;
    la.cleft = s->cleft;
    la.cright = s->cright;
    la.ccount = s->ccount;
    la.cbox = s->cbox;
    la.choice = choice;
    la.placed = s->placed;
    la.nodes = s->wide;
    la.wide_trav = s->wide_trav;
    la.kids = s->wide_kids;
    // levels top-down, one launch each, several between host reads: a level's
    // words (count, first node, first status word, errors) stay on the device,
    // its launch covers an upper bound of its count (8 children per node, at
    // most cap nodes).  The first group is as long as a tree of so many nodes
    // is likely to be deep (an empty level costs less than a host read).
    constexpr uint32_t kMaxGroup = 16;
    uint32_t group = 2;
    while (group < kMaxGroup && (1ull << (2 * (group - 2))) < cap) ++group;
    uint32_t done = 0, levels = 0, n_wide = 0;
    uint64_t ub = 1;
    for (bool more = true; more;) {
        if (done >= max_levels) return fail(ctx, RTQ_EINTERNAL, "wide collapse: more levels than PLOC passes");
        const uint32_t g0 = done, g1 = std::min(done + group, max_levels);
        for (uint32_t g = g0; g < g1; ++g) {
            la.lv = lvl + kLvWords * g;
            la.items = items;
            la.next_items = next;
            la.tickets = tickets + (g & 1u) * kTicketWords;
            la.next_tickets = tickets + (~g & 1u) * kTicketWords;
            hipLaunchKernelGGL(k_wide_level, dim3((uint32_t)((ub + kLevelNodes - 1) / kLevelNodes)),
                               dim3(kLevelThreads), 0, st, la);
            RTQ_HIP(ctx, hipGetLastError());
            std::swap(items, next);
            ub = std::min<uint64_t>(8 * ub, cap);
        }
        uint32_t h_lv[kLvWords * (kMaxGroup + 1)];
        HostReads rd(ctx, st);
        RTQ_HIP(ctx, rd.add(h_lv, lvl + kLvWords * g0, sizeof(uint32_t) * kLvWords * (g1 - g0 + 1)));
        RTQ_HIP(ctx, rd.wait());
        uint32_t err = 0;
        for (uint32_t g = 0; g < g1 - g0; ++g) {
            const uint32_t* const w = h_lv + kLvWords * g;
            err |= w[3];
            if (w[0] == 0) continue;
            ++levels;
            n_wide = w[1] + w[0];
        }
        if (err) return fail(ctx, RTQ_EINTERNAL, "wide collapse overflow");
        more = h_lv[kLvWords * (g1 - g0)] > 0;
        done = g1;
        group = 4;
    }
    s->n_wide = n_wide;
    s->wide_depth = levels;
    return RTQ_OK;
}

rtq_status refit_wide(rtq_ctx* ctx, Scene* s, hipStream_t st) {
    if (!s->wide || !s->wide_kids) return fail(ctx, RTQ_EINTERNAL, "refit: the scene has no 8-wide nodes");
    if (s->n_wide == 0) return RTQ_OK;
    hipLaunchKernelGGL(k_wide_refit, dim3(blocks_for(8ull * s->n_wide)), dim3(kThreads), 0, st, s->n_wide, s->wide_kids,
                       s->cbox, s->n_clusters - 1, s->wide);
    RTQ_HIP(ctx, hipGetLastError());
    s->wide_ordered = false;   // the tables were cleared
    return RTQ_OK;
}

}  // namespace rtq
