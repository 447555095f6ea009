// Learned child ordering for the binary traversal layout.
//
// A 32 -> 64 -> 64 -> 1 MLP (ReLU, ReLU, logistic) predicts, for a node, a ray
// direction octant and a mode (closest / any hit), the probability that
// entering child 0 first costs less work (node visits + triangle tests until
// the closest hit is certain, or until an occluder is found).
//  - Logs: k_order_log walks sampled rays with the plain traversal and emits,
//    at nodes where both children are hit, the node's features, the label and
//    a weight.
//  - Training: k_mlp_grad (forward + backward of 64 samples per block on FP32
//    matrix instructions, per-block partial gradients) and k_mlp_step
//    (deterministic reduction in block order, Adam), all on the GPU.
//  - Inference: k_order_apply evaluates every (node, octant, mode) with BF16
//    MFMA tiles (v_mfma_f32_32x32x16_bf16, FP32 accumulation) and stores 16
//    decision bits and 16 confidence bits in the node's spare word; with
//    RTQ_TRACE_LEARNED the traversal takes the predicted child first where the
//    confidence bit is set and the nearer child elsewhere.  Only the visit
//    order changes, so hit records are exactly those of the plain traversal.
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstring>
#include <vector>

#include "rtq_internal.hpp"

namespace rtq {
namespace {

constexpr int kIn = 32, kH = 64;
constexpr int kW1 = 0, kB1 = kW1 + kIn * kH, kW2 = kB1 + kH, kB2 = kW2 + kH * kH, kW3 = kB2 + kH, kB3 = kW3 + kH;
constexpr int kNP = kB3 + 1;      // 6337 parameters
constexpr int kSample = kIn + 2;  // features, label, weight
static_assert(kNP == RTQ_ORDER_PARAMS && kSample == RTQ_ORDER_SAMPLE, "model sizes");

__device__ __forceinline__ float area(float ex, float ey, float ez) { return 2.0f * (ex * ey + ey * ez + ez * ex); }

// Features of (node, octant, mode): octant bit k set <=> ray direction < 0 on axis k.
__device__ void node_features(float4 n0, float4 n1, float4 n2, float4 n3, uint4 aux, uint32_t octant, uint32_t any,
                              float* f) {
    const float l0[3] = {n0.x, n0.z, n1.x}, h0[3] = {n0.y, n0.w, n1.y};
    const float l1[3] = {n1.z, n2.x, n2.z}, h1[3] = {n1.w, n2.y, n2.w};
    float lo[3], ext[3], e = 1e-30f;
    for (int k = 0; k < 3; ++k) {
        lo[k] = fminf(l0[k], l1[k]);
        ext[k] = fmaxf(h0[k], h1[k]) - lo[k];
        e = fmaxf(e, ext[k]);
    }
    const float inv = 1.0f / e;
    float s[3];
    for (int k = 0; k < 3; ++k) s[k] = ((octant >> k) & 1u) ? -1.0f : 1.0f;
    f[0] = s[0];
    f[1] = s[1];
    f[2] = s[2];
    f[3] = any ? 1.0f : 0.0f;
    f[4] = (float)aux.w * (1.0f / 32.0f);
    float dot = 0.0f;
    for (int k = 0; k < 3; ++k) {
        f[5 + k] = (l0[k] - lo[k]) * inv;
        f[8 + k] = (h0[k] - lo[k]) * inv;
        f[11 + k] = (l1[k] - lo[k]) * inv;
        f[14 + k] = (h1[k] - lo[k]) * inv;
        const float dc = 0.5f * ((l1[k] + h1[k]) - (l0[k] + h0[k])) * inv;
        f[17 + k] = dc;
        dot += dc * s[k];
        f[27 + k] = ext[k] * inv;
    }
    f[20] = dot;
    const float sp = fmaxf(area(ext[0], ext[1], ext[2]), 1e-30f);
    f[21] = area(h0[0] - l0[0], h0[1] - l0[1], h0[2] - l0[2]) / sp;
    f[22] = area(h1[0] - l1[0], h1[1] - l1[1], h1[2] - l1[2]) / sp;
    f[23] = log2f((float)(aux.y - aux.x) + 1.0f) * (1.0f / 24.0f);
    f[24] = log2f((float)(aux.z - aux.y) + 1.0f) * (1.0f / 24.0f);
    f[25] = (__float_as_uint(n3.x) & kLeafBit) ? 1.0f : 0.0f;
    f[26] = (__float_as_uint(n3.y) & kLeafBit) ? 1.0f : 0.0f;
    f[30] = 0.0f;
    f[31] = 0.0f;
}

__device__ __forceinline__ float sel3(float4 v, int k) { return k == 0 ? v.x : (k == 1 ? v.y : v.z); }

// Watertight hit test returning t (the same test as the traversal kernel).
__device__ bool wt_hit(float4 p0, float4 p1, float4 p2, int kx, int ky, int kz, float opx, float opy, float opz,
                       float sx, float sy, float sz, float tmin, float tmax, float& t) {
    const float Akx = sel3(p0, kx) - opx, Aky = sel3(p0, ky) - opy, Akz = sel3(p0, kz) - opz;
    const float Bkx = sel3(p1, kx) - opx, Bky = sel3(p1, ky) - opy, Bkz = sel3(p1, kz) - opz;
    const float Ckx = sel3(p2, kx) - opx, Cky = sel3(p2, ky) - opy, Ckz = sel3(p2, kz) - opz;
    const float Ax = Akx - sx * Akz, Ay = Aky - sy * Akz;
    const float Bx = Bkx - sx * Bkz, By = Bky - sy * Bkz;
    const float Cx = Ckx - sx * Ckz, Cy = Cky - sy * Ckz;
    float U = Cx * By - Cy * Bx, V = Ax * Cy - Ay * Cx, W = Bx * Ay - By * Ax;
    if (U == 0.0f || V == 0.0f || W == 0.0f) {
        U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
        V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
        W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
    }
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    const float det = (U + V) + W;
    if (det == 0.0f) return false;
    const float T = (U * (sz * Akz) + V * (sz * Bkz)) + W * (sz * Ckz);
    const float tt = T / det;
    if (!(tt >= tmin && tt <= tmax)) return false;
    t = tt;
    return true;
}

// Both children's box tests of a binary node (padded boxes, interval [t0, t1]).
__device__ __forceinline__ void child_hits(float4 n0, float4 n1, float4 n2, const float* o, const float* inv, float t0,
                                           float t1, bool& h0, bool& h1, float& tn0, float& tn1) {
    const float oi[3] = {o[0] * inv[0], o[1] * inv[1], o[2] * inv[2]};
    const float ax0 = fmaf(n0.x, inv[0], -oi[0]), bx0 = fmaf(n0.y, inv[0], -oi[0]);
    const float ay0 = fmaf(n0.z, inv[1], -oi[1]), by0 = fmaf(n0.w, inv[1], -oi[1]);
    const float az0 = fmaf(n1.x, inv[2], -oi[2]), bz0 = fmaf(n1.y, inv[2], -oi[2]);
    const float ax1 = fmaf(n1.z, inv[0], -oi[0]), bx1 = fmaf(n1.w, inv[0], -oi[0]);
    const float ay1 = fmaf(n2.x, inv[1], -oi[1]), by1 = fmaf(n2.y, inv[1], -oi[1]);
    const float az1 = fmaf(n2.z, inv[2], -oi[2]), bz1 = fmaf(n2.w, inv[2], -oi[2]);
    tn0 = fmaxf(fmaxf(fminf(ax0, bx0), fminf(ay0, by0)), fmaxf(fminf(az0, bz0), t0));
    const float tf0 = fminf(fminf(fmaxf(ax0, bx0), fmaxf(ay0, by0)), fminf(fmaxf(az0, bz0), t1));
    tn1 = fmaxf(fmaxf(fminf(ax1, bx1), fminf(ay1, by1)), fmaxf(fminf(az1, bz1), t0));
    const float tf1 = fminf(fminf(fmaxf(ax1, bx1), fmaxf(ay1, by1)), fminf(fmaxf(az1, bz1), t1));
    h0 = tn0 <= tf0;
    h1 = tn1 <= tf1;
}

constexpr uint32_t kLogStack = 96;
constexpr uint32_t kLogRecords = 32;       // samples of a ray kept until its wave ends
constexpr uint64_t kLogLaunch = 1u << 24;  // logged rays per launch
constexpr uint32_t kLogBudget = 1u << 14;  // node visits + triangle tests per sub-traversal
// Lanes of a ray that prices 2 or 3 levels at a time: 2 + 4 or 2 + 4 + 8 of
// them, rounded up to a power of two.
constexpr uint32_t log_lanes(int ahead) { return ahead == 2 ? 8 : 16; }

struct LogRay {
    float o[3], inv[3], tmin, tmax;
    int kx, ky, kz;
    float sx, sy, sz, opx, opy, opz;
};

// Traversal of the subtree at `ref` (nearer child first) over [R.tmin, tmax].
// Closest (any = false): returns the leaf-order index of the closest hit and
// shrinks tmax to its t.  Any hit: returns the first hit found.  kNone = no
// hit.  cost = node visits + triangle tests; ok = false when the walk ran past
// kLogBudget or kLogStack entries.  Stack entry k is stack[k * stride] in LDS.
__device__ uint32_t log_walk(const float4* __restrict__ nodes, const float4* __restrict__ tris, const LogRay& R,
                             uint32_t ref, bool any, uint32_t* stack, uint32_t stride, float& tmax, uint32_t& cost,
                             bool& ok) {
    uint32_t sp = 0, cur = ref, target = kNone;
    cost = 0;
    ok = true;
    for (;;) {
        if (++cost > kLogBudget) {
            ok = false;
            return kNone;
        }
        if (!(cur & kLeafBit)) {
            const float4* nd = nodes + 4ull * cur;
            bool h0, h1;
            float tn0, tn1;
            child_hits(nd[0], nd[1], nd[2], R.o, R.inv, R.tmin, tmax, h0, h1, tn0, tn1);
            const float4 n3 = nd[3];
            const uint32_t r0 = __float_as_uint(n3.x), r1 = __float_as_uint(n3.y);
            if (h0 && h1) {
                if (sp >= kLogStack) {
                    ok = false;
                    return kNone;
                }
                const bool f0 = tn0 <= tn1;
                stack[sp++ * stride] = f0 ? r1 : r0;
                cur = f0 ? r0 : r1;
                continue;
            }
            if (h0 || h1) {
                cur = h0 ? r0 : r1;
                continue;
            }
        } else {
            const uint32_t first = (cur >> 3) & 0x0FFFFFFFu, cnt = (cur & 7u) + 1u;
            cost += cnt - 1;  // the leaf's own step counted one test
            for (uint32_t k = 0; k < cnt; ++k) {
                const float4* tp = tris + 3ull * (first + k);
                float t;
                if (wt_hit(tp[0], tp[1], tp[2], R.kx, R.ky, R.kz, R.opx, R.opy, R.opz, R.sx, R.sy, R.sz, R.tmin, tmax,
                           t) &&
                    (t < tmax || target == kNone)) {
                    tmax = t;
                    target = first + k;
                    if (any) return target;
                }
            }
        }
        if (sp == 0) return target;
        cur = stack[--sp * stride];
    }
}

// Sample `slot`: the features of binary node `node` for the octant and mode,
// the label and the weight.
__device__ void emit(float* __restrict__ out, uint32_t cap, uint32_t slot, const float4* __restrict__ nodes,
                     const uint4* __restrict__ aux, uint32_t node, uint32_t octant, uint32_t any, bool child0_first,
                     float weight) {
    if (slot >= cap) return;
    const float4* nd = nodes + 4ull * node;
    float f[kIn];
    node_features(nd[0], nd[1], nd[2], nd[3], aux[node], octant, any, f);
    float* o = out + (size_t)slot * kSample;
    for (int k = 0; k < kIn; ++k) o[k] = f[k];
    o[kIn] = child0_first ? 1.0f : 0.0f;
    o[kIn + 1] = weight;
}

// The first node from `ref` down that has both children hit over the ray's
// interval, following the only hit child to it; its child refs.  kNone: a leaf
// or a node without a hit child comes first.
__device__ uint32_t next_decision(const float4* __restrict__ nodes, const LogRay& R, uint32_t ref, uint32_t& r0,
                                  uint32_t& r1) {
    while (!(ref & kLeafBit)) {
        const float4* nd = nodes + 4ull * ref;
        const float4 n3 = nd[3];
        bool h0, h1;
        float tn0, tn1;
        child_hits(nd[0], nd[1], nd[2], R.o, R.inv, R.tmin, R.tmax, h0, h1, tn0, tn1);
        r0 = __float_as_uint(n3.x);
        r1 = __float_as_uint(n3.y);
        if (h0 && h1) return ref;
        if (!(h0 || h1)) break;
        ref = h0 ? r0 : r1;
    }
    return kNone;
}

// Samples of one ray every `stride`: from the root, each node whose two
// children are both hit is priced in both visit orders with sub-traversals
// (node visits + triangle tests until the closest hit is certain, or until an
// occluder is found for any-hit rays); label = the cheaper child first, weight
// log2(1 + cost difference), no sample on a tie.  The walk continues into the
// cheaper child and stops where no hit lies below it.
// Two lanes price a node: the even one child 0 first, the odd one child 1
// first.  A ray has the pairs of AHEAD levels of such nodes, the 1, 2 or 4 that
// the walk can come to: they are priced together, which takes about as long as
// the first level alone, and the ones off the walk's way are dropped.  The
// stacks lie in LDS, `levels` entries per lane.  A ray's samples wait in
// registers' scratch, so that a wave takes their slots with one atomic at its
// end: atomics of every sample on one word serialise.
// The chains of dependent node loads of a ray's walks bound it.  300,000
// occluded triangles, any-hit rays (closest-hit), with 1, 2 and 3 levels at a
// time: 6,250 rays 0.63 (1.11), 0.51 (0.95), 0.35 (0.65) ms; 25,000 rays 0.88
// (1.48), 0.58 (0.99), 0.58 (0.95); 200,000 rays 2.53 (4.97), 2.36 (4.03), 2.90
// (4.78).
template <int AHEAD>
__global__ __launch_bounds__(64) void k_order_log(const float4* __restrict__ nodes, const uint4* __restrict__ aux,
                                                  const float4* __restrict__ tris, const rtq_ray* __restrict__ rays,
                                                  uint32_t n, uint32_t stride, uint32_t any, float* __restrict__ out, uint32_t cap,
                                                  uint32_t* __restrict__ count) {
    extern __shared__ uint32_t s_log[];
    constexpr uint32_t kGroup = log_lanes(AHEAD), kRays = 64 / kGroup;
    const uint32_t lane = threadIdx.x;
    const uint32_t sub = lane % kGroup, lead = lane - sub;
    // the lane's level and the choices down to it: the child taken at each
    // level before it, then the child it prices first (0 as the level: idle)
    const uint32_t level = sub < 2 ? 1u : sub < 6 ? 2u : AHEAD > 2 && sub < 14 ? 3u : 0u;
    const uint32_t way = sub - (level == 2 ? 2u : level == 3 ? 6u : 0u);
    const bool second = way & 1u;           // prices child 1 first
    uint32_t* const stack = s_log + lane;   // [levels][64]
    uint2 rec[kLogRecords];                 // node | child 0 first << 31, weight (a ray's first lane)
    const uint64_t r = ((uint64_t)blockIdx.x * kRays + lane / kGroup) * stride;
    uint32_t n_rec = 0, octant = 0;
    if (r < n) {
        const rtq_ray ray = rays[r];
        LogRay R;
        for (int k = 0; k < 3; ++k) {
            const float d = fabsf(ray.d[k]) < 1e-30f ? copysignf(1e-30f, ray.d[k]) : ray.d[k];
            R.o[k] = ray.o[k];
            R.inv[k] = 1.0f / d;
        }
        R.tmin = ray.tmin;
        R.tmax = ray.tmax;
        const float ax = fabsf(ray.d[0]), ay = fabsf(ray.d[1]), az = fabsf(ray.d[2]);
        int kz = 0;
        float m = ax;
        if (ay > m) { kz = 1; m = ay; }
        if (az > m) kz = 2;
        int kx = kz + 1 == 3 ? 0 : kz + 1;
        int ky = kx + 1 == 3 ? 0 : kx + 1;
        const float dkz = ray.d[kz];
        if (dkz < 0.0f) { const int tmp = kx; kx = ky; ky = tmp; }
        R.kx = kx;
        R.ky = ky;
        R.kz = kz;
        R.sx = ray.d[kx] / dkz;
        R.sy = ray.d[ky] / dkz;
        R.sz = 1.0f / dkz;
        R.opx = ray.o[kx];
        R.opy = ray.o[ky];
        R.opz = ray.o[kz];
        octant = (ray.d[0] < 0.0f ? 1u : 0u) | (ray.d[1] < 0.0f ? 2u : 0u) | (ray.d[2] < 0.0f ? 4u : 0u);
        // Walk from the root along the child each decision visits first: nothing
        // has been visited before such a node, so its interval is the ray's own.
        // (An empty interval or a zero direction hits nothing: no walk.)
        uint32_t cur = ray.tmin <= ray.tmax && dkz != 0.0f ? 0u : kLeafBit;
        for (bool more = true; more;) {
            uint32_t r0 = 0, r1 = 0;
            uint32_t at = next_decision(nodes, R, cur, r0, r1);   // the node the lane prices
            if (at == kNone) break;
#pragma unroll
            for (uint32_t l = 1; l < (uint32_t)AHEAD; ++l)
                if (level > l && at != kNone)
                    at = next_decision(nodes, R, (way >> (level - l)) & 1u ? r1 : r0, r0, r1);
            // the lane's first child, and for closest-hit rays the other one
            // with the interval the first left (an occluder below the first
            // child ends an any-hit ray there, and the other lane's walk gives
            // the other child's cost)
            uint32_t cost = 0, rest = 0;
            bool found = false, ok = true, ok2 = true;
            if (level > 0 && at != kNone) {
                float t = R.tmax;
                found = log_walk(nodes, tris, R, second ? r1 : r0, any, stack, 64, t, cost, ok) != kNone;
                if (!any) log_walk(nodes, tris, R, second ? r0 : r1, false, stack, 64, t, rest, ok2);
            }
            const uint32_t flags = (found ? 1u : 0u) | (ok && ok2 ? 2u : 0u);
            cost += rest;
            uint32_t choice = 0;   // the children taken since these walks
#pragma unroll
            for (uint32_t l = 0; l < (uint32_t)AHEAD; ++l) {
                const int from = (int)(lead + (2u << l) - 2u + 2u * choice);
                const uint32_t node = __shfl(at, from, 64);
                const uint32_t c0 = __shfl(cost, from, 64), c1 = __shfl(cost, from + 1, 64);
                const uint32_t g0 = __shfl(flags, from, 64), g1 = __shfl(flags, from + 1, 64);
                const uint32_t n0 = __shfl(r0, from, 64), n1 = __shfl(r1, from, 64);
                const bool f0 = g0 & 1u, f1 = g1 & 1u;
                // past the walk's end, a walk past its bounds, or no hit below
                // either child (every order visits the same nodes)
                if (!more || node == kNone || !(g0 & g1 & 2u) || !(f0 || f1)) {
                    more = false;
                    continue;
                }
                const uint32_t cost01 = any && !f0 ? c0 + c1 : c0, cost10 = any && !f1 ? c1 + c0 : c1;
                if (cost01 != cost10 && sub == 0) {
                    const float diff = (float)(cost01 > cost10 ? cost01 - cost10 : cost10 - cost01);
                    const float weight = log2f(1.0f + diff);
                    if (n_rec < kLogRecords) {
                        rec[n_rec++] = make_uint2(node | (cost01 < cost10 ? kLeafBit : 0u), __float_as_uint(weight));
                    } else {   // a path of more levels than the records hold
                        emit(out, cap, atomicAdd(count, 1u), nodes, aux, node, octant, any, cost01 < cost10, weight);
                    }
                }
                const bool go0 = cost01 <= cost10;
                more = go0 ? f0 : f1;
                cur = go0 ? n0 : n1;
                choice = 2 * choice + (go0 ? 0u : 1u);
            }
        }
    }
    // the wave's slots, then each ray's samples by its first two lanes in turn
    const uint32_t incl = wave_inclusive_sum(n_rec);
    const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    if (all == 0) return;
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(count, all);
    base = __shfl(base, 0, 64) + __shfl(incl - n_rec, (int)lead, 64);
    const uint32_t have = __shfl(n_rec, (int)lead, 64);
    for (uint32_t k = 0; k < kLogRecords; k += 2) {
        if (__ballot(k < n_rec) == 0) break;
        // the first lane's records k and k + 1, one for each lane of the pair
        const uint2 a0 = rec[k], a1 = rec[k + 1];
        const uint32_t sx = __shfl(a1.x, (int)lead, 64), sy = __shfl(a1.y, (int)lead, 64);
        const uint2 s = sub == 1 ? make_uint2(sx, sy) : a0;
        if (sub < 2 && k + sub < have)
            emit(out, cap, base + k + sub, nodes, aux, s.x & ~kLeafBit, octant, any, (s.x & kLeafBit) != 0,
                 __uint_as_float(s.y));
    }
}

// ---- training ----------------------------------------------------------------

constexpr int kTB = 64;  // samples per block
constexpr int kGradThreads = 1024;
constexpr uint32_t kGradLaunch = 1u << 16;   // blocks per launch
// Row lengths of the LDS arrays: 20 or 44 mod 64 words, so that the matrix
// operands read along a row (16 rows x 4 columns of a wave) lie in 64 distinct
// banks and the ones read down a column (4 rows x 16 columns) in at most two
// each.
constexpr int kLdX = 44, kLdH = 84;

typedef float f32x4 __attribute__((ext_vector_type(4)));

// 16 x 16 tile of A B + C, FP32: lane l holds A[l % 16][4 t + l / 16] and
// B[4 t + l / 16][l % 16] of step t, and D[4 (l / 16) + r][l % 16] in register
// r.  The instruction adds the 4 products of a step in order, each with one
// rounding, so a chain of steps gives the bits of a loop of fmaf over k
// (checked for ordinary, subnormal and zero products).
__device__ __forceinline__ f32x4 mfma_step(float a, float b, f32x4 acc) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
}

struct GradLds {
    float x[kTB * kLdX];    // features [sample][feature]
    float h1[kTB * kLdH];   // activations [sample][unit]
    float h2[kTB * kLdH];
    float d1[kTB * kLdH];   // gradients of the layers' inputs to ReLU [sample][unit]
    float d2[kTB * kLdH];
    float w2[kH * kLdH];    // [in][out]
    float y[kTB], w[kTB], z[kTB], dz[kTB], loss[kTB], w3[kH];
};
static_assert(sizeof(GradLds) <= 160 * 1024, "one workgroup per CU");

// The order of an epoch: position i of a launch holds sample (base + i * mul) % n,
// base < n, mul <= n, and i (under 64 kGradLaunch = 2^22) times mul under 2^53: it
// is exact in a double, its quotient by n wrong by one at most (a 64-bit remainder
// is 1,000 cycles).  Training has n < 2^31, a single gradient n < 2^32 and mul = 1.
struct SampleOrder {
    uint32_t n, base, mul;
    double inv_n;
    __device__ __forceinline__ uint32_t operator[](uint32_t i) const {
        const uint64_t x = (uint64_t)i * mul;
        const uint32_t q = (uint32_t)((double)x * inv_n);
        int64_t r = (int64_t)(x - (uint64_t)q * n);
        r += r < 0 ? (int64_t)n : 0;
        r -= r >= (int64_t)n ? (int64_t)n : 0;
        r += base;
        return (uint32_t)(r >= (int64_t)n ? r - n : r);
    }
};

// Forward + backward of up to 64 samples at the order's positions from 64 times
// the block on; writes the block's gradient sums and its sum of weighted losses.
// Loss of a sample: weight * BCE(sigmoid(z), label).  Every layer's product is
// 16 tiles of 16 x 16, one per wave, on the FP32 matrix instruction.
// A training step has few blocks (16 at the default batch of 1,024), so its time
// is one block's chain of phases, bound by its CU's matrix and LDS rate: PARTS
// workgroups share a block.  Each goes forward alone and takes 64 / PARTS of the
// columns backward, so the sums are the same.  98.6 us a step with a block in one
// wave (a sample or a column per lane, each product a loop over LDS), 11.5 with
// one workgroup per block, 8.7 with four and every load issued at the start.
template <int PARTS>
__global__ __launch_bounds__(kGradThreads) void k_mlp_grad(const float* __restrict__ P,
                                                           const float* __restrict__ samples, SampleOrder order,
                                                           uint32_t count, float* __restrict__ partial,
                                                           float* __restrict__ loss_part) {
    constexpr int kTiles = 4 / PARTS;     // column tiles of a workgroup going backward
    const uint32_t block = blockIdx.x / PARTS, part = blockIdx.x % PARTS;
    __shared__ GradLds L;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 15, g = lane >> 4;          // operand column and k group
    const int mt = 16 * (wave >> 2), nt = 16 * (wave & 3);   // the wave's tile
    // every load of the block at once: the samples' rows (16 threads each), layer
    // 1's weights straight into operand registers, layer 2's for LDS
    const int s = tid >> 4;
    const bool valid = block * kTB + s < count;
    const float* row = samples + (size_t)(valid ? order[block * kTB + s] : 0u) * kSample;
    float v[3], w1[kIn / 4], w2[kH * kH / kGradThreads];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const int k = (tid & 15) + 16 * r;
        v[r] = valid && k < kSample ? row[k] : 0.0f;
    }
#pragma unroll
    for (int r = 0; r < kH * kH / kGradThreads; ++r) w2[r] = P[kW2 + tid + r * kGradThreads];
#pragma unroll
    for (int t = 0; t < kIn / 4; ++t) w1[t] = P[kW1 + (4 * t + g) * kH + nt + c];
    const float b1 = P[kB1 + nt + c], b2 = P[kB2 + nt + c], w3 = P[kW3 + nt + c];
    const float b3 = c == 0 ? P[kB3] : 0.0f;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const int k = (tid & 15) + 16 * r;
        if (k < kIn) L.x[s * kLdX + k] = v[r];
        if (k == kIn) L.y[s] = v[r];
        if (k == kIn + 1) L.w[s] = v[r];
    }
#pragma unroll
    for (int r = 0; r < kH * kH / kGradThreads; ++r) {
        const int i = tid + r * kGradThreads;
        L.w2[(i / kH) * kLdH + i % kH] = w2[r];
    }
    if (wave < 4 && g == 0) L.w3[nt + c] = w3;
    __syncthreads();
    float h1[4], h2[4];   // the wave's tile of both layers
    {
        f32x4 acc = {b1, b1, b1, b1};
#pragma unroll
        for (int t = 0; t < kIn / 4; ++t) acc = mfma_step(L.x[(mt + c) * kLdX + 4 * t + g], w1[t], acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            h1[r] = fmaxf(acc[r], 0.0f);
            L.h1[(mt + 4 * g + r) * kLdH + nt + c] = h1[r];
        }
    }
    __syncthreads();
    {
        f32x4 acc = {b2, b2, b2, b2};
#pragma unroll
        for (int t = 0; t < kH / 4; ++t)
            acc = mfma_step(L.h1[(mt + c) * kLdH + 4 * t + g], L.w2[(4 * t + g) * kLdH + nt + c], acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            h2[r] = fmaxf(acc[r], 0.0f);
            L.h2[(mt + 4 * g + r) * kLdH + nt + c] = h2[r];
        }
    }
    __syncthreads();
    if (wave < 4) {   // output layer (in a tile's first column) of the wave's 16 samples
        const int m0 = 16 * wave;
        f32x4 acc = {b3, b3, b3, b3};
#pragma unroll
        for (int t = 0; t < kH / 4; ++t)
            acc = mfma_step(L.h2[(m0 + c) * kLdH + 4 * t + g], c == 0 ? L.w3[4 * t + g] : 0.0f, acc);
        if (c == 0)
#pragma unroll
            for (int r = 0; r < 4; ++r) L.z[m0 + 4 * g + r] = acc[r];
        wave_lds_fence();
        if (lane < 16) {   // dL/dz = w (sigmoid(z) - y)
            const int m = m0 + lane;
            const float p = 1.0f / (1.0f + expf(-L.z[m]));
            L.dz[m] = block * kTB + m < count ? L.w[m] * (p - L.y[m]) : 0.0f;
        }
    }
    __syncthreads();
    // dH2 = dz * w3 * (h2 > 0)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = mt + 4 * g + r;
        L.d2[m * kLdH + nt + c] = h2[r] > 0.0f ? L.dz[m] * w3 : 0.0f;
    }
    __syncthreads();
    // backward: the part's columns, a tile of each product per wave
    float* out = partial + (size_t)block * kNP;
    const int col = 16 * kTiles * (int)part;              // the first of them
    const int bt = 16 * (wave / kTiles % 4), bn = col + 16 * (wave % kTiles);
    if (wave < 4 * kTiles) {   // dH1 = (dH2 W2^T) * (h1 > 0)
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < kH / 4; ++t)
            acc = mfma_step(L.d2[(bt + c) * kLdH + 4 * t + g], L.w2[(bn + c) * kLdH + 4 * t + g], acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = bt + 4 * g + r;
            L.d1[m * kLdH + bn + c] = L.h1[m * kLdH + bn + c] > 0.0f ? acc[r] : 0.0f;
        }
    }
    // dW2[k][j] = sum_s h1[s][k] dh2[s][j], by other waves where there are any
    if (PARTS == 1 || (wave >= 4 && wave < 8)) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < kTB / 4; ++t)
            acc = mfma_step(L.h1[(4 * t + g) * kLdH + bt + c], L.d2[(4 * t + g) * kLdH + bn + c], acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) out[kW2 + (bt + 4 * g + r) * kH + bn + c] = acc[r];
    }
    const int j = col + lane;                             // a column per lane
    const bool mine = lane < 16 * kTiles;
    // the sums that need no dH1 beside it, or after it with the others
    const auto column_sums = [&](int w) {
        if (w == 0 && mine) {          // dw3[j] = sum_s h2[s][j] dz[s]
            float acc = 0.0f;
#pragma unroll 8
            for (int s = 0; s < kTB; ++s) acc = fmaf(L.h2[s * kLdH + j], L.dz[s], acc);
            out[kW3 + j] = acc;
        } else if (w == 1 && mine) {   // db2[j] = sum_s dh2[s][j]
            float acc = 0.0f;
#pragma unroll 8
            for (int s = 0; s < kTB; ++s) acc += L.d2[s * kLdH + j];
            out[kB2 + j] = acc;
        } else if (w == 2 && part == 0) {   // db3 = sum of dz (lane 0) and the block's loss (lane 1)
            // BCE with logits: max(z, 0) - z y + log(1 + e^-|z|)
            const float z = L.z[lane];
            const float loss = L.w[lane] * ((fmaxf(z, 0.0f) - z * L.y[lane]) + log1pf(expf(-fabsf(z))));
            L.loss[lane] = block * kTB + lane < count ? loss : 0.0f;
            wave_lds_fence();
            const float* sum = lane == 0 ? L.dz : L.loss;
            float acc = 0.0f;
            if (lane < 2)
#pragma unroll 8
                for (int s = 0; s < kTB; ++s) acc += sum[s];
            if (lane == 0) out[kB3] = acc;
            if (lane == 1) loss_part[block] = acc;
        }
    };
    if (PARTS > 1) column_sums(wave - 8);
    __syncthreads();
    if (wave < 2 * kTiles) {   // dW1[k][j] = sum_s x[s][k] dh1[s][j]
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < kTB / 4; ++t)
            acc = mfma_step(L.x[(4 * t + g) * kLdX + bt + c], L.d1[(4 * t + g) * kLdH + bn + c], acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) out[kW1 + (bt + 4 * g + r) * kH + bn + c] = acc[r];
    } else if (wave == 11) {   // db1[j] = sum_s dh1[s][j]
        float acc = 0.0f;
        if (mine)
#pragma unroll 8
            for (int s = 0; s < kTB; ++s) acc += L.d1[s * kLdH + j];
        if (mine) out[kB1 + j] = acc;
    } else if (PARTS == 1) {
        column_sums(wave - 8);
    }
}

// Workgroups per block of 64 samples: four while the chip has the CUs.
int grad_parts(const rtq_ctx* ctx, uint32_t blocks) { return 4 * blocks <= (uint32_t)std::max(ctx->n_cu, 1) ? 4 : 1; }

hipError_t queue_grad(const rtq_ctx* ctx, const float* params, const float* samples, const SampleOrder& order,
                      uint32_t count, float* partial, float* loss_part, hipStream_t st) {
    const uint32_t blocks = (count + kTB - 1) / kTB;
    const int parts = grad_parts(ctx, blocks);
    // (a launch has fewer than 2^32 threads, a sample 16 of them or more)
    for (uint32_t b = 0; b < blocks; b += kGradLaunch) {
        SampleOrder part = order;
        part.base = (uint32_t)((order.base + (uint64_t)(kTB * b) * order.mul) % order.n);
        hipLaunchKernelGGL(parts == 4 ? &k_mlp_grad<4> : &k_mlp_grad<1>, dim3(std::min(blocks - b, kGradLaunch) * parts),
                           dim3(kGradThreads), 0, st, params, samples, part, count - kTB * b,
                           partial + (size_t)b * kNP, loss_part + b);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// The blocks' gradients of parameter j, summed in block order (deterministic)
// and scaled by 1 / samples.
__device__ __forceinline__ float grad_of(const float* __restrict__ partial, uint32_t blocks, float scale, int j) {
    float acc = 0.0f;
#pragma unroll 16
    for (uint32_t b = 0; b < blocks; ++b) acc += partial[(size_t)b * kNP + j];
    return acc * scale;
}

constexpr int kParamThreads = 64;   // 100 workgroups for the 6,337 parameters
constexpr uint32_t kParamBlocks = (kNP + kParamThreads - 1) / kParamThreads;

__global__ __launch_bounds__(kParamThreads) void k_mlp_reduce(const float* __restrict__ partial, uint32_t blocks,
                                                              float scale, float* __restrict__ grad) {
    const int j = blockIdx.x * kParamThreads + threadIdx.x;
    if (j < kNP) grad[j] = grad_of(partial, blocks, scale, j);
}

// The reduction and the Adam update in one launch (two launches took 9.6 us a
// step at 16 blocks, this one 3.8).
__global__ __launch_bounds__(kParamThreads) void k_mlp_step(const float* __restrict__ partial, uint32_t blocks,
                                                            float scale, float* __restrict__ P, float* __restrict__ M,
                                                            float* __restrict__ V, float lr, float b1, float b2,
                                                            float eps, float c1, float c2) {
    const int j = blockIdx.x * kParamThreads + threadIdx.x;
    if (j >= kNP) return;
    const float m0 = M[j], v0 = V[j], p0 = P[j];
    const float g = grad_of(partial, blocks, scale, j);
    const float m = b1 * m0 + (1.0f - b1) * g;
    const float v = b2 * v0 + (1.0f - b2) * g * g;
    M[j] = m;
    V[j] = v;
    P[j] = p0 - lr * (m / c1) / (sqrtf(v / c2) + eps);
}

// ---- BF16 MFMA inference ---------------------------------------------------------

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

__device__ __forceinline__ uint16_t to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even (finite inputs)
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ bf16x8 load8(const uint16_t* p) {
    const uint4 v = *reinterpret_cast<const uint4*>(p);
    return __builtin_bit_cast(bf16x8, v);
}

constexpr int kIW = 4;  // waves per inference block

// The bf16 operand arrays come first and have sizes that are multiples of 16 B,
// so every 8-element (16-B) operand load is 16-B aligned.
struct alignas(16) InferLds {
    uint16_t w1t[kH][kIn];       // W1 transposed (hidden, feature), bf16
    uint16_t w2t[kH][kH];        // W2 transposed (out, in), bf16
    uint16_t x[kIW][32][kIn];    // per wave: 32 samples x 32 features
    uint16_t h1[kIW][32][kH];    // per wave: layer-1 activations
    float red[kIW][32][33];      // per wave: layer-3 partial products
    float b1[kH], b2[kH], w3[kH];
    float b3;
};
static_assert(offsetof(InferLds, x) % 16 == 0 && offsetof(InferLds, h1) % 16 == 0, "operand alignment");

__device__ void load_weights(InferLds& L, const float* P) {
    for (int i = threadIdx.x; i < kIn * kH; i += blockDim.x) {
        const int k = i / kH, j = i % kH;
        L.w1t[j][k] = to_bf16(P[kW1 + i]);
    }
    for (int i = threadIdx.x; i < kH * kH; i += blockDim.x) {
        const int k = i / kH, j = i % kH;
        L.w2t[j][k] = to_bf16(P[kW2 + i]);
    }
    for (int i = threadIdx.x; i < kH; i += blockDim.x) {
        L.b1[i] = P[kB1 + i];
        L.b2[i] = P[kB2 + i];
        L.w3[i] = P[kW3 + i];
    }
    if (threadIdx.x == 0) L.b3 = P[kB3];
}

// The wave's 32 samples (rows of L.x[w]) through the network; returns the
// logit of sample (lane & 31) in every lane.
// 32x32x16 operand layout: A row m = lane % 32 holds k = 8 * (lane / 32) + 0..7;
// B column n = lane % 32 likewise; D element (m, n) of register r sits in lane
// n + 32 * ((m / 4) % 2) with r = (m % 4) + 4 * (m / 8).
__device__ float mlp_tile(InferLds& L, int w, int lane) {
    const int row = lane & 31, half = lane >> 5;
    f32x16 acc[2] = {};
#pragma unroll
    for (int ks = 0; ks < kIn / 16; ++ks) {
        const bf16x8 a = load8(&L.x[w][row][16 * ks + 8 * half]);
#pragma unroll
        for (int tn = 0; tn < 2; ++tn) {
            const bf16x8 b = load8(&L.w1t[32 * tn + row][16 * ks + 8 * half]);
            acc[tn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[tn], 0, 0, 0);
        }
    }
#pragma unroll
    for (int tn = 0; tn < 2; ++tn) {
        const int ncol = 32 * tn + row;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = (r & 3) + 4 * half + 8 * (r >> 2);
            L.h1[w][m][ncol] = to_bf16(fmaxf(acc[tn][r] + L.b1[ncol], 0.0f));
        }
    }
    __syncthreads();
    f32x16 acc2[2] = {};
#pragma unroll
    for (int ks = 0; ks < kH / 16; ++ks) {
        const bf16x8 a = load8(&L.h1[w][row][16 * ks + 8 * half]);
#pragma unroll
        for (int tn = 0; tn < 2; ++tn) {
            const bf16x8 b = load8(&L.w2t[32 * tn + row][16 * ks + 8 * half]);
            acc2[tn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc2[tn], 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int m = (r & 3) + 4 * half + 8 * (r >> 2);
        float v = 0.0f;
#pragma unroll
        for (int tn = 0; tn < 2; ++tn) {
            const int ncol = 32 * tn + row;
            v = fmaf(fmaxf(acc2[tn][r] + L.b2[ncol], 0.0f), L.w3[ncol], v);
        }
        L.red[w][m][row] = v;
    }
    __syncthreads();
    float z = L.b3;
    for (int c = 0; c < 32; ++c) z += L.red[w][row][c];
    return z;
}

// Probabilities for M feature rows (fp32 in, fp32 out): the MFMA path on any samples.
__global__ __launch_bounds__(64 * kIW) void k_mlp_infer(const float* __restrict__ P, const float* __restrict__ X,
                                                        uint32_t M, uint32_t stride, float* __restrict__ prob) {
    __shared__ InferLds L;
    load_weights(L, P);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t tiles = (M + 31) / 32;
    const uint32_t per_iter = gridDim.x * kIW;
    // every wave of the block runs the same number of iterations (barriers inside)
    const uint32_t iters = (tiles + per_iter - 1) / per_iter;
    __syncthreads();
    for (uint32_t it = 0; it < iters; ++it) {
        const uint32_t tile = it * per_iter + blockIdx.x * kIW + w;
        if (lane < 32) {
            const uint32_t sidx = tile * 32 + lane;
            for (int k = 0; k < kIn; ++k)
                L.x[w][lane][k] = to_bf16((tile < tiles && sidx < M) ? X[(size_t)sidx * stride + k] : 0.0f);
        }
        __syncthreads();
        const float z = mlp_tile(L, w, lane);
        const uint32_t sidx = tile * 32 + lane;
        if (lane < 32 && tile < tiles && sidx < M) prob[sidx] = 1.0f / (1.0f + expf(-z));
        __syncthreads();
    }
}

// Order word of every binary node: 16 samples per node (8 octants x 2 modes);
// bit (any * 8 + octant) set when child 0 should go first, bit 16 + (any * 8 +
// octant) set when the logit's magnitude reaches zmin[any] (the decision is
// used; an infinite zmin never sets it).
__global__ __launch_bounds__(64 * kIW) void k_order_apply(const float* __restrict__ P, float4* __restrict__ nodes,
                                                          const uint4* __restrict__ aux, uint32_t n_nodes,
                                                          float zmin_closest, float zmin_any) {
    __shared__ InferLds L;
    load_weights(L, P);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t tiles = (n_nodes + 1) / 2;  // 2 nodes x 16 samples per tile
    const uint32_t per_iter = gridDim.x * kIW;
    const uint32_t iters = (tiles + per_iter - 1) / per_iter;
    __syncthreads();
    for (uint32_t it = 0; it < iters; ++it) {
        const uint32_t tile = it * per_iter + blockIdx.x * kIW + w;
        const uint32_t node = tile * 2 + ((lane >> 4) & 1);
        const bool live = lane < 32 && tile < tiles && node < n_nodes;
        if (lane < 32) {
            float f[kIn];
            if (live) {
                const float4* nd = nodes + 4ull * node;
                node_features(nd[0], nd[1], nd[2], nd[3], aux[node], lane & 7, (lane >> 3) & 1, f);
            } else {
                for (int k = 0; k < kIn; ++k) f[k] = 0.0f;
            }
            for (int k = 0; k < kIn; ++k) L.x[w][lane][k] = to_bf16(f[k]);
        }
        __syncthreads();
        const float z = mlp_tile(L, w, lane);
        // a NaN logit fails both tests: the node keeps the nearer-child order
        const uint64_t bits = __ballot(live && z > 0.0f);
        const uint64_t sure = __ballot(live && fabsf(z) >= (((lane >> 3) & 1) ? zmin_any : zmin_closest));
        if ((lane == 0 || lane == 16) && live) {
            const uint32_t word = ((uint32_t)(bits >> lane) & 0xFFFFu) | (((uint32_t)(sure >> lane) & 0xFFFFu) << 16);
            float4* n3 = nodes + 4ull * node + 3;
            n3->z = __uint_as_float(word);
        }
        __syncthreads();
    }
}

__global__ void k_order_clear(float4* __restrict__ nodes, uint32_t n_nodes) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n_nodes) nodes[4ull * i + 3].z = 0.0f;
}

// Learned first child of every 8-wide node, per (octant, mode): from the
// binary node of the wide node's root cluster, follow the binary decisions
// (the child order word's decided child) while they are confident, until the
// path reaches one of the wide node's children; that slot is entry
// octant + 8 * any_hit of the table (8 | slot; 0 where a decision is missing).
// The children of a wide node are the frontier of the binary subtree below its
// root, so every decided path reaches one within 7 steps.
__global__ __launch_bounds__(256) void k_wide_order(const float4* __restrict__ nodes, float4* __restrict__ wide,
                                                    const uint32_t* __restrict__ wide_trav, uint32_t n_wide,
                                                    uint32_t n_trav) {
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n_wide) return;
    const float4* wn = wide + 8ull * k;
    const uint32_t valid = __float_as_uint(wn[0].w) >> 24;
    const float4 a = wn[4], b = wn[5];
    const uint32_t refs[8] = {__float_as_uint(a.x), __float_as_uint(a.y), __float_as_uint(a.z), __float_as_uint(a.w),
                              __float_as_uint(b.x), __float_as_uint(b.y), __float_as_uint(b.z), __float_as_uint(b.w)};
    // each child as the binary layout refers to it: a leaf ref is the same in
    // both layouts, an internal child is the binary node of its root cluster
    uint32_t as_binary[8];
    for (int j = 0; j < 8; ++j) {
        const uint32_t r = refs[j];
        as_binary[j] = !((valid >> j) & 1u) ? kNone : ((r & kLeafBit) ? r : wide_trav[r]);
    }
    uint32_t table[2] = {0u, 0u};
    const uint32_t root = wide_trav[k];
    for (uint32_t e = 0; e < 16 && root < n_trav; ++e) {
        uint32_t x = root, entry = 0;
        for (int step = 0; step < 8; ++step) {
            const float4 n3 = nodes[4ull * x + 3];
            const uint32_t ow = __float_as_uint(n3.z);
            if (!((ow >> (16 + e)) & 1u)) break;   // no confident decision
            const uint32_t child = ((ow >> e) & 1u) ? __float_as_uint(n3.x) : __float_as_uint(n3.y);
            int slot = -1;
            for (int j = 0; j < 8; ++j)
                if (as_binary[j] == child) slot = j;
            if (slot >= 0) {
                entry = 8u | (uint32_t)slot;
                break;
            }
            if ((child & kLeafBit) || child >= n_trav) break;   // not inside this node's subtree
            x = child;
        }
        table[e >> 3] |= entry << (4 * (e & 7));
    }
    wide[8ull * k + 6] = make_float4(__uint_as_float(table[0]), __uint_as_float(table[1]), 0.0f, 0.0f);
}

__global__ void k_wide_order_clear(float4* __restrict__ wide, uint32_t n_wide) {
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if (k < n_wide) wide[8ull * k + 6] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

}  // namespace

rtq_status write_wide_order(rtq_ctx* ctx, Scene* s, bool clear, hipStream_t st) {
    s->wide_ordered = false;
    if (!s->wide || s->n_wide == 0) return RTQ_OK;
    const uint32_t blocks = (s->n_wide + 255) / 256;
    if (clear) {
        hipLaunchKernelGGL(k_wide_order_clear, dim3(blocks), dim3(256), 0, st, s->wide, s->n_wide);
    } else {
        hipLaunchKernelGGL(k_wide_order, dim3(blocks), dim3(256), 0, st, s->nodes, s->wide, s->wide_trav, s->n_wide,
                           s->n_trav);
    }
    RTQ_HIP(ctx, hipGetLastError());
    s->wide_ordered = !clear;
    return RTQ_OK;
}

}  // namespace rtq

using namespace rtq;

extern "C" {

rtq_status rtq_order_log(rtq_ctx* ctx, uint32_t scene_id, const rtq_ray* rays_dev, uint64_t n_rays, uint32_t flags,
                         uint32_t stride, float* samples_dev, uint64_t capacity, uint64_t* n_samples) {
    if (!ctx) return RTQ_EINVAL;
    Scene* s = find_scene(ctx, scene_id);
    if (!s) return fail(ctx, RTQ_EINVAL, "order_log: unknown scene %u", scene_id);
    if (!s->built) return fail(ctx, RTQ_ENOTBUILT, "order_log: scene %u has no BVH", scene_id);
    if (!rays_dev || !samples_dev || !n_samples || stride == 0) return fail(ctx, RTQ_EINVAL, "order_log: bad argument");
    if (n_rays > 0xFFFFFFFFull || capacity > 0xFFFFFFFFull) return fail(ctx, RTQ_ECAPACITY, "order_log: too many rays");
    if (flags & ~RTQ_TRACE_ANY) return fail(ctx, RTQ_EINVAL, "order_log: only RTQ_TRACE_ANY may be set");
    RTQ_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    uint32_t* cnt = nullptr;
    RTQ_HIP(ctx, dev_alloc(&cnt, 1));
    hipError_t e = hipMemsetAsync(cnt, 0, sizeof(uint32_t), st);
    const uint64_t threads = (n_rays + stride - 1) / stride;
    if (e == hipSuccess && threads > 0) {
        // three levels at a time (16 lanes per ray) while the waves fit the
        // chip at four per SIMD, else two (8 lanes): the times are at k_order_log
        const int ahead = threads <= 4 * 4 * 4 * (uint64_t)std::max(ctx->n_cu, 1) ? 3 : 2;
        const uint32_t per_wave = 64 / log_lanes(ahead);
        const uint32_t levels = std::min<uint32_t>(kLogStack, s->depth + 1);
        // (a launch has fewer than 2^32 threads, a ray 8 or 16 of them)
        for (uint64_t first = 0; first < threads && e == hipSuccess; first += kLogLaunch) {
            const uint64_t here = std::min<uint64_t>(threads - first, kLogLaunch), at = first * stride;
            hipLaunchKernelGGL(ahead == 3 ? &k_order_log<3> : &k_order_log<2>,
                               dim3((uint32_t)((here + per_wave - 1) / per_wave)), dim3(64),
                               sizeof(uint32_t) * levels * 64, st, s->nodes, s->node_aux, s->tris, rays_dev + at,
                               (uint32_t)std::min<uint64_t>(n_rays - at, here * stride), stride,
                               (flags & RTQ_TRACE_ANY) ? 1u : 0u, samples_dev, (uint32_t)capacity, cnt);
            e = hipGetLastError();
        }
    }
    uint32_t h = 0;
    if (e == hipSuccess) e = hipMemcpyAsync(&h, cnt, sizeof h, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    (void)hipFree(cnt);
    if (e != hipSuccess) return hip_fail(ctx, e, "order_log");
    *n_samples = std::min<uint64_t>(h, capacity);
    return RTQ_OK;
}

// One batch gradient: grad = mean over samples [0, n) of dLoss/dParams.
rtq_status rtq_order_grad(rtq_ctx* ctx, const float* params_dev, const float* samples_dev, uint32_t n,
                          float* grad_dev, float* loss) {
    if (!ctx) return RTQ_EINVAL;
    if (!params_dev || !samples_dev || !grad_dev || n == 0) return fail(ctx, RTQ_EINVAL, "order_grad: bad argument");
    RTQ_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    const uint32_t blocks = (n + kTB - 1) / kTB;
    float *partial = nullptr, *lp = nullptr;
    RTQ_HIP(ctx, dev_alloc(&partial, (size_t)blocks * kNP));
    hipError_t e = dev_alloc(&lp, blocks);
    if (e == hipSuccess) {
        e = queue_grad(ctx, params_dev, samples_dev, SampleOrder{n, 0u, 1u, 1.0 / n}, n, partial, lp, st);
    }
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_mlp_reduce, dim3(kParamBlocks), dim3(kParamThreads), 0, st, partial, blocks,
                           1.0f / (float)n, grad_dev);
        e = hipGetLastError();
    }
    std::vector<float> hl(blocks);
    if (e == hipSuccess) e = hipMemcpyAsync(hl.data(), lp, sizeof(float) * blocks, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    (void)hipFree(partial);
    (void)hipFree(lp);
    if (e != hipSuccess) return hip_fail(ctx, e, "order_grad");
    if (loss) {
        double a = 0.0;
        for (float v : hl) a += v;
        *loss = (float)(a / n);
    }
    return RTQ_OK;
}

rtq_status rtq_order_train(rtq_ctx* ctx, const float* samples_dev, uint64_t n_samples, const rtq_train_params* tp,
                           float* params_dev, float* adam_m_dev, float* adam_v_dev, uint32_t* step,
                           float* epoch_loss) {
    if (!ctx) return RTQ_EINVAL;
    if (!samples_dev || !tp || !params_dev || !adam_m_dev || !adam_v_dev || !step || n_samples == 0)
        return fail(ctx, RTQ_EINVAL, "order_train: bad argument");
    if (n_samples > 0x7FFFFFFFull) return fail(ctx, RTQ_ECAPACITY, "order_train: too many samples");
    if (tp->batch == 0 || tp->batch % kTB || tp->batch > 65536)
        return fail(ctx, RTQ_EINVAL, "order_train: batch must be a multiple of 64, at most 65536");
    RTQ_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    const uint32_t n = (uint32_t)n_samples;
    const uint32_t blocks = tp->batch / kTB;
    float *partial = nullptr, *lp = nullptr;
    RTQ_HIP(ctx, dev_alloc(&partial, (size_t)blocks * kNP));
    hipError_t e = dev_alloc(&lp, (size_t)blocks * ((n + tp->batch - 1) / tp->batch));
    const uint32_t steps_per_epoch = (n + tp->batch - 1) / tp->batch;
    for (uint32_t ep = 0; ep < tp->epochs && e == hipSuccess; ++ep) {
        // a permutation of the samples per epoch: i -> i * mul mod n with mul coprime to n
        uint64_t mul = 1;
        if (n > 1) {
            uint64_t h = (tp->seed + 0x9E3779B97F4A7C15ull * (ep + 1)) ^ 0xD1B54A32D192ED03ull;
            mul = (h % (n - 1)) + 1;
            auto gcd = [](uint64_t a, uint64_t b) { while (b) { uint64_t t = a % b; a = b; b = t; } return a; };
            while (gcd(mul, n) != 1) mul = mul % (n - 1) + 1;
        }
        for (uint32_t sidx = 0; sidx < steps_per_epoch && e == hipSuccess; ++sidx) {
            const uint64_t start = (uint64_t)sidx * tp->batch;
            const uint32_t cnt = (uint32_t)std::min<uint64_t>(tp->batch, n - start);
            const uint32_t bl = (cnt + kTB - 1) / kTB;
            const SampleOrder order{n, (uint32_t)(start * mul % n), (uint32_t)mul, 1.0 / n};
            e = queue_grad(ctx, params_dev, samples_dev, order, cnt, partial, lp + (size_t)sidx * blocks, st);
            if (e != hipSuccess) break;
            const uint32_t tstep = ++*step;
            const float c1 = 1.0f - powf(tp->beta1, (float)tstep), c2 = 1.0f - powf(tp->beta2, (float)tstep);
            hipLaunchKernelGGL(k_mlp_step, dim3(kParamBlocks), dim3(kParamThreads), 0, st, partial, bl,
                               1.0f / (float)cnt, params_dev, adam_m_dev, adam_v_dev, tp->lr, tp->beta1, tp->beta2,
                               1e-8f, c1, c2);
            e = hipGetLastError();
        }
        if (e != hipSuccess) break;
        // loss of the epoch (sum of the per-block sums of all steps)
        std::vector<float> hl((size_t)steps_per_epoch * blocks, 0.0f);
        e = hipMemcpyAsync(hl.data(), lp, sizeof(float) * hl.size(), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e == hipSuccess && epoch_loss) {
            double a = 0.0;
            for (uint32_t si = 0; si < steps_per_epoch; ++si) {
                const uint64_t start = (uint64_t)si * tp->batch;
                const uint32_t cnt = (uint32_t)std::min<uint64_t>(tp->batch, n - start);
                const uint32_t bl = (cnt + kTB - 1) / kTB;
                for (uint32_t b = 0; b < bl; ++b) a += hl[(size_t)si * blocks + b];
            }
            epoch_loss[ep] = (float)(a / n);
        }
    }
    (void)hipFree(partial);
    (void)hipFree(lp);
    if (e != hipSuccess) return hip_fail(ctx, e, "order_train");
    return RTQ_OK;
}

rtq_status rtq_order_predict(rtq_ctx* ctx, const float* params_dev, const float* samples_dev, uint64_t n,
                             uint32_t stride, float* prob_dev) {
    if (!ctx) return RTQ_EINVAL;
    if (!params_dev || !samples_dev || !prob_dev || stride < kIn) return fail(ctx, RTQ_EINVAL, "order_predict: bad argument");
    if (n == 0) return RTQ_OK;
    if (n > 0xFFFFFFFFull) return fail(ctx, RTQ_ECAPACITY, "order_predict: too many samples");
    RTQ_HIP(ctx, hipSetDevice(ctx->device));
    const uint32_t tiles = (uint32_t)((n + 31) / 32);
    const uint32_t blocks = std::min<uint32_t>((tiles + kIW - 1) / kIW, 2048u);
    hipLaunchKernelGGL(k_mlp_infer, dim3(blocks), dim3(64 * kIW), 0, ctx->stream, params_dev, samples_dev, (uint32_t)n,
                       stride, prob_dev);
    RTQ_HIP(ctx, hipGetLastError());
    RTQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return RTQ_OK;
}

rtq_status rtq_order_apply(rtq_ctx* ctx, uint32_t scene_id, const float* params_dev, float confidence_closest,
                           float confidence_any) {
    if (!ctx) return RTQ_EINVAL;
    Scene* s = find_scene(ctx, scene_id);
    if (!s) return fail(ctx, RTQ_EINVAL, "order_apply: unknown scene %u", scene_id);
    if (!s->built) return fail(ctx, RTQ_ENOTBUILT, "order_apply: scene %u has no BVH", scene_id);
    if (params_dev && !(confidence_closest >= 0.5f && confidence_any >= 0.5f))
        return fail(ctx, RTQ_EINVAL, "order_apply: confidences must be >= 0.5 (>= 1 disables a mode)");
    RTQ_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    if (!params_dev) {
        hipLaunchKernelGGL(k_order_clear, dim3((s->n_trav + 255) / 256), dim3(256), 0, st, s->nodes, s->n_trav);
    } else {
        // max(p, 1 - p) >= c  <=>  |logit| >= log(c / (1 - c)); c >= 1: never
        auto zmin = [](float c) {
            return c >= 1.0f ? INFINITY : (float)std::log((double)c / (1.0 - (double)c));
        };
        const uint32_t tiles = (s->n_trav + 1) / 2;
        const uint32_t blocks = std::min<uint32_t>((tiles + kIW - 1) / kIW, 2048u);
        hipLaunchKernelGGL(k_order_apply, dim3(blocks), dim3(64 * kIW), 0, st, params_dev, s->nodes, s->node_aux,
                           s->n_trav, zmin(confidence_closest), zmin(confidence_any));
    }
    RTQ_HIP(ctx, hipGetLastError());
    // the LDS copy of the top of the tree carries the order words too
    rtq_status rs = write_top(ctx, s, nullptr, 0, nullptr, st);
    if (rs != RTQ_OK) return rs;
    // the 8-wide nodes' first-child tables follow the binary decisions
    rs = write_wide_order(ctx, s, params_dev == nullptr, st);
    if (rs != RTQ_OK) return rs;
    RTQ_HIP(ctx, hipStreamSynchronize(st));
    s->ordered = params_dev != nullptr;
    s->order_closest = s->ordered && confidence_closest < 1.0f;
    s->order_any = s->ordered && confidence_any < 1.0f;
    return RTQ_OK;
}

rtq_status rtq_order_init(rtq_ctx* ctx, uint64_t seed, float* params_dev) {
    if (!ctx) return RTQ_EINVAL;
    if (!params_dev) return fail(ctx, RTQ_EINVAL, "order_init: null parameters");
    // He-uniform weights (limit sqrt(6 / fan_in)) from a SplitMix64 stream, zero biases
    std::vector<float> p(kNP, 0.0f);
    uint64_t st = seed;
    auto next = [&]() {
        uint64_t z = (st += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return (double)(z >> 40) * (1.0 / 16777216.0) * 2.0 - 1.0;
    };
    for (int i = 0; i < kIn * kH; ++i) p[kW1 + i] = (float)(next() * std::sqrt(6.0 / kIn));
    for (int i = 0; i < kH * kH; ++i) p[kW2 + i] = (float)(next() * std::sqrt(6.0 / kH));
    for (int i = 0; i < kH; ++i) p[kW3 + i] = (float)(next() * std::sqrt(6.0 / kH));
    RTQ_HIP(ctx, hipSetDevice(ctx->device));
    RTQ_HIP(ctx, hipMemcpy(params_dev, p.data(), sizeof(float) * kNP, hipMemcpyHostToDevice));
    return RTQ_OK;
}

namespace {
constexpr uint32_t kCkptMagic = 0x4d4f5452u;  // "RTOM"
constexpr uint32_t kCkptVersion = 1;

uint64_t fnv1a(const void* data, size_t n, uint64_t h = 0xcbf29ce484222325ull) {
    const unsigned char* p = static_cast<const unsigned char*>(data);
    for (size_t i = 0; i < n; ++i) h = (h ^ p[i]) * 0x100000001b3ull;
    return h;
}
}  // namespace

// File: magic, version, parameter count, step (4 x u32), then params, m, v
// (3 x RTQ_ORDER_PARAMS f32), then FNV-1a 64 of everything before it.
rtq_status rtq_order_save(rtq_ctx* ctx, const char* path, const float* params_dev, const float* adam_m_dev,
                          const float* adam_v_dev, uint32_t step) {
    if (!ctx) return RTQ_EINVAL;
    if (!path || !params_dev || !adam_m_dev || !adam_v_dev) return fail(ctx, RTQ_EINVAL, "order_save: bad argument");
    std::vector<unsigned char> buf(16 + 3 * sizeof(float) * kNP);
    const uint32_t head[4] = {kCkptMagic, kCkptVersion, (uint32_t)kNP, step};
    std::memcpy(buf.data(), head, 16);
    RTQ_HIP(ctx, hipSetDevice(ctx->device));
    const float* src[3] = {params_dev, adam_m_dev, adam_v_dev};
    for (int k = 0; k < 3; ++k)
        RTQ_HIP(ctx, hipMemcpy(buf.data() + 16 + k * sizeof(float) * kNP, src[k], sizeof(float) * kNP,
                               hipMemcpyDeviceToHost));
    const uint64_t h = fnv1a(buf.data(), buf.size());
    FILE* f = std::fopen(path, "wb");
    if (!f) return fail(ctx, RTQ_EINVAL, "order_save: cannot open %s", path);
    const bool ok = std::fwrite(buf.data(), 1, buf.size(), f) == buf.size() && std::fwrite(&h, 8, 1, f) == 1;
    const bool closed = std::fclose(f) == 0;
    if (!ok || !closed) return fail(ctx, RTQ_EINVAL, "order_save: write to %s failed", path);
    return RTQ_OK;
}

rtq_status rtq_order_load(rtq_ctx* ctx, const char* path, float* params_dev, float* adam_m_dev, float* adam_v_dev,
                          uint32_t* step) {
    if (!ctx) return RTQ_EINVAL;
    if (!path || !params_dev) return fail(ctx, RTQ_EINVAL, "order_load: bad argument");
    FILE* f = std::fopen(path, "rb");
    if (!f) return fail(ctx, RTQ_EINVAL, "order_load: cannot open %s", path);
    std::vector<unsigned char> buf(16 + 3 * sizeof(float) * kNP);
    uint64_t h = 0;
    const bool ok = std::fread(buf.data(), 1, buf.size(), f) == buf.size() && std::fread(&h, 8, 1, f) == 1;
    const bool extra = ok && std::fgetc(f) != EOF;
    std::fclose(f);
    if (!ok || extra) return fail(ctx, RTQ_EINVAL, "order_load: %s has the wrong size", path);
    uint32_t head[4];
    std::memcpy(head, buf.data(), 16);
    if (head[0] != kCkptMagic) return fail(ctx, RTQ_EINVAL, "order_load: %s is not an order-model file", path);
    if (head[1] != kCkptVersion) return fail(ctx, RTQ_EINVAL, "order_load: %s: unsupported version %u", path, head[1]);
    if (head[2] != (uint32_t)kNP) return fail(ctx, RTQ_EINVAL, "order_load: %s: %u parameters", path, head[2]);
    if (fnv1a(buf.data(), buf.size()) != h) return fail(ctx, RTQ_EINVAL, "order_load: %s: checksum mismatch", path);
    RTQ_HIP(ctx, hipSetDevice(ctx->device));
    float* dst[3] = {params_dev, adam_m_dev, adam_v_dev};
    for (int k = 0; k < 3; ++k)
        if (dst[k])
            RTQ_HIP(ctx, hipMemcpy(dst[k], buf.data() + 16 + k * sizeof(float) * kNP, sizeof(float) * kNP,
                                   hipMemcpyHostToDevice));
    if (step) *step = head[3];
    return RTQ_OK;
}

}  // extern "C"

// ---- the order model as one object owning its device memory ----------------

struct rtq_order_model {
    rtq_ctx* ctx = nullptr;
    float* params = nullptr;   // kNP
    float* m = nullptr;        // kNP (Adam first moment)
    float* v = nullptr;        // kNP (Adam second moment)
    float* samples = nullptr;  // capacity x kSample
    uint64_t capacity = 0;
    uint64_t n_samples = 0;
    uint32_t step = 0;
};

namespace {
void free_model(rtq_order_model* m) {
    if (m->params) (void)hipFree(m->params);
    if (m->m) (void)hipFree(m->m);
    if (m->v) (void)hipFree(m->v);
    if (m->samples) (void)hipFree(m->samples);
    delete m;
}
}  // namespace

extern "C" {

rtq_status rtq_order_model_create(rtq_ctx* ctx, uint64_t seed, uint64_t sample_capacity, rtq_order_model** out) {
    if (!ctx) return RTQ_EINVAL;
    if (!out) return fail(ctx, RTQ_EINVAL, "order_model_create: null output");
    *out = nullptr;
    if (sample_capacity > 0xFFFFFFFFull)
        return fail(ctx, RTQ_ECAPACITY, "order_model_create: at most 2^32 - 1 samples");
    RTQ_HIP(ctx, hipSetDevice(ctx->device));
    rtq_order_model* m = new rtq_order_model;
    m->ctx = ctx;
    m->capacity = sample_capacity;
    hipError_t e = dev_alloc(&m->params, kNP);
    if (e == hipSuccess) e = dev_alloc(&m->m, kNP);
    if (e == hipSuccess) e = dev_alloc(&m->v, kNP);
    if (e == hipSuccess) e = dev_alloc(&m->samples, (size_t)sample_capacity * kSample);
    if (e == hipSuccess) e = hipMemset(m->m, 0, sizeof(float) * kNP);
    if (e == hipSuccess) e = hipMemset(m->v, 0, sizeof(float) * kNP);
    if (e != hipSuccess) {
        free_model(m);
        return hip_fail(ctx, e, "order_model_create");
    }
    const rtq_status s = rtq_order_init(ctx, seed, m->params);
    if (s != RTQ_OK) {
        free_model(m);
        return s;
    }
    *out = m;
    return RTQ_OK;
}

void rtq_order_model_destroy(rtq_order_model* model) {
    if (!model) return;
    (void)hipSetDevice(model->ctx->device);
    free_model(model);
}

rtq_status rtq_order_model_log(rtq_order_model* model, uint32_t scene_id, const rtq_ray* rays_dev, uint64_t n_rays,
                               uint32_t flags, uint32_t stride, uint64_t* n_added) {
    if (!model) return RTQ_EINVAL;
    uint64_t k = 0;
    const uint64_t room = model->capacity - model->n_samples;
    if (room > 0) {
        const rtq_status s = rtq_order_log(model->ctx, scene_id, rays_dev, n_rays, flags, stride,
                                           model->samples + model->n_samples * kSample, room, &k);
        if (s != RTQ_OK) return s;
    }
    model->n_samples += k;
    if (n_added) *n_added = k;
    return RTQ_OK;
}

rtq_status rtq_order_model_clear_samples(rtq_order_model* model) {
    if (!model) return RTQ_EINVAL;
    model->n_samples = 0;
    return RTQ_OK;
}

rtq_status rtq_order_model_train(rtq_order_model* model, const rtq_train_params* tp, float* epoch_loss) {
    if (!model) return RTQ_EINVAL;
    if (model->n_samples == 0) return fail(model->ctx, RTQ_EINVAL, "order_model_train: no samples logged");
    return rtq_order_train(model->ctx, model->samples, model->n_samples, tp, model->params, model->m, model->v,
                           &model->step, epoch_loss);
}

rtq_status rtq_order_model_apply(rtq_order_model* model, uint32_t scene_id, float confidence_closest,
                                 float confidence_any) {
    if (!model) return RTQ_EINVAL;
    return rtq_order_apply(model->ctx, scene_id, model->params, confidence_closest, confidence_any);
}

rtq_status rtq_order_model_save(rtq_order_model* model, const char* path) {
    if (!model) return RTQ_EINVAL;
    return rtq_order_save(model->ctx, path, model->params, model->m, model->v, model->step);
}

rtq_status rtq_order_model_load(rtq_order_model* model, const char* path) {
    if (!model) return RTQ_EINVAL;
    return rtq_order_load(model->ctx, path, model->params, model->m, model->v, &model->step);
}

rtq_status rtq_order_model_info(const rtq_order_model* model, uint64_t* n_samples, uint32_t* step) {
    if (!model) return RTQ_EINVAL;
    if (n_samples) *n_samples = model->n_samples;
    if (step) *step = model->step;
    return RTQ_OK;
}

}  // extern "C"
