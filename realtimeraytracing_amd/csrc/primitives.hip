// Device primitives for the build: exclusive scan and stable LSD radix sort.
//
// Scan: reduce-then-scan over 2048-element tiles (256 threads x 8 items,
// blocked), tile sums scanned recursively, then a block scan per tile.
// Radix sort: 8-bit digits; one launch counts every digit position, then one
// Onesweep launch per digit (decoupled look-back over tiles for the digit
// offsets, a sort of the tile in LDS, then the scatter); up to 8,192 pairs are
// sorted by one workgroup in one launch.  Keys are ranked stably inside a tile
// with wave-wide digit match masks (8 ballots per key) and per-wave digit
// counts in LDS, so equal keys keep their input order: with iota values this
// is std::sort on (code, index) pairs (bvh.cpp:223-231).  The reference's own GPU sort never got past a
// set-bit histogram and a per-group scan (histogramOfGlobalDigitCounts.glsl,
// prefixSumOfGlobalDigitCounts.glsl, chainedScanDigitBinning.glsl:31-32 empty).
#include "rtq_internal.hpp"

namespace rtq {
namespace {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

__device__ inline uint32_t shfl_up_u32(uint32_t x, int o) { return __shfl_up(x, o, 64); }

struct U1 {
    uint32_t x;
    __device__ U1 operator+(const U1& b) const { return {x + b.x}; }
    __device__ U1 shfl_up(int o) const { return {shfl_up_u32(x, o)}; }
};
struct U2 {
    uint32_t x, y;
    __device__ U2 operator+(const U2& b) const { return {x + b.x, y + b.y}; }
    __device__ U2 shfl_up(int o) const { return {shfl_up_u32(x, o), shfl_up_u32(y, o)}; }
};

template <typename T>
__global__ __launch_bounds__(kScanThreads) void k_tile_reduce(const T* __restrict__ in, uint64_t n,
                                                              T* __restrict__ sums) {
    __shared__ T s_wave[kScanThreads / 64];
    const uint64_t base = (uint64_t)blockIdx.x * kScanTile;
    T acc{};
    for (int r = 0; r < kScanItems; ++r) {
        uint64_t i = base + (uint64_t)r * kScanThreads + threadIdx.x;
        if (i < n) acc = acc + in[i];
    }
    for (int o = 1; o < 64; o <<= 1) {
        T y = acc.shfl_up(o);
        if ((threadIdx.x & 63) >= (unsigned)o) acc = acc + y;
    }
    if ((threadIdx.x & 63) == 63) s_wave[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        T t{};
        for (int w = 0; w < kScanThreads / 64; ++w) t = t + s_wave[w];
        sums[blockIdx.x] = t;
    }
}

template <typename T>
__global__ __launch_bounds__(kScanThreads) void k_tile_scan(const T* __restrict__ in, T* __restrict__ out,
                                                            uint64_t n, const T* __restrict__ offsets,
                                                            T* __restrict__ total) {
    __shared__ T s_wave[kScanThreads / 64];
    const uint64_t base = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * kScanItems;
    T v[kScanItems];
    T tsum{};
#pragma unroll
    for (int r = 0; r < kScanItems; ++r) {
        uint64_t i = base + r;
        v[r] = (i < n) ? in[i] : T{};
        tsum = tsum + v[r];
    }
    T x = tsum;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int o = 1; o < 64; o <<= 1) {
        T y = x.shfl_up(o);
        if (lane >= o) x = x + y;
    }
    if (lane == 63) s_wave[wid] = x;
    __syncthreads();
    T off = offsets ? offsets[blockIdx.x] : T{};
    T block_total{};
    for (int w = 0; w < kScanThreads / 64; ++w) {
        if (w < wid) off = off + s_wave[w];
        block_total = block_total + s_wave[w];
    }
    // exclusive prefix of this thread = off + (x - tsum); computed additively
    T run = off;
    {
        // x - tsum == inclusive-of-previous-lanes; rebuild it with a shifted scan value
        T prev = x.shfl_up(1);
        if (lane > 0) run = run + prev;
    }
#pragma unroll
    for (int r = 0; r < kScanItems; ++r) {
        uint64_t i = base + r;
        if (i < n) out[i] = run;
        run = run + v[r];
    }
    if (total && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        T o = offsets ? offsets[blockIdx.x] : T{};
        *total = o + block_total;
    }
}

template <typename T>
rtq_status scan_impl(rtq_ctx* ctx, const T* in, T* out, uint64_t n, T* total, hipStream_t st) {
    if (n == 0) {
        if (total) RTQ_HIP(ctx, hipMemsetAsync(total, 0, sizeof(T), st));
        return RTQ_OK;
    }
    const uint64_t nb = (n + kScanTile - 1) / kScanTile;
    if (nb == 1) {
        hipLaunchKernelGGL(k_tile_scan<T>, dim3(1), dim3(kScanThreads), 0, st, in, out, n,
                           (const T*)nullptr, total);
        RTQ_HIP(ctx, hipGetLastError());
        return RTQ_OK;
    }
    Temps tmp(ctx);
    T* sums = nullptr;
    RTQ_HIP(ctx, tmp.get(&sums, 2 * nb));
    T* offs = sums + nb;
    hipLaunchKernelGGL(k_tile_reduce<T>, dim3((uint32_t)nb), dim3(kScanThreads), 0, st, in, n, sums);
    RTQ_HIP(ctx, hipGetLastError());
    const rtq_status s = scan_impl<T>(ctx, sums, offs, nb, nullptr, st);
    if (s != RTQ_OK) return s;
    hipLaunchKernelGGL(k_tile_scan<T>, dim3((uint32_t)nb), dim3(kScanThreads), 0, st, in, out, n,
                       (const T*)offs, total);
    RTQ_HIP(ctx, hipGetLastError());
    return RTQ_OK;
}

// Elements of workspace scan_impl_ws needs for n elements (the tile sums and
// their offsets at every level).
template <typename T>
uint64_t scan_workspace(uint64_t n) {
    uint64_t total = 0;
    while (n > (uint64_t)kScanTile) {
        const uint64_t nb = (n + kScanTile - 1) / kScanTile;
        total += 2 * nb;
        n = nb;
    }
    return total;
}

// The same scan with the caller's workspace: no allocation and no
// synchronisation, so it can be queued back to back.
template <typename T>
rtq_status scan_impl_ws(rtq_ctx* ctx, const T* in, T* out, uint64_t n, T* total, T* ws, hipStream_t st) {
    if (n == 0) return fail(ctx, RTQ_EINTERNAL, "scan_ws: n must be > 0");
    const uint64_t nb = (n + kScanTile - 1) / kScanTile;
    if (nb == 1) {
        hipLaunchKernelGGL(k_tile_scan<T>, dim3(1), dim3(kScanThreads), 0, st, in, out, n,
                           (const T*)nullptr, total);
        RTQ_HIP(ctx, hipGetLastError());
        return RTQ_OK;
    }
    T* sums = ws;
    T* offs = ws + nb;
    hipLaunchKernelGGL(k_tile_reduce<T>, dim3((uint32_t)nb), dim3(kScanThreads), 0, st, in, n, sums);
    RTQ_HIP(ctx, hipGetLastError());
    rtq_status s = scan_impl_ws<T>(ctx, sums, offs, nb, nullptr, ws + 2 * nb, st);
    if (s != RTQ_OK) return s;
    hipLaunchKernelGGL(k_tile_scan<T>, dim3((uint32_t)nb), dim3(kScanThreads), 0, st, in, out, n,
                       (const T*)offs, total);
    RTQ_HIP(ctx, hipGetLastError());
    return RTQ_OK;
}

// ---------------------------------------------------------------- radix sort

constexpr int kSortThreads = 512;
constexpr int kSortWaves = kSortThreads / 64;
constexpr int kSmallThreads = 1024;
constexpr int kHistItems = 16;
constexpr uint32_t kHistBlocks = 256;
constexpr uint32_t kHistCopies = 8;
// Look-back status word of (tile, digit): flags in the top two bits, a count
// (below 2^30) in the others.  Aggregate = the tile's own count of the digit,
// prefix = its count plus every earlier tile's.
constexpr uint32_t kDigitAgg = 1u << 30;
constexpr uint32_t kDigitPre = 2u << 30;
constexpr uint32_t kDigitFlags = 3u << 30;

// Counts of every digit at every digit position in one read of the keys:
// hist[p * 256 + d] = keys whose digit p (bits 8p .. 8p+7) is d, p < n_digits.
// Each workgroup counts its tiles in LDS (a tile's loads together, then its
// counts) and adds its non-zero bins: 256 workgroups, since the additions to
// one bin serialise.  Neighbouring triangles' codes share their high digits,
// and the lanes that add to one bin serialise too: each bin has a word per
// eighth of a wave (2,093,058 Morton codes: 22.0 us with one word, 10.6 now;
// 5,000,000 random keys 15.1 and 15.6).
__global__ __launch_bounds__(kSortThreads) void k_sort_hist(const uint32_t* __restrict__ keys, uint32_t n,
                                                            uint32_t n_digits, uint32_t* __restrict__ hist) {
    constexpr uint32_t kTile = kSortThreads * kHistItems;
    __shared__ uint32_t s_h[4 * 256 * kHistCopies];
    const uint32_t copy = threadIdx.x % kHistCopies;
    for (uint32_t i = threadIdx.x; i < 4 * 256 * kHistCopies; i += kSortThreads) s_h[i] = 0;
    __syncthreads();
    for (uint32_t base = blockIdx.x * kTile; base < n; base += gridDim.x * kTile) {
        uint32_t k[kHistItems];
#pragma unroll
        for (int r = 0; r < kHistItems; ++r) {
            const uint32_t i = base + r * kSortThreads + threadIdx.x;
            k[r] = i < n ? keys[i] : 0u;
        }
#pragma unroll
        for (int r = 0; r < kHistItems; ++r)
            if (base + r * kSortThreads + threadIdx.x < n)
                for (uint32_t p = 0; p < n_digits; ++p) {
                    const uint32_t d = (k[r] >> (8 * p)) & 0xFFu;
                    atomicAdd(&s_h[(p * 256 + d) * kHistCopies + copy], 1u);
                }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < 256 * n_digits; i += kSortThreads) {
        uint32_t c = 0;
#pragma unroll
        for (uint32_t j = 0; j < kHistCopies; ++j) c += s_h[i * kHistCopies + j];
        if (c) atomicAdd(&hist[i], c);
    }
}

// Exclusive sum over the 256 digits of thread d's count c (threads past the
// digits pass 0).  Every thread of the workgroup calls it; s_w: 4 words.
__device__ __forceinline__ uint32_t digit_exclusive_sum(uint32_t c, uint32_t* s_w) {
    const uint32_t incl = wave_inclusive_sum(c);
    if (threadIdx.x < 256 && (threadIdx.x & 63u) == 63u) s_w[threadIdx.x >> 6] = incl;
    __syncthreads();
    uint32_t before = 0;
#pragma unroll
    for (uint32_t w = 0; w < 4; ++w) before += w < (threadIdx.x >> 6) ? s_w[w] : 0u;
    __syncthreads();
    return before + incl - c;
}

// Stable ranks of a tile's keys by one digit.  Wave w holds the tile's
// positions [w, w + 1) * 64 ITEMS, item r of lane l the r-th 64 of them's l-th;
// n_wave of them are keys.  rank[r] = keys before this one in its wave with the
// same digit; counts = the wave's row of 256 digit counts (zero before, the
// wave's totals after).  The lanes with equal digits find each other by 8
// ballots, the first one adds their number to the wave's count.
template <int ITEMS>
__device__ __forceinline__ void rank_digits(const uint32_t* key, uint32_t shift, uint32_t n_wave,
                                            uint32_t* counts, uint32_t* rank) {
    const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t d = (key[r] >> shift) & 0xFFu;
        const bool valid = r * 64u + lane < n_wave;
        uint64_t m = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bb = __ballot(bit);
            m &= bit ? bb : ~bb;
        }
        const uint32_t before = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        const uint32_t seen = counts[d];
        rank[r] = seen + before;
        // the wave's instructions keep their order: every lane has read its
        // count before the first of its group replaces it
        asm volatile("" ::: "memory");
        if (valid && before == 0) counts[d] = seen + (uint32_t)__popcll(m);
        asm volatile("" ::: "memory");
    }
}

// Thread d < 256: the waves' counts of digit d become the counts of the waves
// before; returns their total (0 for the other threads).
template <int WAVES>
__device__ __forceinline__ uint32_t digit_totals(uint32_t (*counts)[256]) {
    uint32_t total = 0;
    if (threadIdx.x < 256) {
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const uint32_t c = counts[w][threadIdx.x];
            counts[w][threadIdx.x] = total;
            total += c;
        }
    }
    return total;
}

// One digit pass in one launch (Adinets & Merrill, "Onesweep: A Faster Least
// Significant Digit Radix Sort for GPUs", 2022): a workgroup takes the next
// tile (take_tile), ranks its
// keys by digit, publishes its counts and sums those of the earlier tiles by
// decoupled look-back per digit (Merrill & Garland 2016), 8 tiles at a time (a
// tile waits for a chain of loads as long as the tiles that run beside it).  It
// sorts its pairs in LDS, so that each digit's keys leave as one run: written
// from where they were read they took a 64-B sector each.  A thread that has
// waited for its digit's count of a tile for long (kTilePatience) counts that
// tile's keys itself.  5M pairs:
// 90.6 us a pass with 4,096-pair tiles written in place, 38.0 now (15 us of
// memory traffic at the card's copy rate).
template <int ITEMS>
__global__ __launch_bounds__(kSortThreads) void k_onesweep(
    const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals, uint32_t n, uint32_t shift,
    const uint32_t* __restrict__ hist, uint32_t* __restrict__ tile_ctr, uint32_t* __restrict__ status,
    uint32_t* __restrict__ out_k, uint32_t* __restrict__ out_v) {
    constexpr uint32_t kTile = kSortThreads * ITEMS;
    __shared__ uint2 s_kv[kTile];
    __shared__ uint32_t s_cnt[kSortWaves][256];
    __shared__ uint32_t s_start[256];   // digit's first position in the sorted tile
    __shared__ uint32_t s_off[256];     // digit's global position minus that
    __shared__ uint32_t s_w[4];
    __shared__ uint32_t s_tile;
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63u;
    if (tid == 0) s_tile = take_tile(tile_ctr);
    for (uint32_t i = tid; i < kSortWaves * 256; i += kSortThreads) (&s_cnt[0][0])[i] = 0;
    __syncthreads();
    const uint32_t tile = s_tile;
    const uint32_t base = tile * kTile;
    const uint32_t n_tile = min(kTile, n - base);
    const uint32_t first = wave * 64u * ITEMS;
    const uint32_t n_wave = n_tile > first ? n_tile - first : 0u;
    uint32_t key[ITEMS], val[ITEMS], rank[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t i = first + r * 64u + lane;
        key[r] = i < n_tile ? keys[base + i] : 0u;
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t i = first + r * 64u + lane;
        val[r] = i < n_tile ? vals[base + i] : 0u;
    }
    rank_digits<ITEMS>(key, shift, n_wave, s_cnt[wave], rank);
    __syncthreads();
    const uint32_t c = digit_totals<kSortWaves>(s_cnt);
    uint32_t* const mine = status + (size_t)tile * 256 + tid;
    if (tid < 256)
        __hip_atomic_store(mine, (tile == 0 ? kDigitPre : kDigitAgg) | c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t start = digit_exclusive_sum(c, s_w);
    const uint32_t digit_base = digit_exclusive_sum(tid < 256 ? hist[tid] : 0u, s_w);
    if (tid < 256) s_start[tid] = start;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
        if (first + r * 64u + lane < n_tile) {
            const uint32_t d = (key[r] >> shift) & 0xFFu;
            s_kv[s_start[d] + s_cnt[wave][d] + rank[r]] = make_uint2(key[r], val[r]);
        }
    if (tid < 256) {
        uint32_t excl = 0;
        if (tile > 0) {
            constexpr uint32_t kAhead = 8;
            uint32_t k = tile, polls = 0;   // tiles from k on are summed
            bool done = false;
            while (!done) {
                uint32_t w[kAhead];
#pragma unroll
                for (uint32_t q = 0; q < kAhead; ++q)
                    w[q] = k > q ? __hip_atomic_load(status + (size_t)(k - 1 - q) * 256 + tid, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT)
                                 : kDigitPre;   // before tile 0: an empty prefix
                uint32_t taken = 0;
                bool ready = true;
#pragma unroll
                for (uint32_t q = 0; q < kAhead; ++q) {
                    const uint32_t f = w[q] & kDigitFlags;
                    ready = ready && f != 0 && !done;
                    if (ready) {
                        excl += w[q] & ~kDigitFlags;
                        ++taken;
                        done = f == kDigitPre;
                    }
                }
                k -= taken;
                if (taken == 0) {
                    if (++polls > kTilePatience) {
                        // tile k - 1, a whole one: only the last may be short
                        const uint32_t* const missing = keys + (size_t)(k - 1) * kTile;
                        uint32_t count = 0;
                        for (uint32_t i = 0; i < kTile; ++i) count += ((missing[i] >> shift) & 0xFFu) == tid;
                        publish_for(status + (size_t)(k - 1) * 256 + tid, kDigitAgg | count);
                    } else {
                        __builtin_amdgcn_s_sleep(1);
                    }
                }
            }
            __hip_atomic_store(mine, kDigitPre | (excl + c), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        s_off[tid] = digit_base + excl - start;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t i = r * kSortThreads + tid;
        if (i < n_tile) {
            const uint2 kv = s_kv[i];
            const uint32_t pos = s_off[(kv.x >> shift) & 0xFFu] + i;
            out_k[pos] = kv.x;
            out_v[pos] = kv.y;
        }
    }
}

// Every pass of a sort of at most kSmallThreads * ITEMS pairs in one workgroup,
// in place: the pairs stay in registers and LDS, so a small sort is one launch
// instead of a clear, a count and a launch per digit (960 pairs: 57 us in nine
// launches, 10 us now).
template <int ITEMS>
__global__ __launch_bounds__(kSmallThreads) void k_sort_small(uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                                              uint32_t n, uint32_t passes) {
    constexpr int kWaves = kSmallThreads / 64;
    __shared__ uint2 s_kv[kSmallThreads * ITEMS];
    __shared__ uint32_t s_cnt[kWaves][256];
    __shared__ uint32_t s_start[256];
    __shared__ uint32_t s_w[4];
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63u;
    const uint32_t first = wave * 64u * ITEMS;
    const uint32_t n_wave = n > first ? n - first : 0u;
    uint32_t key[ITEMS], val[ITEMS], rank[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t i = first + r * 64u + lane;
        key[r] = i < n ? keys[i] : 0u;
        val[r] = i < n ? vals[i] : 0u;
    }
    for (uint32_t p = 0; p < passes; ++p) {
        const uint32_t shift = 8 * p;
        for (uint32_t i = tid; i < kWaves * 256; i += kSmallThreads) (&s_cnt[0][0])[i] = 0;
        __syncthreads();
        rank_digits<ITEMS>(key, shift, n_wave, s_cnt[wave], rank);
        __syncthreads();
        const uint32_t start = digit_exclusive_sum(digit_totals<kWaves>(s_cnt), s_w);
        if (tid < 256) s_start[tid] = start;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; ++r)
            if (first + r * 64u + lane < n) {
                const uint32_t d = (key[r] >> shift) & 0xFFu;
                s_kv[s_start[d] + s_cnt[wave][d] + rank[r]] = make_uint2(key[r], val[r]);
            }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            const uint32_t i = first + r * 64u + lane;
            if (i < n) {
                const uint2 kv = s_kv[i];
                key[r] = kv.x;
                val[r] = kv.y;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t i = first + r * 64u + lane;
        if (i < n) {
            keys[i] = key[r];
            vals[i] = val[r];
        }
    }
}

}  // namespace

rtq_status scan_u32(rtq_ctx* ctx, const uint32_t* in, uint32_t* out, uint64_t n, uint32_t* total,
                    hipStream_t st) {
    return scan_impl<U1>(ctx, reinterpret_cast<const U1*>(in), reinterpret_cast<U1*>(out), n,
                         reinterpret_cast<U1*>(total), st);
}

uint64_t scan_u32x2_workspace(uint64_t n) { return scan_workspace<U2>(n); }

rtq_status scan_u32x2_ws(rtq_ctx* ctx, const uint2* in, uint2* out, uint64_t n, uint2* total, uint2* ws,
                         hipStream_t st) {
    return scan_impl_ws<U2>(ctx, reinterpret_cast<const U2*>(in), reinterpret_cast<U2*>(out), n,
                            reinterpret_cast<U2*>(total), reinterpret_cast<U2*>(ws), st);
}

rtq_status radix_sort_pairs(rtq_ctx* ctx, uint32_t* keys, uint32_t* vals, uint32_t* tmp_k,
                            uint32_t* tmp_v, uint64_t n, uint32_t key_bits, hipStream_t st) {
    if (n == 0 || key_bits == 0) return RTQ_OK;
    if (n >= (1ull << 30)) return fail(ctx, RTQ_ECAPACITY, "sort: n must be < 2^30");
    const uint32_t nn = (uint32_t)n;
    const uint32_t passes = (key_bits + 7) / 8;
    if (nn <= kSmallThreads * 8) {
        if (nn <= kSmallThreads * 2)
            hipLaunchKernelGGL(k_sort_small<2>, dim3(1), dim3(kSmallThreads), 0, st, keys, vals, nn, passes);
        else
            hipLaunchKernelGGL(k_sort_small<8>, dim3(1), dim3(kSmallThreads), 0, st, keys, vals, nn, passes);
        RTQ_HIP(ctx, hipGetLastError());
        return RTQ_OK;
    }
    // tiles of 8,192 pairs, or of 2,048 while one for each CU takes them all
    const bool small_tiles = nn <= (uint32_t)std::max(ctx->n_cu, 1) * 2048u;
    const uint32_t tile = kSortThreads * (small_tiles ? 4 : 16);
    const uint32_t n_tiles = (nn + tile - 1) / tile;
    // digit counts and tile counters of every pass, then the passes' look-back
    // status words (one clear for all while they are few, else one set, cleared
    // before each pass): the passes queue without synchronising
    Temps tmp(ctx);
    constexpr size_t kHead = 4 * 256 + 4 * kTicketWords;
    const size_t rows = (size_t)n_tiles * 256;
    const bool one_clear = n_tiles <= 2048;
    uint32_t* hist = nullptr;
    RTQ_HIP(ctx, tmp.get(&hist, kHead + rows * (one_clear ? passes : 1)));
    uint32_t* const ctr = hist + 4 * 256;
    uint32_t* const status = hist + kHead;
    RTQ_HIP(ctx, hipMemsetAsync(hist, 0, sizeof(uint32_t) * (kHead + (one_clear ? rows * passes : 0)), st));
    const uint32_t hist_tiles = (nn + kSortThreads * kHistItems - 1) / (kSortThreads * kHistItems);
    hipLaunchKernelGGL(k_sort_hist, dim3(std::min(hist_tiles, kHistBlocks)), dim3(kSortThreads), 0, st, keys, nn,
                       passes, hist);
    RTQ_HIP(ctx, hipGetLastError());
    uint32_t *src_k = keys, *src_v = vals, *dst_k = tmp_k, *dst_v = tmp_v;
    for (uint32_t p = 0; p < passes; ++p) {
        if (!one_clear) RTQ_HIP(ctx, hipMemsetAsync(status, 0, sizeof(uint32_t) * rows, st));
        const auto sweep = small_tiles ? &k_onesweep<4> : &k_onesweep<16>;
        hipLaunchKernelGGL(sweep, dim3(n_tiles), dim3(kSortThreads), 0, st, src_k, src_v, nn, 8 * p, hist + 256 * p,
                           ctr + p * kTicketWords, status + (one_clear ? rows * p : 0), dst_k, dst_v);
        RTQ_HIP(ctx, hipGetLastError());
        std::swap(src_k, dst_k);
        std::swap(src_v, dst_v);
    }
    if (passes & 1) {
        RTQ_HIP(ctx, hipMemcpyAsync(keys, src_k, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, st));
        RTQ_HIP(ctx, hipMemcpyAsync(vals, src_v, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, st));
    }
    return RTQ_OK;
}

}  // namespace rtq
