// roadmap.hip -- the roadmap glue of mainPUMP.cu:257-392 on the device:
//   * rn = k-th smallest pair cost (thrust::sort + index, mainPUMP.cu:303-304)
//     over order-preserving uint32 keys: a sample brackets it, one pass over
//     the array counts the keys below the bracket and collects those inside,
//     and histograms of 2048 bins narrow these down to one;
//   * edge numbering (copts < rn, row-major i then j, mainPUMP.cu:327-346):
//     per-row counts, an exclusive scan, then an order-preserving per-row
//     compaction with wave ballots;
//   * maxNNSize and the padded neighbour tables (mainPUMP.cu:362-392);
//   * waypoint offsets for a fixed or per-edge waypoint count.
// All of this is HBM-streaming integer/compare work over the pair arrays.
#include <algorithm>

#include "pump_internal.hpp"

namespace pump {
namespace {

// ---- k-th smallest key ----------------------------------------------------
constexpr int kSelBins = 2048;
constexpr int kSelSample = 16384; // keys of the sample, 16 per thread of one workgroup
constexpr int kSelRun = 16;       // neighbouring keys per place of the sample: one 64-byte line
constexpr int kSelTile = 8192;    // keys per workgroup and round of the bracket pass
constexpr int kSelMaxRegions = 1024;
constexpr int64_t kSelScatterMax = 1 << 25;

// The keys still in question are those with key - lo <= span; k is the rank
// sought among them.  The next pass bins them by (key - lo) >> shift.
struct SelState {
    unsigned long long k;
    unsigned long long below;  // keys under lo (bracket pass)
    unsigned long long n_cand; // keys inside the bracket (bracket pass)
    uint32_t full;             // regions whose keys did not fit (bracket pass)
    uint32_t lo, span, shift;
    int counted; // k is a rank among the keys in question (not before the first pick)
    int done;    // result holds the answer
    int missed;  // the collected keys do not do: passes go over the array
    float result;

    // rank k lies inside the bracket
    __device__ bool inside() const { return k >= below && k - below < n_cand; }
    __device__ bool bracket_holds() const { return inside() && full == 0; }
};

__device__ __forceinline__ uint32_t order_key(float f)
{
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float key_float(uint32_t k)
{
    uint32_t u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
    return __uint_as_float(u);
}

// the bins of a span of keys: 2048 at most
__device__ __forceinline__ uint32_t sel_shift(uint32_t span)
{
    return (uint32_t)max(0, 32 - 11 - (int)__clz((int)(span | 1u)));
}

// every key is in question
__device__ __forceinline__ void sel_whole_range(SelState *st)
{
    st->lo = 0;
    st->span = 0xffffffffu;
    st->shift = sel_shift(st->span);
}

// The ranks in a sample of m keys that bracket rank k of n: five standard
// deviations to either side of k's place.  One past an end of the sample
// leaves the bracket open there, whatever lies beyond.
struct SelRanks {
    int lo, hi;
    bool open_lo, open_hi;
};

__host__ __device__ __forceinline__ SelRanks sel_ranks(int64_t k, int64_t n, int m)
{
    const float place = (float)k / (float)n * (float)m;
    const int margin = (int)(5.0f * sqrtf(fminf(place, (float)m - place) + 1.0f)) + 4;
    SelRanks r;
    r.lo = (int)place - margin;
    r.hi = (int)place + margin;
    r.open_lo = r.lo <= 0;
    r.open_hi = r.hi >= m - 1;
    r.lo = r.lo > 0 ? r.lo : 0;
    r.hi = r.hi < m - 1 ? r.hi : m - 1;
    return r;
}

// inclusive scan of v over the workgroup; sh: one entry per wave
template <typename T>
__device__ __forceinline__ T block_scan(T v, T *sh)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int off = 1; off < 64; off <<= 1) {
        const T y = __shfl_up(v, off, 64);
        if (lane >= off)
            v += y;
    }
    __syncthreads(); // sh may be in use
    if (lane == 63)
        sh[wid] = v;
    __syncthreads();
    for (int w = 0; w < wid; ++w)
        v += sh[w];
    return v;
}

__global__ __launch_bounds__(256) void k_sel_init(SelState *st, unsigned long long *hist,
                                                  unsigned long long k)
{
    for (int b = threadIdx.x; b < kSelBins; b += blockDim.x)
        hist[b] = 0;
    if (threadIdx.x == 0) {
        *st = SelState{};
        st->k = k;
        st->counted = 1;
        sel_whole_range(st);
    }
}

// One workgroup: keys that bracket rank k, from a sample (kSelRun neighbours at
// a scattered place in each of 1024 equal stretches), after two rounds of 2048
// bins each (sel_ranks; a bracket that misses rank k all the same is found out
// by its counts).  With n <= kSelSample the sample is the array and the key of
// rank k itself comes out (done).  Lines, not single keys: the scattered loads
// of 16384 keys took 20 us more on an array of 6.4e7; bins between the
// smallest and the largest key, not of the leading bits: costs span a few
// binary orders, whose handful of counters took another 10 us.
__global__ __launch_bounds__(1024) void k_sel_sample(const float *__restrict__ keys, int64_t n,
                                                     unsigned long long k, SelState *st,
                                                     unsigned long long *hist)
{
    constexpr int kPer = kSelSample / 1024;
    __shared__ uint32_t h[2][kSelBins];
    __shared__ uint32_t sh[16];
    __shared__ uint32_t least, most;
    __shared__ uint32_t bin[2], before[2];
    const int t = threadIdx.x;
    const bool whole = n <= kSelSample;
    const int m = whole ? (int)n : kSelSample;
    uint32_t key[kPer];
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        int64_t at = q * 1024 + t;
        if (!whole) {
            constexpr int kPlaces = kSelSample / kSelRun;
            const int j = (q * 1024 + t) / kSelRun;
            const int64_t step = n / kPlaces; // >= kSelRun
            at = j * step + (int64_t)(((uint32_t)j * 2654435769u) >> 7) % (step - kSelRun + 1) +
                 t % kSelRun;
        }
        key[q] = q * 1024 + t < m ? order_key(keys[at]) : 0u;
    }
    if (t == 0) {
        least = 0xffffffffu;
        most = 0u;
    }
    for (int b = t; b < kSelBins; b += 1024)
        hist[b] = 0;
    uint32_t lo_key = 0xffffffffu, hi_key = 0u;
#pragma unroll
    for (int q = 0; q < kPer; ++q)
        if (q * 1024 + t < m) {
            lo_key = min(lo_key, key[q]);
            hi_key = max(hi_key, key[q]);
        }
    for (int off = 32; off > 0; off >>= 1) {
        lo_key = min(lo_key, (uint32_t)__shfl_xor((int)lo_key, off, 64));
        hi_key = max(hi_key, (uint32_t)__shfl_xor((int)hi_key, off, 64));
    }
    __syncthreads();
    if ((t & 63) == 0) {
        atomicMin(&least, lo_key);
        atomicMax(&most, hi_key);
    }
    const SelRanks R = sel_ranks((int64_t)k, n, m);
    uint32_t rank[2], lo[2], span[2], shift[2];
    rank[0] = whole ? (uint32_t)k : (uint32_t)R.lo;
    rank[1] = whole ? (uint32_t)k : (uint32_t)R.hi;
    __syncthreads();
    for (int e = 0; e < 2; ++e) {
        lo[e] = least;
        span[e] = most - least;
        shift[e] = sel_shift(span[e]);
    }
    for (int pass = 0; whole ? span[0] != 0 || pass == 0 : pass < 2; ++pass) {
        for (int b = t; b < 2 * kSelBins; b += 1024)
            (&h[0][0])[b] = 0;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            if (q * 1024 + t >= m)
                continue;
            if (key[q] - lo[0] <= span[0])
                atomicAdd(&h[0][(key[q] - lo[0]) >> shift[0]], 1u);
            if (pass > 0 && key[q] - lo[1] <= span[1])
                atomicAdd(&h[1][(key[q] - lo[1]) >> shift[1]], 1u);
        }
        __syncthreads();
        for (int e = 0; e < 2; ++e) {
            const int from = pass > 0 ? e : 0; // the first pass is the same for both
            const uint32_t c0 = h[from][2 * t], c1 = h[from][2 * t + 1];
            const uint32_t c = block_scan(c0 + c1, sh) - c0 - c1;
            if (rank[e] >= c && rank[e] < c + c0 + c1) {
                const bool second = rank[e] >= c + c0;
                bin[e] = 2 * t + (second ? 1 : 0);
                before[e] = second ? c + c0 : c;
            }
        }
        __syncthreads();
        for (int e = 0; e < 2; ++e) {
            lo[e] += bin[e] << shift[e];
            rank[e] -= before[e];
            span[e] = (1u << shift[e]) - 1u;
            shift[e] = sel_shift(span[e]);
        }
        __syncthreads();
    }
    if (t == 0) {
        *st = SelState{};
        st->k = k;
        if (whole) {
            st->done = 1;
            st->result = key_float(lo[0]);
        } else {
            const uint32_t hi = R.open_hi ? 0xffffffffu : lo[1] + span[1];
            st->lo = R.open_lo ? 0u : lo[0];
            st->span = hi - st->lo;
            st->shift = sel_shift(st->span);
        }
    }
}

// One pass over all keys: counts those below the bracket and collects those
// inside it (a percent or so) in cand, each workgroup in a region of its own
// (region_cap keys; its count in counts).  With scatter a workgroup reads
// 1024 keys at a time, all over the array, and not 8192, so that a stretch
// with many keys of the bracket (an array in order, a sample near all others)
// goes to many regions: 1e6 keys in order 66 us for 90.  Long arrays go
// without (kSelScatterMax): 6.4e7 keys take 121 us for 118, and there the
// passes that follow a full region cost less than they did before the bracket
// (in order 214 us, 344 before; the middle rank 230, 276 before).  Bound by the read of the array:
// 6.4e7 keys in 60 us (4.3 TB/s); the selection 225 -> 107 us against three
// histogram passes over the array, 5 launches for 7.  (Turning the counts into
// the next state in the workgroup that ends last cost 100 us: every wave's
// device-scope release writes its L2 back.  A launch costs 5.)
__global__ __launch_bounds__(256) void k_sel_bracket(const float *__restrict__ keys, int64_t n,
                                                     SelState *st, float *__restrict__ cand,
                                                     uint32_t *__restrict__ counts,
                                                     uint32_t region_cap, bool scatter)
{
    __shared__ uint32_t held;
    __shared__ unsigned long long sh[4];
    constexpr int kVec = kSelTile / 4 / 256;
    const uint32_t lo = st->lo, span = st->span;
    const int lane = threadIdx.x & 63;
    const uint64_t lower = (1ull << lane) - 1ull;
    float *region = cand + (int64_t)blockIdx.x * region_cap;
    // 16-byte loads from the first aligned key on; up to 3 keys before and after
    const int64_t head = min((int64_t)((16 - ((uintptr_t)keys & 15)) & 15) / 4, n);
    const float4 *vec = reinterpret_cast<const float4 *>(keys + head);
    const int64_t n4 = (n - head) / 4;
    uint32_t below = 0;
    if (threadIdx.x == 0)
        held = 0;
    __syncthreads();
    const auto keep = [&](float f, uint32_t pos) {
        if (pos < region_cap)
            region[pos] = f;
    };
    if (blockIdx.x == 0 && threadIdx.x < 8) {
        const int64_t i = threadIdx.x < 4 ? (int64_t)threadIdx.x : head + 4 * n4 + threadIdx.x - 4;
        if (threadIdx.x < 4 ? i < head : i < n) {
            const uint32_t key = order_key(keys[i]);
            below += key < lo;
            if (key - lo <= span)
                keep(keys[i], atomicAdd(&held, 1u));
        }
    }
    // a thread's kVec vectors lie hop apart
    const int64_t hop = scatter ? (int64_t)gridDim.x * 256 : 256;
    for (int64_t q0 = (int64_t)blockIdx.x * (scatter ? 256 : 256 * kVec); q0 < n4;
         q0 += (int64_t)gridDim.x * (256 * kVec)) {
        float4 v[kVec];
#pragma unroll
        for (int j = 0; j < kVec; ++j) {
            const int64_t q = q0 + j * hop + threadIdx.x;
            v[j] = vec[q < n4 ? q : n4 - 1];
        }
#pragma unroll
        for (int j = 0; j < kVec; ++j) {
            const bool have = q0 + j * hop + threadIdx.x < n4;
            const float f[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
            uint64_t in[4], any = 0ull;
            uint32_t c = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t key = order_key(f[e]);
                below += have && key < lo;
                in[e] = __ballot(have && key - lo <= span);
                any |= in[e];
                c += __popcll(in[e]);
            }
            if (any == 0ull)
                continue;
            uint32_t pos = 0;
            if (lane == 0)
                pos = atomicAdd(&held, c);
            pos = __builtin_amdgcn_readfirstlane(pos);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if ((in[e] >> lane) & 1ull)
                    keep(f[e], pos + __popcll(in[e] & lower));
                pos += __popcll(in[e]);
            }
        }
    }
    const unsigned long long total = block_scan((unsigned long long)below, sh);
    if (threadIdx.x == 255) {
        const uint32_t c = held;
        counts[blockIdx.x] = c;
        atomicAdd(&st->below, total);
        atomicAdd(&st->n_cand, (unsigned long long)c);
        if (c > region_cap)
            atomicAdd(&st->full, 1u);
    }
}

// Histogram of the keys in question in 2048 bins.  keys == nullptr: the
// collected keys, a wave per region; few workgroups then, since each adds up
// to 2048 counters to the device's.
__global__ __launch_bounds__(1024) void k_sel_pass(const float *__restrict__ keys, int64_t n,
                                                   const float *__restrict__ cand,
                                                   const uint32_t *__restrict__ counts,
                                                   int regions, uint32_t region_cap,
                                                   const SelState *__restrict__ st,
                                                   unsigned long long *__restrict__ hist)
{
    __shared__ uint32_t h[kSelBins];
    if (st->done || (!keys && (st->missed || (!st->counted && !st->bracket_holds()))))
        return;
    const uint32_t lo = st->lo, span = st->span, shift = st->shift;
    for (int b = threadIdx.x; b < kSelBins; b += 1024)
        h[b] = 0;
    __syncthreads();
    const auto add = [&](float f) {
        const uint32_t t = order_key(f) - lo;
        if (t <= span)
            atomicAdd(&h[t >> shift], 1u);
    };
    // four loads in flight
    const auto stream = [&](const float *src, int64_t first, int64_t stride, int64_t count) {
        int64_t i = first;
        for (; i + 3 * stride < count; i += 4 * stride) {
            const float f0 = src[i], f1 = src[i + stride], f2 = src[i + 2 * stride],
                        f3 = src[i + 3 * stride];
            add(f0);
            add(f1);
            add(f2);
            add(f3);
        }
        for (; i < count; i += stride)
            add(src[i]);
    };
    if (keys) {
        stream(keys, (int64_t)blockIdx.x * 1024 + threadIdx.x, (int64_t)gridDim.x * 1024, n);
    } else {
        const int wave = blockIdx.x * 16 + (threadIdx.x >> 6);
        for (int r = wave; r < regions; r += gridDim.x * 16)
            stream(cand + (int64_t)r * region_cap, threadIdx.x & 63, 64, counts[r]);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < kSelBins; b += 1024)
        if (h[b])
            atomicAdd(&hist[b], (unsigned long long)h[b]);
}

// One workgroup: narrows the keys in question to the bin of rank k (2 or 3
// passes leave one key) and clears the histogram.  Where the bracket holds
// rank k but the regions do not hold its keys, the passes that follow go over
// the array and count only the keys of the bracket: no more than the two that
// 22 bits take, and none if they are all equal.
__global__ __launch_bounds__(1024) void k_sel_pick(SelState *st, unsigned long long *hist,
                                                   bool whole)
{
    __shared__ unsigned long long sh[16];
    SelState now = *st;
    __syncthreads();
    if (now.done || (now.missed && !whole)) // whole: the pass was over the array
        return;
    if (!now.counted) {
        now.missed = !now.bracket_holds();
        now.counted = 1;
        if (now.inside())
            now.k -= now.below;
        else
            sel_whole_range(&now);
        if (now.missed) {
            if (now.span == 0) {
                now.result = key_float(now.lo);
                now.done = 1;
            }
            if (threadIdx.x == 0)
                *st = now;
            return;
        }
    }
    const int b0 = 2 * threadIdx.x;
    const unsigned long long c0 = hist[b0], c1 = hist[b0 + 1];
    hist[b0] = 0;
    hist[b0 + 1] = 0;
    const unsigned long long c = block_scan(c0 + c1, sh) - c0 - c1;
    if (now.k < c || now.k >= c + c0 + c1)
        return;
    // one thread: rank k lies in one of its two bins
    const bool second = now.k >= c + c0;
    now.lo += (uint32_t)(b0 + (second ? 1 : 0)) << now.shift;
    now.span = (1u << now.shift) - 1u;
    now.k -= second ? c + c0 : c;
    now.counted = 1;
    if (now.shift == 0) {
        now.result = key_float(now.lo);
        now.done = 1;
    }
    now.shift = sel_shift(now.span);
    *st = now;
}

// ---- exclusive scan of int64 (in place, total appended at a[n]) ---------
constexpr int kScanTile = 2048; // 1024 threads x 2

__device__ __forceinline__ int64_t block_exclusive_scan_1024(int64_t v, int64_t *sh,
                                                             int64_t &total)
{
    // v: this thread's value; returns exclusive prefix within the block
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int64_t x = v;
    for (int off = 1; off < 64; off <<= 1) {
        int64_t y = __shfl_up(x, off, 64);
        if (lane >= off)
            x += y;
    }
    if (lane == 63)
        sh[wid] = x;
    __syncthreads();
    if (wid == 0) {
        int64_t w = lane < 16 ? sh[lane] : 0;
        for (int off = 1; off < 16; off <<= 1) {
            int64_t y = __shfl_up(w, off, 64);
            if (lane >= off)
                w += y;
        }
        if (lane < 16)
            sh[16 + lane] = w;
    }
    __syncthreads();
    int64_t wave_before = wid > 0 ? sh[16 + wid - 1] : 0;
    total = sh[16 + 15];
    __syncthreads();
    return wave_before + x - v;
}

__global__ __launch_bounds__(1024) void k_scan_tiles(const int64_t *__restrict__ a, int64_t n,
                                                     int64_t *__restrict__ tile_sums)
{
    __shared__ int64_t sh[32];
    int64_t base = (int64_t)blockIdx.x * kScanTile + 2 * threadIdx.x;
    int64_t v = (base < n ? a[base] : 0) + (base + 1 < n ? a[base + 1] : 0);
    int64_t total;
    block_exclusive_scan_1024(v, sh, total);
    if (threadIdx.x == 0)
        tile_sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(1024) void k_scan_sums(int64_t *__restrict__ tile_sums, int64_t nt)
{
    __shared__ int64_t sh[32];
    int64_t carry = 0;
    for (int64_t b = 0; b < nt; b += 1024) {
        int64_t idx = b + threadIdx.x;
        int64_t v = idx < nt ? tile_sums[idx] : 0;
        int64_t total;
        int64_t ex = block_exclusive_scan_1024(v, sh, total);
        if (idx < nt)
            tile_sums[idx] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0)
        tile_sums[nt] = carry;
}

// the whole scan in one workgroup, tile after tile with a running carry
// (short arrays: one launch instead of three)
__global__ __launch_bounds__(1024) void k_scan_small(int64_t *__restrict__ a, int64_t n)
{
    __shared__ int64_t sh[32];
    int64_t carry = 0;
    for (int64_t t0 = 0; t0 < n; t0 += kScanTile) {
        const int64_t base = t0 + 2 * threadIdx.x;
        const int64_t v0 = base < n ? a[base] : 0;
        const int64_t v1 = base + 1 < n ? a[base + 1] : 0;
        int64_t total;
        const int64_t ex = block_exclusive_scan_1024(v0 + v1, sh, total);
        if (base < n)
            a[base] = carry + ex;
        if (base + 1 < n)
            a[base + 1] = carry + ex + v0;
        carry += total;
    }
    if (threadIdx.x == 0)
        a[n] = carry;
}

__global__ __launch_bounds__(1024) void k_scan_apply(int64_t *__restrict__ a, int64_t n,
                                                     const int64_t *__restrict__ tile_sums,
                                                     int64_t nt)
{
    __shared__ int64_t sh[32];
    int64_t base = (int64_t)blockIdx.x * kScanTile + 2 * threadIdx.x;
    int64_t v0 = base < n ? a[base] : 0;
    int64_t v1 = base + 1 < n ? a[base + 1] : 0;
    int64_t total;
    int64_t ex = block_exclusive_scan_1024(v0 + v1, sh, total);
    int64_t off = tile_sums[blockIdx.x] + ex;
    if (base < n)
        a[base] = off;
    if (base + 1 < n)
        a[base + 1] = off + v0;
    if (blockIdx.x == 0 && threadIdx.x == 0)
        a[n] = tile_sums[nt];
}

// ---- edges ----------------------------------------------------------------
// A row of the pair arrays in 16-byte units: rows start at any float, so unit
// u covers the row's elements 4u - shift .. 4u - shift + 3, loaded as one
// vector unless it runs over the row's ends.
struct RowUnits {
    const float *row;
    int len, shift;

    __device__ RowUnits(const float *r, int n) : row(r), len(n)
    {
        shift = (int)(((uintptr_t)r >> 2) & 3);
    }
    __device__ int units() const { return (len + shift + 3) >> 2; }
    // elements outside the row read as +inf, below no threshold
    __device__ float4 load(int u) const
    {
        const int k = 4 * u - shift;
        if (k >= 0 && k + 4 <= len)
            return *reinterpret_cast<const float4 *>(row + k);
        const float none = INFINITY;
        return make_float4(k >= 0 && k < len ? row[k] : none,
                           k + 1 >= 0 && k + 1 < len ? row[k + 1] : none,
                           k + 2 >= 0 && k + 2 < len ? row[k + 2] : none,
                           k + 3 >= 0 && k + 3 < len ? row[k + 3] : none);
    }
};

constexpr int kRowUnits = 8; // 16-byte units in flight per thread

// Bound by the read: 256 MB in 38 us, 53 with 4-byte loads one at a time.

__global__ __launch_bounds__(256) void k_count_rows(const float *__restrict__ copts, int num,
                                                    float rn, int64_t *__restrict__ counts)
{
    __shared__ int sh[4];
    const int i = blockIdx.x;
    const RowUnits R(copts + (int64_t)i * (num - 1), num - 1);
    const int n = R.units();
    int c = 0;
    for (int u0 = 0; u0 < n; u0 += 256 * kRowUnits) {
        float4 v[kRowUnits];
#pragma unroll
        for (int j = 0; j < kRowUnits; ++j)
            v[j] = R.load(u0 + j * 256 + threadIdx.x);
#pragma unroll
        for (int j = 0; j < kRowUnits; ++j)
            c += (v[j].x < rn) + (v[j].y < rn) + (v[j].z < rn) + (v[j].w < rn);
    }
    for (int off = 32; off > 0; off >>= 1)
        c += __shfl_down(c, off, 64);
    if ((threadIdx.x & 63) == 0)
        sh[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0)
        counts[i] = (int64_t)(sh[0] + sh[1] + sh[2] + sh[3]);
}

// Order-preserving compaction of one row: a thread's units come in strips of
// 256, so the order is strip, then thread, then element.  A wave's place in a
// strip comes from ballots, the strips' and waves' places from one scan of
// their 4 * kRowUnits counts.  The kept elements' indexes go to LDS first, so
// that the gathers of the two values are in flight together and the four
// stores are coalesced.  Bound by the read of the costs and one line of topts
// per edge; 8000 rows with 6 of 1000 kept: 131 us with 256 elements and two
// barriers at a time, 67 us with the stores made by the element's lane, 55 us so.
__global__ __launch_bounds__(256) void k_fill_rows(const float *__restrict__ copts,
                                                   const float *__restrict__ topts, int num,
                                                   float rn, const int64_t *__restrict__ row_start,
                                                   int *__restrict__ edge_src,
                                                   int *__restrict__ edge_dst,
                                                   float *__restrict__ copts_edge,
                                                   float *__restrict__ topts_edge)
{
    __shared__ int cnt[kRowUnits * 4];
    __shared__ uint16_t kept[kRowUnits * 256 * 4];
    const int i = blockIdx.x;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int64_t rbase = (int64_t)i * (num - 1);
    const RowUnits R(copts + rbase, num - 1);
    const int n = R.units();
    const uint64_t lower = (1ull << lane) - 1ull;
    int64_t out = row_start[i];
    for (int u0 = 0; u0 < n; u0 += 256 * kRowUnits) {
        int before[kRowUnits]; // kept elements of lower lanes in the strip
        uint32_t mine = 0;     // 4 bits per strip
        float4 v[kRowUnits];
#pragma unroll
        for (int j = 0; j < kRowUnits; ++j)
            v[j] = R.load(u0 + j * 256 + threadIdx.x);
#pragma unroll
        for (int j = 0; j < kRowUnits; ++j) {
            const uint64_t m0 = __ballot(v[j].x < rn), m1 = __ballot(v[j].y < rn),
                           m2 = __ballot(v[j].z < rn), m3 = __ballot(v[j].w < rn);
            before[j] = __popcll(m0 & lower) + __popcll(m1 & lower) + __popcll(m2 & lower) +
                        __popcll(m3 & lower);
            mine |= (uint32_t)((v[j].x < rn) | (v[j].y < rn) << 1 | (v[j].z < rn) << 2 |
                               (v[j].w < rn) << 3)
                    << (4 * j);
            if (lane == 0)
                cnt[j * 4 + wid] = __popcll(m0) + __popcll(m1) + __popcll(m2) + __popcll(m3);
        }
        __syncthreads();
        int incl = lane < 4 * kRowUnits ? cnt[lane] : 0;
        const int own = incl;
        for (int off = 1; off < 4 * kRowUnits; off <<= 1) {
            const int y = __shfl_up(incl, off, 64);
            if (lane >= off)
                incl += y;
        }
        const int excl = incl - own;
#pragma unroll
        for (int j = 0; j < kRowUnits; ++j) {
            int e = __shfl(excl, j * 4 + wid, 64) + before[j];
            uint32_t bits = (mine >> (4 * j)) & 15u;
            while (bits) {
                kept[e++] = (uint16_t)(4 * (j * 256 + (int)threadIdx.x) + __builtin_ctz(bits));
                bits &= bits - 1u;
            }
        }
        const int total = __shfl(incl, 4 * kRowUnits - 1, 64);
        __syncthreads();
        for (int q = threadIdx.x; q < total; q += 256) {
            const int k = 4 * u0 - R.shift + kept[q];
            const float c = R.row[k], t = topts[rbase + k];
            edge_src[out + q] = i;
            edge_dst[out + q] = k + (k >= i ? 1 : 0);
            copts_edge[out + q] = c;
            topts_edge[out + q] = t;
        }
        out += total;
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) void k_zero_i32(int *__restrict__ a, int64_t n)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        a[i] = 0;
}

__global__ __launch_bounds__(256) void k_fill_i32(int *__restrict__ a, int64_t n, int v)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        a[i] = v;
}

// In-degrees, counted in LDS first: a workgroup takes a share of the edges
// (blockIdx.x) and kDegTile destinations (blockIdx.y).  Bound by the device's
// counters, 12 additions per ns: 4e5 edges into 8000 took 33 us one by one and
// take 6 us with kDegShares workgroups that add 8000 counters each.
constexpr int kDegTile = 16384;
constexpr int kDegShares = 16;

__global__ __launch_bounds__(1024) void k_in_degree(const int *__restrict__ edge_dst, int64_t n,
                                                    int num, int *__restrict__ indeg)
{
    extern __shared__ int deg[];
    const int d0 = blockIdx.y * kDegTile;
    const int nd = min(num - d0, kDegTile);
    for (int d = threadIdx.x; d < nd; d += 1024)
        deg[d] = 0;
    __syncthreads();
    const int64_t stride = (int64_t)gridDim.x * 1024;
    int64_t e = (int64_t)blockIdx.x * 1024 + threadIdx.x;
    const auto add = [&](int dst) {
        if ((unsigned)(dst - d0) < (unsigned)nd)
            atomicAdd(&deg[dst - d0], 1);
    };
    for (; e + 7 * stride < n; e += 8 * stride) {
        int dst[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            dst[j] = edge_dst[e + j * stride];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            add(dst[j]);
    }
    for (; e < n; e += stride)
        add(edge_dst[e]);
    __syncthreads();
    for (int d = threadIdx.x; d < nd; d += 1024)
        if (deg[d])
            atomicAdd(&indeg[d0 + d], deg[d]);
}

// one workgroup: the largest degree
__global__ __launch_bounds__(1024) void k_max_deg(const int64_t *__restrict__ row_start,
                                                  const int *__restrict__ indeg, int num,
                                                  int *__restrict__ out)
{
    __shared__ int sh[16];
    int m = 0;
    for (int i = threadIdx.x; i < num; i += 1024) {
        const int go = (int)(row_start[i + 1] - row_start[i]);
        m = max(m, max(go, indeg[i]));
    }
    for (int off = 32; off > 0; off >>= 1)
        m = max(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0)
        sh[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; ++w)
            m = max(m, sh[w]);
        *out = m;
    }
}

__global__ __launch_bounds__(256) void k_nn_go(const int64_t *__restrict__ row_start,
                                               const int *__restrict__ edge_dst, int num,
                                               int max_nn, int *__restrict__ go)
{
    const int64_t n = (int64_t)num * max_nn;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += stride) {
        int i = (int)(q / max_nn);
        int nn = (int)(q - (int64_t)i * max_nn);
        int64_t deg = row_start[i + 1] - row_start[i];
        go[q] = nn < deg ? edge_dst[row_start[i] + nn] : -1;
    }
}

// unordered in-lists, then each node's list sorted by source (sources of one
// destination are distinct, so rank = number of smaller sources)
__global__ __launch_bounds__(256) void k_come_scatter(const int *__restrict__ edge_src,
                                                      const int *__restrict__ edge_dst,
                                                      const float *__restrict__ copts_edge,
                                                      int64_t n, int max_nn,
                                                      int *__restrict__ fill,
                                                      int *__restrict__ come,
                                                      float *__restrict__ dist)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += stride) {
        int j = edge_dst[e];
        int slot = atomicAdd(&fill[j], 1);
        come[(int64_t)j * max_nn + slot] = edge_src[e];
        dist[(int64_t)j * max_nn + slot] = copts_edge[e];
    }
}

__global__ __launch_bounds__(256) void k_come_sort(const int *__restrict__ fill, int max_nn,
                                                   int *__restrict__ come,
                                                   float *__restrict__ dist)
{
    extern __shared__ unsigned char smem[];
    int *src = reinterpret_cast<int *>(smem);
    float *dd = reinterpret_cast<float *>(src + max_nn);
    const int j = blockIdx.x;
    const int n = fill[j];
    int *row = come + (int64_t)j * max_nn;
    float *drow = dist + (int64_t)j * max_nn;
    for (int q = threadIdx.x; q < n; q += blockDim.x) {
        src[q] = row[q];
        dd[q] = drow[q];
    }
    __syncthreads();
    for (int q = threadIdx.x; q < n; q += blockDim.x) {
        int s = src[q];
        int r = 0;
        for (int m = 0; m < n; ++m)
            r += src[m] < s;
        row[r] = s;
        drow[r] = dd[q];
    }
}

__global__ __launch_bounds__(256) void k_nn_idxs(const int *__restrict__ edge_src,
                                                 const int *__restrict__ edge_dst, int64_t n,
                                                 int num, int *__restrict__ nn_idxs)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += stride)
        nn_idxs[(int64_t)edge_dst[e] * num + edge_src[e]] = (int)e;
}

__global__ __launch_bounds__(256) void k_wcount(const float *__restrict__ topts_edge, int64_t n,
                                                int w_fixed, float wp_dt, int w_cap,
                                                int64_t *__restrict__ w)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += stride) {
        int c;
        if (w_fixed > 0) {
            c = w_fixed;
        } else {
            c = (int)ceilf(topts_edge[e] / wp_dt);
            c = c < 2 ? 2 : c;
            c = c > w_cap ? w_cap : c;
        }
        w[e] = c;
    }
}

} // namespace

// in-place exclusive scan of a[0..n), total into a[n]
int scan_exclusive_i64(int64_t *d_a, int64_t n, void *d_ws, size_t ws_bytes, hipStream_t s)
{
    const int64_t nt = (n + kScanTile - 1) / kScanTile;
    if (n >= 0 && nt <= 8) {
        hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(1024), 0, s, d_a, n);
        PUMP_LAUNCHED();
        return PUMP_OK;
    }
    if (ws_bytes < (size_t)(nt + 1) * sizeof(int64_t) || !d_ws)
        return PUMP_E_CAPACITY;
    int64_t *sums = reinterpret_cast<int64_t *>(d_ws);
    if (nt > 0) {
        hipLaunchKernelGGL(k_scan_tiles, dim3((unsigned)nt), dim3(1024), 0, s, d_a, n, sums);
        PUMP_LAUNCHED();
    }
    hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(1024), 0, s, sums, nt);
    PUMP_LAUNCHED();
    if (nt > 0) {
        hipLaunchKernelGGL(k_scan_apply, dim3((unsigned)nt), dim3(1024), 0, s, d_a, n, sums, nt);
        PUMP_LAUNCHED();
    } else {
        PUMP_HIP(hipMemsetAsync(d_a, 0, sizeof(int64_t), s));
    }
    return PUMP_OK;
}

} // namespace pump

using namespace pump;

extern "C" int64_t pump_rn_index(int64_t num, float rn_perc)
{
    float prod = (float)((num - 1) * num) * rn_perc;
    return (int64_t)prod;
}

// state and histogram; the bracket's keys follow when the workspace holds them
constexpr size_t kSelHist = 280;
static_assert(sizeof(SelState) <= kSelHist && kSelHist % 8 == 0, "layout of the selection");
static size_t select_rn_base() { return kSelHist + kSelBins * sizeof(unsigned long long); }

// Room for the bracket's keys, in equal regions: 10 sqrt(16384 p) + 8 of 16384
// where a share p or 1 - p of the keys lies below, 5.7% at most (p = 1/2; 0.8%
// for the 50 nearest of 8000), of the 6.25% and more that there is room for.
// Past it the passes go over the array: a middle rank of clustered keys can.
static int64_t select_rn_cand(int64_t n) { return n <= kSelSample ? 0 : n / 16 + 131072; }

extern "C" size_t pump_select_rn_workspace(int64_t n_pairs)
{
    return select_rn_base() + kSelMaxRegions * sizeof(uint32_t) +
           (size_t)select_rn_cand(n_pairs) * sizeof(float);
}

extern "C" int pump_select_rn(const float *d_copts, int64_t n_pairs, int64_t rn_idx, float *rn_host,
                              void *d_ws, size_t ws_bytes, pump_stream_t stream)
{
    PUMP_REQUIRE(d_copts && rn_host && n_pairs > 0 && rn_idx >= 0 && rn_idx < n_pairs);
    if (!d_ws || ws_bytes < select_rn_base())
        return PUMP_E_CAPACITY;
    hipStream_t s = as_stream(stream);
    SelState *st = reinterpret_cast<SelState *>(d_ws);
    unsigned long long *hist =
        reinterpret_cast<unsigned long long *>(reinterpret_cast<char *>(d_ws) + kSelHist);
    uint32_t *counts = reinterpret_cast<uint32_t *>(hist + kSelBins);
    float *cand = reinterpret_cast<float *>(counts + kSelMaxRegions);
    const unsigned long long k = (unsigned long long)rn_idx;
    int dev = 0, cus = 256;
    hipGetDevice(&dev);
    hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    const int regions = (int)grid_for(n_pairs, kSelTile, std::min(cus * 4, kSelMaxRegions));
    const uint32_t region_cap = (uint32_t)(select_rn_cand(n_pairs) / regions);
    const auto pass = [&](const float *keys) {
        const unsigned blocks = keys ? grid_for(n_pairs / 4 + 1, 1024, (int64_t)cus * 2) : 16u;
        hipLaunchKernelGGL(k_sel_pass, dim3(blocks), dim3(1024), 0, s, keys, n_pairs, cand, counts,
                           regions, region_cap, st, hist);
        hipLaunchKernelGGL(k_sel_pick, dim3(1), dim3(1024), 0, s, st, hist,
                           keys != nullptr);
    };
    const bool bracket = ws_bytes >= pump_select_rn_workspace(n_pairs);
    if (bracket) {
        hipLaunchKernelGGL(k_sel_sample, dim3(1), dim3(1024), 0, s, d_copts, n_pairs, k, st, hist);
        PUMP_LAUNCHED();
        if (n_pairs > kSelSample) {
            hipLaunchKernelGGL(k_sel_bracket, dim3(regions), dim3(256), 0, s, d_copts, n_pairs, st,
                               cand, counts, region_cap, n_pairs <= kSelScatterMax);
            PUMP_LAUNCHED();
            // an open bracket has more than 22 bits
            const SelRanks R = sel_ranks(rn_idx, n_pairs, kSelSample);
            for (int p = 0; p < (R.open_lo || R.open_hi ? 3 : 2); ++p) {
                pass(nullptr);
                PUMP_LAUNCHED();
            }
        }
    } else {
        hipLaunchKernelGGL(k_sel_init, dim3(1), dim3(256), 0, s, st, hist, k);
        PUMP_LAUNCHED();
        for (int p = 0; p < 3; ++p) {
            pass(d_copts);
            PUMP_LAUNCHED();
        }
    }
    SelState got;
    PUMP_HIP(hipMemcpyAsync(&got, st, sizeof(got), hipMemcpyDeviceToHost, s));
    PUMP_HIP(hipStreamSynchronize(s));
    if (!got.done) {
        // 11 bits a pass: over the array where the collected keys do not do
        for (uint32_t left = got.span; left; left >>= 11) {
            pass(got.missed ? d_copts : nullptr);
            PUMP_LAUNCHED();
        }
        PUMP_HIP(hipMemcpyAsync(&got, st, sizeof(got), hipMemcpyDeviceToHost, s));
        PUMP_HIP(hipStreamSynchronize(s));
    }
    *rn_host = got.result;
    return PUMP_OK;
}

extern "C" size_t pump_scan_workspace(int64_t n)
{
    return (size_t)((n + kScanTile - 1) / kScanTile + 2) * sizeof(int64_t);
}

extern "C" int pump_count_edges(const float *d_copts, int num, float rn, int64_t *d_row_start,
                                int64_t *n_edges_host, void *d_ws, size_t ws_bytes,
                                pump_stream_t stream)
{
    PUMP_REQUIRE(d_copts && d_row_start && n_edges_host && num >= 2);
    hipStream_t s = as_stream(stream);
    hipLaunchKernelGGL(k_count_rows, dim3(num), dim3(256), 0, s, d_copts, num, rn, d_row_start);
    PUMP_LAUNCHED();
    int r = scan_exclusive_i64(d_row_start, num, d_ws, ws_bytes, s);
    if (r != PUMP_OK)
        return r;
    int64_t total = 0;
    PUMP_HIP(hipMemcpyAsync(&total, d_row_start + num, sizeof(int64_t), hipMemcpyDeviceToHost, s));
    PUMP_HIP(hipStreamSynchronize(s));
    *n_edges_host = total;
    return PUMP_OK;
}

extern "C" int pump_fill_edges(const float *d_copts, const float *d_topts, int num, float rn,
                               const int64_t *d_row_start, int *d_edge_src, int *d_edge_dst,
                               float *d_copts_edge, float *d_topts_edge, pump_stream_t stream)
{
    PUMP_REQUIRE(d_copts && d_topts && d_row_start && d_edge_src && d_edge_dst && d_copts_edge &&
                 d_topts_edge && num >= 2);
    hipLaunchKernelGGL(k_fill_rows, dim3(num), dim3(256), 0, as_stream(stream), d_copts, d_topts,
                       num, rn, d_row_start, d_edge_src, d_edge_dst, d_copts_edge, d_topts_edge);
    PUMP_LAUNCHED();
    return PUMP_OK;
}

extern "C" int pump_max_nn_size(const int64_t *d_row_start, const int *d_edge_dst, int64_t n_edges,
                                int num, int *d_in_degree, int *max_nn_host, pump_stream_t stream)
{
    PUMP_REQUIRE(d_row_start && d_in_degree && max_nn_host && num >= 1);
    PUMP_REQUIRE(n_edges == 0 || d_edge_dst);
    hipStream_t s = as_stream(stream);
    int *d_max = nullptr;
    PUMP_HIP(hipMalloc((void **)&d_max, sizeof(int)));
    hipLaunchKernelGGL(k_zero_i32, dim3(grid_for(num + 1, 256)), dim3(256), 0, s, d_in_degree,
                       (int64_t)num);
    if (n_edges > 0)
        hipLaunchKernelGGL(k_in_degree,
                           dim3(grid_for(n_edges, 4096, kDegShares),
                                (unsigned)((num + kDegTile - 1) / kDegTile)),
                           dim3(1024), sizeof(int) * (size_t)std::min(num, kDegTile), s,
                           d_edge_dst, n_edges, num, d_in_degree);
    hipLaunchKernelGGL(k_max_deg, dim3(1), dim3(1024), 0, s, d_row_start, d_in_degree, num, d_max);
    hipError_t le = hipGetLastError();
    int m = 0;
    hipError_t ce = hipMemcpyAsync(&m, d_max, sizeof(int), hipMemcpyDeviceToHost, s);
    hipError_t se = hipStreamSynchronize(s);
    hipFree(d_max);
    PUMP_HIP(le);
    PUMP_HIP(ce);
    PUMP_HIP(se);
    *max_nn_host = m;
    return PUMP_OK;
}

extern "C" int pump_nn_tables(const int64_t *d_row_start, const int *d_edge_src,
                              const int *d_edge_dst, const float *d_copts_edge, int64_t n_edges,
                              int num, int max_nn, int *d_nn_go_edges, int *d_nn_come_edges,
                              float *d_distances_come, int *d_nn_idxs, pump_stream_t stream)
{
    PUMP_REQUIRE(d_row_start && num >= 1 && max_nn >= 0);
    hipStream_t s = as_stream(stream);
    const int64_t tab = (int64_t)num * max_nn;
    if (d_nn_go_edges && tab > 0) {
        hipLaunchKernelGGL(k_nn_go, dim3(grid_for(tab, 256)), dim3(256), 0, s, d_row_start,
                           d_edge_dst, num, max_nn, d_nn_go_edges);
        PUMP_LAUNCHED();
    }
    if (d_nn_come_edges && d_distances_come && tab > 0) {
        int *fill = nullptr;
        PUMP_HIP(hipMalloc((void **)&fill, sizeof(int) * (size_t)num));
        hipLaunchKernelGGL(k_zero_i32, dim3(grid_for(num, 256)), dim3(256), 0, s, fill,
                           (int64_t)num);
        hipLaunchKernelGGL(k_fill_i32, dim3(grid_for(tab, 256)), dim3(256), 0, s,
                           d_nn_come_edges, tab, -1);
        hipLaunchKernelGGL(k_zero_i32, dim3(grid_for(tab, 256)), dim3(256), 0, s,
                           reinterpret_cast<int *>(d_distances_come), tab);
        if (n_edges > 0) {
            hipLaunchKernelGGL(k_come_scatter, dim3(grid_for(n_edges, 256)), dim3(256), 0, s,
                               d_edge_src, d_edge_dst, d_copts_edge, n_edges, max_nn, fill,
                               d_nn_come_edges, d_distances_come);
            hipLaunchKernelGGL(k_come_sort, dim3(num), dim3(256),
                               (size_t)max_nn * (sizeof(int) + sizeof(float)), s, fill, max_nn,
                               d_nn_come_edges, d_distances_come);
        }
        hipError_t le = hipGetLastError();
        hipError_t se = hipStreamSynchronize(s);
        hipFree(fill);
        PUMP_HIP(le);
        PUMP_HIP(se);
    }
    if (d_nn_idxs) {
        const int64_t nn2 = (int64_t)num * num;
        hipLaunchKernelGGL(k_fill_i32, dim3(grid_for(nn2, 256)), dim3(256), 0, s, d_nn_idxs, nn2,
                           -3);
        if (n_edges > 0)
            hipLaunchKernelGGL(k_nn_idxs, dim3(grid_for(n_edges, 256)), dim3(256), 0, s,
                               d_edge_src, d_edge_dst, n_edges, num, d_nn_idxs);
        PUMP_LAUNCHED();
    }
    return PUMP_OK;
}

extern "C" int pump_waypoint_offsets(const float *d_topts_edge, int64_t n_edges, int w_fixed,
                                     float wp_dt, int w_cap, int64_t *d_wp_offsets,
                                     int64_t *total_host, void *d_ws, size_t ws_bytes,
                                     pump_stream_t stream)
{
    PUMP_REQUIRE(d_wp_offsets && total_host && n_edges >= 0);
    PUMP_REQUIRE(w_fixed >= 2 || (w_fixed <= 0 && w_cap >= 2 && wp_dt > 0.0f && d_topts_edge));
    PUMP_REQUIRE(w_fixed < kMaxWaypointsPerEdge && w_cap < kMaxWaypointsPerEdge);
    hipStream_t s = as_stream(stream);
    if (n_edges > 0) {
        hipLaunchKernelGGL(k_wcount, dim3(grid_for(n_edges, 256)), dim3(256), 0, s, d_topts_edge,
                           n_edges, w_fixed, wp_dt, w_cap, d_wp_offsets);
        PUMP_LAUNCHED();
    }
    int r = scan_exclusive_i64(d_wp_offsets, n_edges, d_ws, ws_bytes, s);
    if (r != PUMP_OK)
        return r;
    int64_t total = 0;
    PUMP_HIP(hipMemcpyAsync(&total, d_wp_offsets + n_edges, sizeof(int64_t),
                            hipMemcpyDeviceToHost, s));
    PUMP_HIP(hipStreamSynchronize(s));
    *total_host = total;
    return PUMP_OK;
}
